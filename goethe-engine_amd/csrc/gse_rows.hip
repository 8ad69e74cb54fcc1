// Row passes: selection work on whole rows of probabilities, each row spread over slices of RS tokens so that a call of
// a few rows still fills the device. A slice's workgroup reads its tokens once, writes the slice's sums, and takes an
// atomic ticket; the row's last slice finishes the row in the same launch from the slices' sums (a draw reads the
// crossing slice's 64 segment sums and then one segment: three dependent reads, not a pass over the row).
//
//   draw  sampling.py:100-104  inverse CDF in vocabulary order of fp64 rows
//   mss   spec.py:88-103       multi-step speculative sampling: one launch per residual level, at most MSS_LEVELS of them
//   pick  spec.py:151-159      the drafter's children (TreeDrafter._pick) of rows of logits, one launch
//   qprob spec.py:157          the drafter's fp64 softmax rows, two launches
//
// What bounds them: a slice is one round of coalesced 512-byte reads per wave (16 tokens a thread), so at the sizes of a
// decode step a launch is latency: load, sums, ticket, the last slice's reads. One workgroup per row, each thread summing
// a contiguous run (128 tokens at V = 128256: every load of a wave touched 64 cache lines, one CU per row), took 0.9 ms
// for 16 mss nodes of V = 128256 and two kids, 85 % of a dist + mss call (1014 us); sliced, that call takes 106 us.
#include <type_traits>

#include "gse_dev.h"
#include "gse_int.h"

namespace gse {

namespace {

constexpr int RT = 256;           // threads of a slice's workgroup
constexpr int RW = RT / WAVE;     // its waves
constexpr int RSEG = 64;          // segments per slice (segment g: the wave g % RW's 64 * sub tokens)
constexpr int RGS = RSEG / RW;    // segments per wave
static_assert(RS == RSEG * WAVE, "a segment of a slice that is not widened is one token per lane");

// The rows' slicing: slice s of a row holds the tokens [s len, (s + 1) len) of the row, len = RS * sub; its segment g the
// tokens [g, g + 1) * 64 sub of it. sub is 1 unless the vocabulary is far larger than the handle was opened for (the
// workspace holds a fixed number of slices per row).
struct RowSlices {
  int ns, sub;
};

struct RowsShared {
  double seg[RSEG];
  double red[RW];
  int lastw[RW];
  uint32_t ticket;
};

// Sums the weights of slice s of a row of V tokens: load(t) issues the loads of token t (called for in-range tokens; past
// the row it is called with the row's last token and the weight dropped), ev(t, loaded) gives its weight. The segment
// sums go to segs[0, RSEG), the slice's sum to *sum and the last token with a positive weight (-1 none) to *last, all
// with agent-scope stores by the workgroup, which are complete when this returns (after a barrier). Fixed association:
// the same sums for the same row whatever else the call holds.
template <typename LD, typename EV>
__device__ __forceinline__ void slice_sum(const RowSlices &rs, int s, int V, LD load, EV ev, double *segs, double *sum,
                                          int32_t *last, RowsShared &sh) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  // (unsigned: past the end of a row of nearly 2^31 tokens)
  const uint32_t s0 = (uint32_t)(s * RS * rs.sub), end = (uint32_t)V;
  int lst = -1;
  if (rs.sub == 1) {
    // eight segments' loads in flight at a time
#pragma unroll
    for (int h = 0; h < RGS; h += 8) {
      decltype(load(0)) r[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) r[k] = load((int)min(s0 + (uint32_t)(((h + k) * RW + w) * WAVE + lane), end - 1u));
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int g = (h + k) * RW + w;
        const uint32_t t = s0 + (uint32_t)(g * WAVE + lane);
        const double v = t < end ? ev((int)t, r[k]) : 0.0;
        if (v > 0.0) lst = (int)t;
        const double sg = wave_sum_f64(v);
        if (lane == 0) sh.seg[g] = sg;
      }
    }
  } else {
#pragma unroll 1
    for (int q = 0; q < RGS; ++q) {
      const int g = q * RW + w;
      double sg = 0.0;
      for (int c = 0; c < rs.sub; ++c) {
        const uint32_t t = s0 + (uint32_t)((g * rs.sub + c) * WAVE + lane);
        const double v = t < end ? ev((int)t, load((int)t)) : 0.0;
        if (v > 0.0) lst = (int)t;
        sg += wave_sum_f64(v);
      }
      if (lane == 0) sh.seg[g] = sg;
    }
  }
  lst = (int)wave_max_u32((uint32_t)(lst + 1)) - 1;
  if (lane == 0) sh.lastw[w] = lst;
  __syncthreads();
  if (threadIdx.x < RSEG) {
    const double sg = sh.seg[threadIdx.x];
    st_ag(&segs[threadIdx.x], sg);
    const double tot = wave_sum_f64(sg);
    if (threadIdx.x == 0) {
      int l = sh.lastw[0];
      for (int k = 1; k < RW; ++k) l = max(l, sh.lastw[k]);
      st_ag(sum, tot);
      st_ag(last, l);
    }
  }
  store_wait();
  __syncthreads();
}

// The total of a row's ns slice sums (every lane of the wave gets it), in a fixed order.
__device__ __forceinline__ double row_total(const double *sums, int ns) {
  double t = 0.0;
  for (int j0 = 0; j0 < ns; j0 += WAVE) {
    const int j = j0 + lane_id();
    t += wave_sum_f64(j < ns ? ld_ag(&sums[j]) : 0.0);
  }
  return t;
}

// The first j in [0, n) with v(j) > 0 whose inclusive prefix before + sum(v(0..j)) reaches thr, 64 values at a time; before
// becomes the prefix ahead of it. -1 when none does. lastp: the last j seen with v(j) > 0 (-1 none). (A zero is never the
// answer: the wave's scan adds in a tree, so a prefix may pass thr at a zero that follows the value that reached it.)
template <typename VF>
__device__ __forceinline__ int cross(int n, double thr, double &before, int &lastp, VF v) {
  lastp = -1;
  for (int j0 = 0; j0 < n; j0 += WAVE) {
    const int j = j0 + lane_id();
    const double x = j < n ? v(j) : 0.0;
    const double inc = before + wave_incl_scan_f64(x);
    const uint64_t pos = ballot64(x > 0.0), hit = ballot64(x > 0.0 && inc >= thr);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      before = l > 0 ? shfl_f64(inc, l - 1) : before;
      return j0 + l;
    }
    if (pos) lastp = j0 + 63 - (int)__builtin_clzll(pos);
    before = shfl_f64(inc, WAVE - 1);
  }
  return -1;
}

// draw() of a row whose slices have been summed (by one wave; every lane gets it): the first token whose inclusive
// prefix reaches u * total, at most the last token with a positive weight; -1 when no weight is positive. A total that
// is NaN gives the first token (count(c < NaN) = 0), and so does u = 0; any other token has a positive weight. The sums of
// slices, segments and tokens round apart, so a slice's segments, or a segment's tokens, may stay below what the sum
// above them reached: the draw then takes the last of them with a positive weight.
template <typename EW>
__device__ __forceinline__ int row_draw(const RowSlices &rs, int V, double u, double total, const double *sums,
                                        const double *segs, const int32_t *lasts, EW ev) {
  int lst = -1;
  for (int j = lane_id(); j < rs.ns; j += WAVE) lst = max(lst, ld_ag(&lasts[j]));
  lst = (int)wave_max_u32((uint32_t)(lst + 1)) - 1;
  if (lst < 0) return -1;
  const double thr = u * total;
  if (!(thr > 0.0)) return 0;
  double before = 0.0;
  int lp;
  const int sx = cross(rs.ns, thr, before, lp, [&](int j) { return ld_ag(&sums[j]); });
  if (sx < 0) return lst;
  const double *sg = segs + (size_t)sx * RSEG;
  const int g = cross(RSEG, thr, before, lp, [&](int j) { return ld_ag(&sg[j]); });
  if (g < 0) return ld_ag(&lasts[sx]);
  const int t0 = (sx * RSEG + g) * WAVE * rs.sub, nt = min(WAVE * rs.sub, V - t0);
  const int k = cross(nt, thr, before, lp, [&](int j) { return ev(t0 + j); });
  return t0 + (k < 0 ? lp : k);
}

struct DrawArgs {
  const double *q;
  int64_t ld;
  int V, row0;
  RowSlices rs;
  const double *u;
  int32_t *out;
  double *sum, *seg;   // [rows][ns], [rows][ns][RSEG]
  int32_t *last;       // [rows][ns]
  uint32_t *tick;      // [rows]
};

// ---- draw: sampling.py:100-104 ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(RT) void draw_kernel(DrawArgs a) {
  __shared__ RowsShared sh;
  const int s = blockIdx.x, r = blockIdx.y, row = a.row0 + r;
  const double *q = a.q + (int64_t)row * a.ld;
  const size_t o = (size_t)r * a.rs.ns;
  slice_sum(a.rs, s, a.V, [&](int t) { return q[t]; }, [](int, double v) { return v; }, a.seg + (o + s) * RSEG,
            a.sum + o + s, a.last + o + s, sh);
  if (threadIdx.x == 0) sh.ticket = ticket_add(&a.tick[r]);
  __syncthreads();
  if (sh.ticket != (uint32_t)(a.rs.ns - 1) || threadIdx.x >= WAVE) return;
  const double total = row_total(a.sum + o, a.rs.ns);
  const int j = row_draw(a.rs, a.V, a.u[row], total, a.sum + o, a.seg + o * RSEG, a.last + o, [&](int t) { return q[t]; });
  if (threadIdx.x == 0) {
    a.out[row] = j;
    a.tick[r] = 0;
  }
}

// ---- mss: spec.py:88-103 ---------------------------------------------------------------------------------------------
// Level d: d kids have been rejected and the row's distribution is res_d / sum(res_d), where res_d = max(p_{d-1} - q, 0)
// (one-hot kid: p_{d-1} with its token at 0) and p_{d-1} = res_{d-1} / sum(res_{d-1}) (res_{d-1} itself when that sum is
// not positive), p_0 = p. Launch d recomputes the levels from p and the q rows at every token and sums res_d (no level is
// written: a launch's slices see each other's inputs only); the row's last slice then tests the next kid against
// res_d / sum, or draws. A row with more than MSS_LEVELS kids rejected goes on in its last slice's workgroup alone, in
// place in p, one coalesced pass per kid.
constexpr int MSS_LEVELS = 3;
constexpr uint64_t SALT_ACC = 1ull << 40, SALT_RES = 1ull << 41;

struct MssArgs {
  gse_mss_batch b;
  int node0;
  RowSlices rs;
  TreeNode *st;        // [nodes] next (the level to run), ticket, sig (the levels' sums)
  double *sum, *seg;
  int32_t *last;
};

struct MssKid {
  int r, x;            // its index among the node's kids (r < 0: none), its token
  const double *q;     // its draft distribution, null: one-hot
};

// The node's kids in draft order: the first at or after index r whose token lies in the vocabulary (a token past it is
// skipped, a negative one ends the list).
__device__ __forceinline__ MssKid kid_from(const gse_mss_batch &b, int node, int r) {
  for (; r < (int)b.max_kids; ++r) {
    const int64_t i = (int64_t)node * b.max_kids + r;
    const int x = b.kid_tok[i], qr = b.kid_q[i];
    if (x < 0) break;
    if (x < (int)b.vocab) return MssKid{r, x, qr >= 0 ? b.q + (int64_t)qr * b.q_ld : nullptr};
  }
  return MssKid{-1, -1, nullptr};
}

__device__ __forceinline__ bool mss_accepts(const gse_mss_batch &b, int node, const MssKid &k, double px) {
  const double qx = k.q ? k.q[k.x] : 1.0;
  return qx > 0.0 && uniform64(mix64(b.seed[node], SALT_ACC + (uint64_t)k.r), b.idx[node]) * qx < px;
}

__device__ __forceinline__ void mss_out(const gse_mss_batch &b, int node, int tok, int kid) {
  b.out_token[node] = tok;
  b.out_kid[node] = kid;
}

__device__ __forceinline__ double residual(double p, const MssKid &k, double q, int t) {
  if (!k.q) return t == k.x ? 0.0 : p;
  const double v = p - q;
  return v > 0.0 ? v : 0.0;
}

// res_D at one token from its p and q values; sig[d] the sum of res_d.
template <int D>
__device__ __forceinline__ double level(const MssKid (&k)[MSS_LEVELS], const double (&sig)[MSS_LEVELS + 1], double p,
                                        const double *q, int t) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (d > 0 && sig[d] > 0.0) p = p / sig[d];
    p = residual(p, k[d], q[d], t);
  }
  return p;
}

template <int D>
struct MssTok {
  double p, q[D > 0 ? D : 1];
};
template <int D>
__device__ __forceinline__ MssTok<D> mss_load(const double *p, const MssKid (&k)[MSS_LEVELS], int t) {
  MssTok<D> m;
  m.p = p[t];
#pragma unroll
  for (int d = 0; d < D; ++d) m.q[d] = (k[d].q ? k[d].q : p)[t];  // (one-hot: a load that is dropped)
  return m;
}

// The kids past level MSS_LEVELS, by one workgroup, in place in p: the residual of the level before (written by this
// workgroup), total its sum. A kid is one pass over the row: the division by the sum before, the residual, and the slices'
// sums, which the next test and the draw use (a residual that is not divided draws the same), eight tokens a
// thread loading at a time. Bound by the chain of one workgroup's slices. Every kid rejected, us a call:
//   16 nodes of 128256: 4 kids 517, 16 kids 3070 (two passes a kid of 256 tokens at a time and a third for the draw: 819,
//   5700; one workgroup of 1024 threads a node over contiguous runs: 1823, 6790)
//   64 nodes of 151936: 4 kids 1240, 16 kids 8110, one-hot 850, 5150 (1840, 13400, 1410, 8720; 3380, 12600, 2700, 9860)
__device__ __noinline__ void mss_rest(const MssArgs &a, int node, MssKid k, double total, RowsShared &sh) {
  const gse_mss_batch &b = a.b;
  const int V = (int)b.vocab, tid = threadIdx.x;
  double *p = b.p + (int64_t)node * b.p_ld;
  const size_t o = (size_t)(node - a.node0) * a.rs.ns;
  for (;;) {
    __syncthreads();  // (p is written)
    const double px = p[k.x];
    if (mss_accepts(b, node, k, total > 0.0 ? px / total : px)) {
      if (tid == 0) mss_out(b, node, k.x, k.r);
      return;
    }
    __syncthreads();  // every thread has read p[x] before it changes
    const double *q = k.q ? k.q : p;  // (one-hot: a load that is dropped)
    for (int s = 0; s < a.rs.ns; ++s) {
      slice_sum(a.rs, s, V, [&](int t) { return MssTok<1>{p[t], {q[t]}}; },
                [&](int t, const MssTok<1> &m) {
                  return p[t] = residual(total > 0.0 ? m.p / total : m.p, k, m.q[0], t);
                },
                a.seg + (o + s) * RSEG, a.sum + o + s, a.last + o + s, sh);
    }
    total = row_total(a.sum + o, a.rs.ns);
    k = kid_from(b, node, k.r + 1);
    if (k.r < 0) break;
  }
  if (tid >= WAVE) return;
  const int j = row_draw(a.rs, V, uniform64(mix64(b.seed[node], SALT_RES), b.idx[node]), total, a.sum + o,
                         a.seg + o * RSEG, a.last + o, [&](int t) { return p[t]; });
  if (tid == 0) mss_out(b, node, j, -1);
}

// (at least three waves per SIMD: without the bound mss_rest's registers leave two, and 64 nodes of 151936 with three kids
// rejected take 137 us instead of 128)
template <int D>
__global__ __launch_bounds__(RT) __attribute__((amdgpu_waves_per_eu(3, 8))) void mss_kernel(MssArgs a) {
  __shared__ RowsShared sh;
  const gse_mss_batch &b = a.b;
  const int s = blockIdx.x, n = blockIdx.y, node = a.node0 + n, tid = threadIdx.x;
  const int V = (int)b.vocab;
  TreeNode &nd = a.st[n];
  double *p = b.p + (int64_t)node * b.p_ld;
  if (D > 1 && nd.next != (uint32_t)D) return;  // (level 1 runs for every node and sets next)
  MssKid k[MSS_LEVELS];
  double sig[MSS_LEVELS + 1] = {};
  bool any = true;
#pragma unroll
  for (int d = 0; d < MSS_LEVELS; ++d) k[d] = MssKid{-1, -1, nullptr};
  if constexpr (D >= 1) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      k[d] = kid_from(b, node, d > 0 ? k[d - 1].r + 1 : 0);
      if (d > 0) sig[d] = nd.sig[d];
    }
  }
  if constexpr (D == 1) {
    any = k[0].r >= 0;
    // kid 0 (every slice makes the same test; slice 0 writes the answer)
    if (any && mss_accepts(b, node, k[0], p[k[0].x])) {
      if (s == 0 && tid == 0) {
        mss_out(b, node, k[0].x, k[0].r);
        nd.next = 0;
      }
      return;
    }
  }
  const size_t o = (size_t)n * a.rs.ns;
  double *seg = a.seg + (o + s) * RSEG;
  if (any)
    slice_sum(a.rs, s, V, [&](int t) { return mss_load<D>(p, k, t); },
              [&](int t, const MssTok<D> &m) { return level<D>(k, sig, m.p, m.q, t); }, seg, a.sum + o + s,
              a.last + o + s, sh);
  else  // no kids: draw(p)
    slice_sum(a.rs, s, V, [&](int t) { return p[t]; }, [](int, double v) { return v; }, seg, a.sum + o + s,
              a.last + o + s, sh);
  if (tid == 0) sh.ticket = ticket_add(&nd.ticket);
  __syncthreads();
  if (sh.ticket != (uint32_t)(a.rs.ns - 1)) return;
  // the node's last slice
  const double total = row_total(a.sum + o, a.rs.ns);
  if (tid == 0) {
    nd.ticket = 0;
    nd.next = 0;
  }
  auto at = [&](int t) {
    if (!any) return p[t];
    const MssTok<D> m = mss_load<D>(p, k, t);
    return level<D>(k, sig, m.p, m.q, t);
  };
  const MssKid kn = any ? kid_from(b, node, k[D - 1].r + 1) : MssKid{-1, -1, nullptr};
  if (kn.r >= 0) {
    const double r = at(kn.x);
    if (mss_accepts(b, node, kn, total > 0.0 ? r / total : r)) {
      if (tid == 0) mss_out(b, node, kn.x, kn.r);
      return;
    }
    if constexpr (D < MSS_LEVELS) {
      if (tid == 0) {
        nd.sig[D] = total;
        nd.next = (uint32_t)(D + 1);
      }
    } else {
      __syncthreads();  // (every wave has read p[kn.x], which the loop writes)
      for (uint32_t t0 = 0; t0 < (uint32_t)V; t0 += 4 * RT) {
        MssTok<D> m[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = mss_load<D>(p, k, (int)min(t0 + i * RT + tid, (uint32_t)V - 1u));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t t = t0 + i * RT + tid;
          if (t < (uint32_t)V) p[t] = level<D>(k, sig, m[i].p, m[i].q, (int)t);
        }
      }
      mss_rest(a, node, kn, total, sh);  // (tests kid kn once more: the same answer)
    }
    return;
  }
  if (tid >= WAVE) return;
  const int j = row_draw(a.rs, V, uniform64(mix64(b.seed[node], SALT_RES), b.idx[node]), total, a.sum + o,
                         a.seg + o * RSEG, a.last + o, at);
  if (tid == 0) mss_out(b, node, j, -1);
}

// ---- a slice of a row of logits in registers ---------------------------------------------------------------------------
// Thread tid holds RE tokens of its slice: vector v of VEC consecutive tokens at s0 + (v RT + tid) VEC, so that a wave's
// vector is one segment of 64 VEC tokens. Rows whose start is 16-byte aligned (AL) read whole vectors.
constexpr int RE = RS / RT;
template <int DT>
struct RLay {
  static constexpr int VEC = DT == GSE_BF16 ? 8 : 4, NV = RE / VEC, SEG = WAVE * VEC, NSEG = RS / SEG;
};

template <int DT, bool AL>
__device__ __forceinline__ void load_vec(const char *base, uint32_t t0, int V, float *x) {
  using L = RLay<DT>;  // (t0 unsigned: it may lie past the end of a row of nearly 2^31 tokens)
  if (AL && t0 + L::VEC <= (uint32_t)V) {
    if constexpr (DT == GSE_BF16) {
      const uint4 u = *reinterpret_cast<const uint4 *>(base + (size_t)t0 * 2);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(w[i] << 16);
        x[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
      }
    } else {
      const float4 f = *reinterpret_cast<const float4 *>(base + (size_t)t0 * 4);
      x[0] = f.x;
      x[1] = f.y;
      x[2] = f.z;
      x[3] = f.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < L::VEC; ++e) {
      const uint32_t t = min(t0 + e, (uint32_t)V - 1u);
      float f;
      if constexpr (DT == GSE_BF16) f = bf16_to_f32(((const uint16_t *)base)[t]);
      else f = ((const float *)base)[t];
      x[e] = t0 + e < (uint32_t)V ? f : -INFINITY;
    }
  }
}

template <int DT>
__device__ __forceinline__ double logit_at(const char *base, int t) {
  if constexpr (DT == GSE_BF16) return (double)bf16_to_f32(((const uint16_t *)base)[t]);
  else return (double)((const float *)base)[t];
}

// ---- pick: spec.py:151-159 -------------------------------------------------------------------------------------------
// t > 0: n draws from softmax(x / t). A slice takes its own maximum m of z = x / t and the exact fixed-point masses
// exp(z - m) of its segments in one read; the row's last slice scales the slices' masses by exp(m - M) (M the row's
// maximum), in slice order, and its waves make the draws: crossing slice, crossing segment, crossing token.
// t == 0: the n best in stable descending order. A wave's n-th largest lane maximum bounds its n-th largest element from
// below, so the elements at or above it (n and a few) go to a list in LDS and are ranked by counting; the row's last
// workgroup ranks the others' bests the same way. One launch: 64 bf16 rows of 128256 tokens,
// n = 4, take 13.3 us (106 us with n rounds of a wave-wide 64-bit maximum over every element and a bitonic merge), two draws
// of 32 f32 rows of 32000 tokens 11.6 us (45 us as three launches: maximum, masses, draws).
constexpr uint64_t SALT_DRAFT = 1ull << 42;
constexpr int TOPL = GSE_MAX_KIDS * RE;  // list entries of a wave, at most (n lanes of RE elements)

struct PickArgs {
  gse_pick_batch b;
  int ns;
  double *max;      // [rows][ns] slice maxima of z
  Fx *mass, *seg;   // [rows][ns], [rows][ns][NSEG]: masses exp(z - slice maximum)
  int32_t *last;    // [rows][ns] last token with a positive mass
  uint64_t *top;    // [rows][ns][GSE_MAX_KIDS] packed (key, id), descending, 0 pads
  uint32_t *tick;   // [rows]
};

struct PickShared {
  union {
    uint64_t list[RW][TOPL];
    struct {
      uint64_t shi[RW], slo[RW];
      float mx[RW];
      int last[RW];
    } d;
  };
  uint64_t best[GSE_MAX_KIDS];
  uint32_t cnt[RW];
  uint32_t ticket;
  double etab[64];
};

// The n-th largest of the lanes' packed keys (token ids below 2^21); 0 when fewer than n lanes hold one.
__device__ __forceinline__ uint64_t wave_kth_packed(uint64_t v, int n) {
  auto enough = [&](uint64_t c) { return (int)__popcll(ballot64(v >= c)) >= n; };
  uint64_t r = 0;
#pragma unroll 4
  for (int b = 63; b >= 32; --b)
    if (enough(r | 1ull << b)) r |= 1ull << b;
  if (!enough(r | 0xFFE00000ull)) return 0ull;
  r |= 0xFFE00000ull;
#pragma unroll 4
  for (int b = 20; b >= 0; --b)
    if (enough(r | 1ull << b)) r |= 1ull << b;
  return r;
}

// Ranks the waves' lists against each other: sh.best[0, n) = the n largest listed, descending (0 pads). c: this wave's
// list length. Barriers before (the lists) and after.
__device__ __forceinline__ void rank_lists(uint32_t c, int n, PickShared &sh) {
  const int tid = threadIdx.x, w = tid >> 6;
  if (lane_id() == 0) sh.cnt[w] = c;
  if (tid < GSE_MAX_KIDS) sh.best[tid] = 0ull;
  __syncthreads();
  for (uint32_t i = lane_id(); i < c; i += WAVE) {
    const uint64_t x = sh.list[w][i];
    int r = 0;
#pragma unroll 1
    for (int q = 0; q < RW; ++q) {
      const uint32_t m = sh.cnt[q];
#pragma unroll 4
      for (uint32_t j = 0; j < m; ++j) r += sh.list[q][j] > x ? 1 : 0;
    }
    if (r < n) sh.best[r] = x;
  }
  __syncthreads();
}

// sh.best[0, n): the n largest of the workgroup's packed keys v (0: none), descending.
__device__ __forceinline__ void top_packed(const uint64_t (&v)[RE], int n, PickShared &sh) {
  const int w = threadIdx.x >> 6;
  uint64_t lm = 0;
#pragma unroll
  for (int i = 0; i < RE; ++i) lm = v[i] > lm ? v[i] : lm;
  uint64_t thr = wave_kth_packed(lm, n);
  thr = thr ? thr : 1ull;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < RE; ++i) {
    const uint64_t bl = ballot64(v[i] >= thr);
    if (bl) {
      if (v[i] >= thr) sh.list[w][c + lanes_below(bl)] = v[i];
      c += (uint32_t)__popcll(bl);
    }
  }
  rank_lists(c, n, sh);
}

// A wave's n best tokens among its NV vectors from s0 on, one wave-wide maximum per token (read again each time): for a
// wave whose elements at its threshold do not fit its list (many ties) or that has no threshold.
template <int DT, bool AL>
__device__ __noinline__ uint32_t top_by_rounds(const char *base, int s0, int V, int nv, int n, uint64_t *list) {
  using L = RLay<DT>;
  uint64_t prev = ~0ull;
  uint32_t c = 0;
  for (; c < (uint32_t)n; ++c) {
    uint64_t m = 0;
    for (int v = 0; v < nv; ++v) {
      const int t0 = s0 + (v * RT + (int)threadIdx.x) * L::VEC;
      float x[L::VEC];
      load_vec<DT, AL>(base, t0, V, x);
#pragma unroll
      for (int e = 0; e < L::VEC; ++e) {
        const uint64_t k = t0 + e < V ? pack(fkey(x[e]), (uint32_t)(t0 + e)) : 0ull;
        m = k < prev && k > m ? k : m;
      }
    }
    m = wave_max_u64(m);
    if (!m) break;
    if (lane_id() == 0) list[c] = m;
    prev = m;
  }
  return c;
}

// sh.best[0, n): the packed keys of the n best tokens of the slice of NV vectors a thread from s0 on. A wave lists the
// elements from the upper 16 key bits of its n-th largest lane maximum on: one maximum and one comparison per element.
template <int DT, bool AL, int NV>
__device__ __forceinline__ void top_tokens(const char *base, int s0, int V, int n, PickShared &sh) {
  using L = RLay<DT>;
  const int tid = threadIdx.x, w = tid >> 6;
  float x[NV * L::VEC];
#pragma unroll
  for (int v = 0; v < NV; ++v) load_vec<DT, AL>(base, s0 + (v * RT + tid) * L::VEC, V, &x[v * L::VEC]);
  float lm = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV * L::VEC; ++i) lm = fmaxf(lm, x[i]);
  const uint32_t thr = wave_kth_largest_u16(fkey(lm) >> 16, n) << 16;
  uint32_t c = TOPL + 1;
  if (thr > KEY_NEGINF) {
    const float xt = fkey_inv(thr);
    c = 0;
#pragma unroll
    for (int i = 0; i < NV * L::VEC; ++i) {
      const uint64_t bl = ballot64(x[i] >= xt);
      if (bl) {
        const uint32_t pos = c + lanes_below(bl);
        if (x[i] >= xt && pos < (uint32_t)TOPL)
          sh.list[w][pos] = pack(fkey(x[i]), (uint32_t)(s0 + (i / L::VEC * RT + tid) * L::VEC + i % L::VEC));
        c += (uint32_t)__popcll(bl);
      }
    }
  }
  if (c > (uint32_t)TOPL) c = top_by_rounds<DT, AL>(base, s0, V, NV, n, sh.list[w]);
  rank_lists(c, n, sh);
}

// Draw kd of a row whose slices are summed, by one wave.
template <int DT>
__device__ __forceinline__ void pick_draw(const PickArgs &a, int row, int kd, const char *base, double t,
                                          const double *etab) {
  using L = RLay<DT>;
  const int lane = lane_id();
  const size_t o = (size_t)row * a.ns;
  const double *mx = a.max + o;
  const Fx *ms = a.mass + o;
  double M = -INFINITY;
  for (int j = lane; j < a.ns; j += WAVE) M = fmax(M, ld_ag(&mx[j]));
  M = lane63(wave_scan(M, (double)-INFINITY, [](double p, double q) { return fmax(p, q); }));
  int tok = -1;
  double lq = __builtin_nan("");
  if (fabs(M) < INFINITY) {
    auto weight = [&](int j) {
      const double m = ld_ag(&mx[j]);
      const Fx f{ld_ag(&ms[j].hi), ld_ag(&ms[j].lo)};
      return m > -INFINITY ? fx_val(f) * exp_nonpos(m - M, etab) : 0.0;
    };
    double E = 0.0;
    int last = -1;
    for (int j0 = 0; j0 < a.ns; j0 += WAVE) {
      const int j = j0 + lane;
      const double x = j < a.ns ? weight(j) : 0.0;
      if (x > 0.0) last = max(last, ld_ag(&a.last[o + j]));
      E += wave_sum_f64(x);
    }
    last = (int)wave_max_u32((uint32_t)(last + 1)) - 1;
    const double thr = uniform64(mix64(a.b.seed[row], SALT_DRAFT + (uint64_t)kd), a.b.at[row]) * E;
    double before = 0.0;
    int lp;
    const int sx = cross(a.ns, thr, before, lp, weight);
    tok = thr > 0.0 ? last : 0;  // (u = 0 draws the first token, whatever its mass)
    if (thr > 0.0 && sx >= 0) {
      const double m = ld_ag(&mx[sx]), sc = exp_nonpos(m - M, etab);
      // the threshold in the slice's own masses (positive: a token of mass 0 never reaches it)
      const double ts = fmax((thr - before) / sc, 0x1p-1000);
      const Fx *sg = a.seg + (o + sx) * (RSEG / 2);
      Fx f = lane < L::NSEG ? Fx{ld_ag(&sg[lane].hi), ld_ag(&sg[lane].lo)} : Fx{0, 0};
      Fx inc{wave_incl_scan_u64(f.hi), wave_incl_scan_u64(f.lo)};
      uint64_t hit = ballot64(lane < L::NSEG && fx_val(inc) >= ts);
      tok = min(ld_ag(&a.last[o + sx]), last);  // (none: the slice's last token of positive mass)
      if (hit) {
        const int g = (int)__builtin_ctzll(hit);
        const Fx b0{shfl_u64(inc.hi - f.hi, g), shfl_u64(inc.lo - f.lo, g)};
        // the segment's masses again: lane l's VEC consecutive tokens
        const int t0 = sx * RS + g * L::SEG + lane * L::VEC, V = (int)a.b.vocab;
        Fx e[L::VEC], s{0, 0};
#pragma unroll
        for (int k = 0; k < L::VEC; ++k) {
          const double z = logit_at<DT>(base, min(t0 + k, V - 1)) / t;
          e[k] = t0 + k < V ? fx_of(exp_nonpos(z - m, etab)) : Fx{0, 0};
          s = fx_add(s, e[k]);
        }
        Fx run = fx_add(b0, Fx{wave_incl_scan_u64(s.hi) - s.hi, wave_incl_scan_u64(s.lo) - s.lo});
        int at = -1;
#pragma unroll
        for (int k = 0; k < L::VEC; ++k) {
          run = fx_add(run, e[k]);
          if (at < 0 && fx_val(run) >= ts) at = t0 + k;
        }
        hit = ballot64(at >= 0);
        if (hit) tok = min(__shfl(at, (int)__builtin_ctzll(hit), WAVE), last);
      }
    }
    if (tok >= 0) lq = (logit_at<DT>(base, tok) / t - M) - log(E);
  }
  if (lane == 0) {
    a.b.out_tokens[(int64_t)row * a.b.out_ld + kd] = tok;
    a.b.out_logq[(int64_t)row * a.b.out_ld + kd] = lq;
  }
}

// The masses of one slice of a t > 0 row (slice index o over the rows' slices).
template <int DT, bool AL>
__device__ __forceinline__ void pick_masses(const PickArgs &a, const char *base, int s0, size_t o, double t,
                                            PickShared &sh) {
  using L = RLay<DT>;
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6, V = (int)a.b.vocab;
  float x[RE];
#pragma unroll
  for (int v = 0; v < L::NV; ++v) load_vec<DT, AL>(base, s0 + (v * RT + tid) * L::VEC, V, &x[v * L::VEC]);
  float xm = -INFINITY;
#pragma unroll
  for (int i = 0; i < RE; ++i) xm = fmaxf(xm, x[i]);
  xm = wave_max_f32(xm);
  if (lane == 0) sh.d.mx[w] = xm;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < RW; ++k) xm = fmaxf(xm, sh.d.mx[k]);
  // (z = x / t is monotone in x and rounds once: the maximum of z is that of x divided)
  const double m = t == 1.0 ? (double)xm : (double)xm / t;
  int last = -1;
  Fx tot{0, 0};
#pragma unroll
  for (int v = 0; v < L::NV; ++v) {
    Fx f{0, 0};
#pragma unroll
    for (int e = 0; e < L::VEC; ++e) {
      const double xd = (double)x[v * L::VEC + e], z = t == 1.0 ? xd : xd / t;
      const double y = exp_nonpos(z - m, sh.etab);  // (0 for NaN and -inf)
      f = fx_add(f, fx_of(y));
      if (y > 0.0) last = s0 + (v * RT + tid) * L::VEC + e;
    }
    const Fx g{wave_sum_u64(f.hi), wave_sum_u64(f.lo)};
    tot = fx_add(tot, g);
    if (lane == 0) {  // segment v RW + w
      Fx *sg = a.seg + o * (RSEG / 2) + v * RW + w;
      st_ag(&sg->hi, g.hi);
      st_ag(&sg->lo, g.lo);
    }
  }
  last = (int)wave_max_u32((uint32_t)(last + 1)) - 1;
  if (lane == 0) {
    sh.d.shi[w] = tot.hi;
    sh.d.slo[w] = tot.lo;
    sh.d.last[w] = last;
  }
  __syncthreads();
  if (tid == 0) {
    Fx f{0, 0};
    int l = -1;
    for (int k = 0; k < RW; ++k) {
      f = fx_add(f, Fx{sh.d.shi[k], sh.d.slo[k]});
      l = max(l, sh.d.last[k]);
    }
    st_ag(&a.max[o], m);
    st_ag(&a.mass[o].hi, f.hi);
    st_ag(&a.mass[o].lo, f.lo);
    st_ag(&a.last[o], l);
  }
}

// A workgroup takes SUB slices of its row: the slices of a t > 0 row one after the other, of a t == 0 row all at once.
template <int DT, bool AL, int SUB>
__global__ __launch_bounds__(RT) void pick_kernel(PickArgs a) {
  using L = RLay<DT>;
  __shared__ PickShared sh;
  const int s = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, w = tid >> 6;
  const int V = (int)a.b.vocab, ng = (int)gridDim.x;
  const char *base = (const char *)a.b.x + (size_t)row * (size_t)a.b.ld * (DT == GSE_BF16 ? 2 : 4);
  const double t = a.b.temperature[row];
  const int n = min(max(a.b.n[row], 0), (int)min((int64_t)GSE_MAX_KIDS, a.b.out_ld));
  if (n == 0) return;
  if (tid < 64) sh.etab[tid] = EXP2_64[tid];  // (published by the first barrier)
  const bool drawn = t > 0.0;
  uint64_t *top = a.top + (size_t)row * a.ns * GSE_MAX_KIDS;
  if (drawn) {
    for (int j = s * SUB; j < min((s + 1) * SUB, a.ns); ++j) {
      if (j > s * SUB) __syncthreads();  // (the LDS of the slice before)
      pick_masses<DT, AL>(a, base, j * RS, (size_t)row * a.ns + j, t, sh);
    }
  } else {
    top_tokens<DT, AL, SUB * L::NV>(base, s * SUB * RS, V, n, sh);
    if (tid < n) st_ag(&top[s * GSE_MAX_KIDS + tid], sh.best[tid]);
  }
  store_wait();
  __syncthreads();
  if (tid == 0) sh.ticket = ticket_add(&a.tick[row]);
  __syncthreads();
  if (sh.ticket != (uint32_t)(ng - 1)) return;
  // the row's last workgroup
  if (tid == 0) a.tick[row] = 0;
  if (drawn) {
    for (int kd = w; kd < n; kd += RW) pick_draw<DT>(a, row, kd, base, t, sh.etab);
    return;
  }
  const int N = ng * n;  // entry i: the (i % n)-th best of workgroup i / n
  for (int i0 = 0; i0 < N; i0 += RT * (RE - 1)) {  // (the last element of each thread carries the best so far)
    uint64_t v[RE];
#pragma unroll
    for (int k = 0; k < RE; ++k) {
      const int i = i0 + k * RT + tid;
      v[k] = 0ull;
      if (k == RE - 1) v[k] = i0 > 0 && tid < n ? sh.best[tid] : 0ull;
      else if (i0 + k * RT < N && i < N) v[k] = ld_ag(&top[(size_t)(i / n) * GSE_MAX_KIDS + i % n]);
    }
    __syncthreads();
    top_packed(v, n, sh);
  }
  if (tid < n) {
    const uint64_t pk = sh.best[tid];
    const int id = pk ? (int)pk_id(pk) : -1;
    a.b.out_tokens[(int64_t)row * a.b.out_ld + tid] = id;
    a.b.out_logq[(int64_t)row * a.b.out_ld + tid] = id >= 0 ? logit_at<DT>(base, id) : __builtin_nan("");
  }
}

// ---- q of a drafter row: spec.py:157 (q = softmax(float64(x) / t)) -----------------------------------------------------
// Two launches over the slices: each slice's maximum m of z = x / t and mass E_s = sum exp(z - m) (exact fixed point,
// exp_nonpos within 1.5 ulp), one read; then M = max m and E = sum E_s exp(m - M) from the row's slices, in slice order,
// by every workgroup, and q = exp(z - M) / E. A row holding NaN, +inf, or no value above -inf gives NaN everywhere, as
// torch.softmax does. 32 f32 rows of 32000 tokens: 39 us with one workgroup of 1024 threads per row in three passes, 32 of
// the 256 CUs busy; sliced 12.0 us (4.4 + 7.6).
struct QprobArgs {
  gse_qrows q;
  int V, row0;
  RowSlices rs;
  double *out;
  int64_t ld;
  double *max, *mass;  // [rows][ns] (a slice holding NaN: its maximum is NaN)
};

struct QprobShared {
  float mx[RW];
  uint64_t hi[RW], lo[RW];
  uint32_t nan[RW];
  double M, E;
  double etab[64];
};

template <int DT, bool AL>
__global__ __launch_bounds__(RT) void qstats_kernel(QprobArgs a) {
  using L = RLay<DT>;
  __shared__ QprobShared sh;
  const int s = blockIdx.x, r = blockIdx.y, row = a.row0 + r, tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const char *base = (const char *)a.q.q + (size_t)row * (size_t)a.q.ld * (DT == GSE_BF16 ? 2 : 4);
  const double t = a.q.temperature[row];
  if (tid < 64) sh.etab[tid] = EXP2_64[tid];
  double M = -INFINITY, E = 0.0;
  for (int c = 0; c < a.rs.sub; ++c) {  // (one slice, unless the workspace's slices widen)
    const uint32_t s0 = (uint32_t)(s * a.rs.sub + c) * RS;
    if (s0 >= (uint32_t)a.V) break;
    float x[RE], xm = -INFINITY;
    bool nan = false;
#pragma unroll
    for (int v = 0; v < L::NV; ++v) load_vec<DT, AL>(base, s0 + (v * RT + tid) * L::VEC, a.V, &x[v * L::VEC]);
#pragma unroll
    for (int i = 0; i < RE; ++i) {
      xm = fmaxf(xm, x[i]);
      nan |= x[i] != x[i];
    }
    xm = wave_max_f32(xm);
    const bool wnan = ballot64(nan) != 0ull;
    __syncthreads();  // (the LDS of the slice before)
    if (lane == 0) {
      sh.mx[w] = xm;
      sh.nan[w] = wnan ? 1u : 0u;
    }
    __syncthreads();
    uint32_t bad = 0;
#pragma unroll
    for (int k = 0; k < RW; ++k) {
      xm = fmaxf(xm, sh.mx[k]);
      bad |= sh.nan[k];
    }
    const double m = bad ? __builtin_nan("") : (double)xm / t;  // (z is monotone in x and rounds once)
    Fx f{0, 0};
    if (fabs(m) < INFINITY) {
#pragma unroll
      for (int i = 0; i < RE; ++i) f = fx_add(f, fx_of(exp_nonpos((double)x[i] / t - m, sh.etab)));
    }
    f.hi = wave_sum_u64(f.hi);
    f.lo = wave_sum_u64(f.lo);
    if (lane == 0) {
      sh.hi[w] = f.hi;
      sh.lo[w] = f.lo;
    }
    __syncthreads();
    Fx tot{0, 0};
#pragma unroll
    for (int k = 0; k < RW; ++k) tot = fx_add(tot, Fx{sh.hi[k], sh.lo[k]});
    const double e = fx_val(tot);
    if (m != m || M != M) {
      M = __builtin_nan("");
    } else if (m > M) {
      E = (M > -INFINITY ? E * exp_nonpos(M - m, sh.etab) : 0.0) + e;
      M = m;
    } else if (m > -INFINITY) {
      E += e * exp_nonpos(m - M, sh.etab);
    }
  }
  if (tid == 0) {
    a.max[(size_t)r * a.rs.ns + s] = M;
    a.mass[(size_t)r * a.rs.ns + s] = E;
  }
}

template <int DT, bool AL>
__global__ __launch_bounds__(RT) void qprob_kernel(QprobArgs a) {
  using L = RLay<DT>;
  __shared__ QprobShared sh;
  const int s = blockIdx.x, r = blockIdx.y, row = a.row0 + r, tid = threadIdx.x, lane = lane_id();
  const char *base = (const char *)a.q.q + (size_t)row * (size_t)a.q.ld * (DT == GSE_BF16 ? 2 : 4);
  const double t = a.q.temperature[row];
  double *o = a.out + (int64_t)row * a.ld;
  if (tid < 64) sh.etab[tid] = EXP2_64[tid];
  __syncthreads();
  if (tid < WAVE) {  // the row's M and E
    const double *mx = a.max + (size_t)r * a.rs.ns, *ms = a.mass + (size_t)r * a.rs.ns;
    double M = -INFINITY, E = 0.0;
    bool bad = false;
    for (int j = lane; j < a.rs.ns; j += WAVE) {
      bad |= mx[j] != mx[j];
      M = fmax(M, mx[j]);
    }
    M = lane63(wave_scan(M, (double)-INFINITY, [](double p, double q) { return fmax(p, q); }));
    if (ballot64(bad) != 0ull || !(fabs(M) < INFINITY)) M = __builtin_nan("");
    for (int j0 = 0; j0 < a.rs.ns; j0 += WAVE) {
      const int j = j0 + lane;
      E += wave_sum_f64(j < a.rs.ns && mx[j] > -INFINITY ? ms[j] * exp_nonpos(mx[j] - M, sh.etab) : 0.0);
    }
    if (lane == 0) {
      sh.M = M;
      sh.E = E;
    }
  }
  // (the slice's loads overlap the row's sums)
  for (int c = 0; c < a.rs.sub; ++c) {
    const uint32_t s0 = (uint32_t)(s * a.rs.sub + c) * RS;
    if (s0 >= (uint32_t)a.V) break;
    float x[RE];
#pragma unroll
    for (int v = 0; v < L::NV; ++v) load_vec<DT, AL>(base, s0 + (v * RT + tid) * L::VEC, a.V, &x[v * L::VEC]);
    if (c == 0) __syncthreads();
    const double M = sh.M, E = sh.E;
#pragma unroll
    for (int v = 0; v < L::NV; ++v) {
      const uint32_t t0 = s0 + (v * RT + tid) * L::VEC;
#pragma unroll
      for (int e = 0; e < L::VEC; ++e) {
        const double q = M != M ? M : exp_nonpos((double)x[v * L::VEC + e] / t - M, sh.etab) / E;
        if (t0 + e < (uint32_t)a.V) o[t0 + e] = q;
      }
    }
  }
}

// The slicing of rows of V tokens, and the rows that one launch takes (at least 1) of the workspace's R rows of S slices.
RowSlices slices_of(const RowsWs &w, int V, int *rows) {
  const int64_t cap = (int64_t)w.rows * w.slices;
  int64_t ns = ((int64_t)V + RS - 1) / RS, sub = 1;
  if (ns > cap) {
    sub = (ns + cap - 1) / cap;
    ns = (V + RS * sub - 1) / (RS * sub);
  }
  *rows = (int)min(min(cap / ns, (int64_t)w.rows), (int64_t)65535);
  return RowSlices{(int)ns, (int)sub};
}

}  // namespace

hipError_t launch_draw(const RowsWs &w, const double *q, int64_t ld, int rows, int V, const double *u, int32_t *out,
                       hipStream_t s) {
  DrawArgs a;
  a.q = q;
  a.ld = ld;
  a.V = V;
  a.u = u;
  a.out = out;
  a.sum = w.sum;
  a.seg = w.seg;
  a.last = w.last;
  a.tick = w.tick;
  int per;
  a.rs = slices_of(w, V, &per);
  for (a.row0 = 0; a.row0 < rows; a.row0 += per)
    hipLaunchKernelGGL(draw_kernel, dim3(a.rs.ns, min(per, rows - a.row0)), dim3(RT), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_mss(const RowsWs &w, const gse_mss_batch &b, hipStream_t s) {
  MssArgs a;
  a.b = b;
  a.st = w.st;
  a.sum = w.sum;
  a.seg = w.seg;
  a.last = w.last;
  int per;
  a.rs = slices_of(w, (int)b.vocab, &per);
  const int nodes = (int)b.nodes;
  for (a.node0 = 0; a.node0 < nodes; a.node0 += per) {
    const dim3 grid(a.rs.ns, min(per, nodes - a.node0)), block(RT);
    hipLaunchKernelGGL(mss_kernel<1>, grid, block, 0, s, a);
    if (b.max_kids > 1) hipLaunchKernelGGL(mss_kernel<2>, grid, block, 0, s, a);
    if (b.max_kids > 2) hipLaunchKernelGGL(mss_kernel<3>, grid, block, 0, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_pick(const RowsWs &w, const gse_pick_batch &b, hipStream_t s) {
  PickArgs a;
  a.b = b;
  a.ns = ((int)b.vocab + RS - 1) / RS;  // (at most w.slices, and at most w.rows rows: the caller's checks)
  a.max = w.sum;
  a.mass = w.mass;
  a.seg = (Fx *)w.seg;
  a.last = w.last;
  a.top = w.top;
  a.tick = w.tick;
  // whole 16-byte vectors when every row starts on a 16-byte boundary
  const bool al = ((((uintptr_t)b.x) | ((uintptr_t)b.ld * (b.dtype == GSE_BF16 ? 2u : 4u))) & 15u) == 0;
  // One slice per workgroup while the call's slices fit the device at once (four workgroups per CU), else four: every
  // workgroup ends with the same chain (list, ranks, store, ticket), so past one round the longer ones win.
  const bool wide = (int64_t)a.ns * b.rows > w.round;
  auto go = [&](auto dt, auto aligned, auto sub) {
    constexpr int SUB = decltype(sub)::value;
    hipLaunchKernelGGL((pick_kernel<decltype(dt)::value, decltype(aligned)::value, SUB>),
                       dim3((a.ns + SUB - 1) / SUB, b.rows), dim3(RT), 0, s, a);
  };
  auto by_sub = [&](auto dt, auto aligned) {
    if (wide) go(dt, aligned, std::integral_constant<int, 4>{});
    else go(dt, aligned, std::integral_constant<int, 1>{});
  };
  auto by_al = [&](auto dt) {
    if (al) by_sub(dt, std::true_type{});
    else by_sub(dt, std::false_type{});
  };
  if (b.dtype == GSE_BF16) by_al(std::integral_constant<int, (int)GSE_BF16>{});
  else by_al(std::integral_constant<int, (int)GSE_F32>{});
  return hipGetLastError();
}

hipError_t launch_qprob(const RowsWs &w, const gse_qrows &q, int V, double *out, int64_t ld, hipStream_t s) {
  QprobArgs a;
  a.q = q;
  a.V = V;
  a.out = out;
  a.ld = ld;
  a.max = w.sum;
  a.mass = w.seg;
  int per;
  a.rs = slices_of(w, V, &per);
  const int rows = (int)q.rows;
  const bool bf = q.kind == GSE_Q_LOGITS_BF16;
  const bool al = ((((uintptr_t)q.q) | ((uintptr_t)q.ld * (bf ? 2u : 4u))) & 15u) == 0;
  auto go = [&](auto dt, auto aligned) {
    constexpr int DT = decltype(dt)::value;
    constexpr bool AL = decltype(aligned)::value;
    for (a.row0 = 0; a.row0 < rows; a.row0 += per) {
      const dim3 grid(a.rs.ns, min(per, rows - a.row0)), block(RT);
      hipLaunchKernelGGL((qstats_kernel<DT, AL>), grid, block, 0, s, a);
      hipLaunchKernelGGL((qprob_kernel<DT, AL>), grid, block, 0, s, a);
    }
  };
  auto by_al = [&](auto dt) {
    if (al) go(dt, std::true_type{});
    else go(dt, std::false_type{});
  };
  if (bf) by_al(std::integral_constant<int, (int)GSE_BF16>{});
  else by_al(std::integral_constant<int, (int)GSE_F32>{});
  return hipGetLastError();
}

}  // namespace gse
