// Row passes: selection work on whole rows of probabilities, each row spread over slices of RS tokens so that a call of
// a few rows still fills the device. A slice's workgroup reads its tokens once, writes the slice's sums, and takes an
// atomic ticket; the row's last slice finishes the row in the same launch from the slices' sums (a draw reads the
// crossing slice's 64 segment sums and then one segment: three dependent reads, not a pass over the row).
//
//   draw  sampling.py:100-104  inverse CDF in vocabulary order of fp64 rows
//   mss   spec.py:88-103       multi-step speculative sampling: one launch per residual level, at most MSS_LEVELS of them
//
// What bounds them: a slice is one round of coalesced 512-byte reads per wave (16 tokens a thread), so at the sizes of a
// decode step a launch is latency: load, sums, ticket, the last slice's reads. One workgroup per row, each thread summing
// a contiguous run (128 tokens at V = 128256: every load of a wave touched 64 cache lines, one CU per row), took 0.9 ms
// for 16 mss nodes of V = 128256 and two kids, 85 % of a dist + mss call (1014 us); sliced, that call takes 106 us.
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
  const int s0 = s * RS * rs.sub;
  int lst = -1;
  if (rs.sub == 1) {
    // eight segments' loads in flight at a time
#pragma unroll
    for (int h = 0; h < RGS; h += 8) {
      decltype(load(0)) r[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) r[k] = load(min(s0 + ((h + k) * RW + w) * WAVE + lane, V - 1));
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int g = (h + k) * RW + w, t = s0 + g * WAVE + lane;
        const double v = t < V ? ev(t, r[k]) : 0.0;
        if (v > 0.0) lst = t;
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
        const int t = s0 + (g * rs.sub + c) * WAVE + lane;
        const double v = t < V ? ev(t, load(t)) : 0.0;
        if (v > 0.0) lst = t;
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

// The first j in [0, n) whose inclusive prefix before + sum(v(0..j)) reaches thr, 64 values at a time; before becomes
// the prefix ahead of it. -1 when none does (before is then the whole sum).
template <typename VF>
__device__ __forceinline__ int cross(int n, double thr, double &before, VF v) {
  for (int j0 = 0; j0 < n; j0 += WAVE) {
    const int j = j0 + lane_id();
    const double x = j < n ? v(j) : 0.0;
    const double inc = before + wave_incl_scan_f64(x);
    const uint64_t hit = ballot64(j < n && inc >= thr);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      before = l > 0 ? shfl_f64(inc, l - 1) : before;
      return j0 + l;
    }
    before = shfl_f64(inc, WAVE - 1);
  }
  return -1;
}

// draw() of a row whose slices have been summed (by one wave; every lane gets it): the first token whose inclusive
// prefix reaches u * total, at most the last token with a positive weight; -1 when no weight is positive. A total that
// is NaN gives the first token (count(c < NaN) = 0). A prefix of tokens may round below the slice's own sum: the draw
// then takes the crossing segment's (or slice's) last token.
template <typename EW>
__device__ __forceinline__ int row_draw(const RowSlices &rs, int V, double u, double total, const double *sums,
                                        const double *segs, const int32_t *lasts, EW ev) {
  int lst = -1;
  for (int j = lane_id(); j < rs.ns; j += WAVE) lst = max(lst, ld_ag(&lasts[j]));
  lst = (int)wave_max_u32((uint32_t)(lst + 1)) - 1;
  if (lst < 0) return -1;
  const double thr = u * total;
  if (thr != thr) return 0;
  double before = 0.0;
  const int sx = cross(rs.ns, thr, before, [&](int j) { return ld_ag(&sums[j]); });
  if (sx < 0) return lst;
  const double *sg = segs + (size_t)sx * RSEG;
  const int g = cross(RSEG, thr, before, [&](int j) { return ld_ag(&sg[j]); });
  const int s1 = (sx + 1) * RS * rs.sub;
  if (g < 0) return min(min(s1, V) - 1, lst);
  const int t0 = (sx * RSEG + g) * WAVE * rs.sub, t1 = min(t0 + WAVE * rs.sub, V);
  const int k = cross(t1 - t0, thr, before, [&](int j) { return ev(t0 + j); });
  return min(k < 0 ? t1 - 1 : t0 + k, lst);
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

// The kids past level MSS_LEVELS, by one workgroup, in place in p (p: the distribution before kid k's test, written by
// this workgroup): the draw's sums are left in the node's workspace.
__device__ __noinline__ void mss_rest(const MssArgs &a, int node, MssKid k, RowsShared &sh) {
  const gse_mss_batch &b = a.b;
  const int V = (int)b.vocab, tid = threadIdx.x;
  double *p = b.p + (int64_t)node * b.p_ld;
  while (k.r >= 0) {
    const double px = p[k.x];
    if (mss_accepts(b, node, k, px)) {
      if (tid == 0) mss_out(b, node, k.x, k.r);
      return;
    }
    __syncthreads();  // every thread has read p[x] before it changes
    double s = 0.0;
    for (int t = tid; t < V; t += RT) {
      const double v = residual(p[t], k, k.q ? k.q[t] : 0.0, t);
      p[t] = v;
      s += v;
    }
    s = wave_sum_f64(s);
    if (lane_id() == 0) sh.red[tid >> 6] = s;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < RW; ++w) tot += sh.red[w];
    if (tot > 0.0)
      for (int t = tid; t < V; t += RT) p[t] = p[t] / tot;
    __syncthreads();
    k = kid_from(b, node, k.r + 1);
  }
  const size_t o = (size_t)(node - a.node0) * a.rs.ns;
  for (int s = 0; s < a.rs.ns; ++s) {
    slice_sum(a.rs, s, V, [&](int t) { return p[t]; }, [](int, double v) { return v; }, a.seg + (o + s) * RSEG,
              a.sum + o + s, a.last + o + s, sh);
  }
  if (tid >= WAVE) return;
  const double total = row_total(a.sum + o, a.rs.ns);
  const int j = row_draw(a.rs, V, uniform64(mix64(b.seed[node], SALT_RES), b.idx[node]), total, a.sum + o,
                         a.seg + o * RSEG, a.last + o, [&](int t) { return p[t]; });
  if (tid == 0) mss_out(b, node, j, -1);
}

template <int D>
__global__ __launch_bounds__(RT) void mss_kernel(MssArgs a) {
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
      for (int t = tid; t < V; t += RT) {
        const double v = at(t);
        p[t] = total > 0.0 ? v / total : v;
      }
      __syncthreads();
      mss_rest(a, node, kn, sh);  // (tests kid kn once more: the same answer)
    }
    return;
  }
  if (tid >= WAVE) return;
  const int j = row_draw(a.rs, V, uniform64(mix64(b.seed[node], SALT_RES), b.idx[node]), total, a.sum + o,
                         a.seg + o * RSEG, a.last + o, at);
  if (tid == 0) mss_out(b, node, j, -1);
}

// The slicing of rows of V tokens, and the rows that one launch takes (at least 1) of the workspace's R rows of S slices.
RowSlices slices_of(const RowsWs &w, int V, int *rows) {
  const int64_t cap = (int64_t)w.rows * w.slices;
  int64_t ns = (V + RS - 1) / RS, sub = 1;
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

}  // namespace gse
