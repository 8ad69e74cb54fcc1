// The rest of the selection call surface: dist (vocabulary-order fp64 probabilities) and the bool -> packed mask
// conversion.
#include "gse_rowctx.h"

namespace gse {

namespace {

constexpr int AT = 256;  // threads of the elementwise kernels

// ---- dist: sampling.py:88-97 -------------------------------------------------------------------------------------------
// out[t] = q_t * keep_t / sum(q * keep) with q = exp(z - z_max) / S; keep_t = packed(key_t, t) >= packed key of the last
// kept rank. Rows whose z holds +inf / NaN or whose maximum is -inf give NaN everywhere, as numpy does.
// A workgroup takes DSL tokens, DPT a thread, every load issued before the first is used: at the sizes of a step the launch
// is one round of loads, exponentials and stores (16 rows of 128256: 23.0 us with 8192 tokens a workgroup, a load at a time
// behind each element's branches; 9.6 us so). S Z is formed once, so an element takes one division.
constexpr int DPT = 8, DSL = AT * DPT;

__global__ __launch_bounds__(AT) void dist_kernel(ScanArgs a, double *probs, int64_t pld) {
  __shared__ uint32_t cnt[DSL];
  const int row = blockIdx.y, c0 = blockIdx.x * DSL, tid = threadIdx.x;
  const gse_row P = a.params[row];
  const RowCtx c = make_ctx(a, row, P);
  const RowInfo ri = a.info[row];
  double *out = probs + (int64_t)row * pld;
  const bool nan_row = !(ri.flags & R_DONE) || (ri.flags & (R_SPECIAL | R_BAD));
  float x[DPT];
  uint32_t mw[DPT];
#pragma unroll
  for (int k = 0; k < DPT; ++k) {
    const int t = min(c0 + k * AT + tid, c.V - 1);
    x[k] = load_one(c, t);
    mw[k] = c.mw ? c.mw[t >> 5] : 0xFFFFFFFFu;
  }
  if (c.pen && !nan_row) build_counts<DSL>(c, a.hist, c0, cnt);
  const double M = (double)fkey_inv(pk_key(ri.cmax)), SZ = ri.S * ri.Z;
#pragma unroll
  for (int k = 0; k < DPT; ++k) {
    const int t = c0 + k * AT + tid;
    bool fn = false, ff = false;
    float xm;
    const uint32_t key = elem_key(c, x[k], c.pen && !nan_row ? cnt[k * AT + tid] : 0u, (mw[k] >> (t & 31)) & 1u, fn, ff, xm);
    double v = 0.0;
    if (nan_row) v = __builtin_nan("");
    else if (pack(key, (uint32_t)t) >= ri.kkeep && key > KEY_NEGINF) v = exp((double)fkey_inv(key) - M) / SZ;
    if (t < c.V) out[t] = v;
  }
}

// ---- bool rows -> packed words (grammar.py:44-45 inverted) ---------------------------------------------------------------
__global__ __launch_bounds__(AT) void pack_kernel(const uint8_t *bools, int64_t bld, int V, int32_t *words, int64_t wld) {
  const int row = blockIdx.y;
  const int w = blockIdx.x * AT + threadIdx.x;
  const int nw = (V + 31) / 32;
  if (w >= nw) return;
  const uint8_t *src = bools + (int64_t)row * bld + (int64_t)w * 32;
  uint32_t v = 0;
  for (int k = 0; k < 32; ++k) {
    const int t = w * 32 + k;
    if (t < V && src[k]) v |= 1u << k;
  }
  words[(int64_t)row * wld + w] = (int32_t)v;
}

// ---- zero fill (a kernel, not hipMemsetAsync, so that a caller may capture it in a graph) ----------------------------
__global__ __launch_bounds__(AT) void zero_kernel(uint4 *p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * AT + threadIdx.x; i < n; i += (size_t)gridDim.x * AT) p[i] = make_uint4(0, 0, 0, 0);
}

}  // namespace

hipError_t launch_zero(void *p, size_t bytes, hipStream_t s) {
  const size_t n = bytes / sizeof(uint4);  // (bytes: a multiple of 256)
  const unsigned g = (unsigned)(n / AT < 4096 ? (n + AT - 1) / AT : 4096);
  if (n) hipLaunchKernelGGL(zero_kernel, dim3(g > 0 ? g : 1), dim3(AT), 0, s, (uint4 *)p, n);
  return hipGetLastError();
}

hipError_t launch_dist_write(const ScanArgs &a, double *probs, int64_t probs_ld, hipStream_t s) {
  hipLaunchKernelGGL(dist_kernel, dim3((a.V + DSL - 1) / DSL, a.rows), dim3(AT), 0, s, a, probs, probs_ld);
  return hipGetLastError();
}

hipError_t launch_pack(const uint8_t *bools, int64_t bld, int rows, int V, int32_t *words, int64_t wld, hipStream_t s) {
  const int nw = (V + 31) / 32;
  hipLaunchKernelGGL(pack_kernel, dim3((nw + AT - 1) / AT, rows), dim3(AT), 0, s, bools, bld, V, words, wld);
  return hipGetLastError();
}

}  // namespace gse
