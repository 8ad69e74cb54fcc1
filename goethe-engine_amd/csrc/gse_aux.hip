// The rest of the selection call surface: dist (vocabulary-order fp64 probabilities) and the bool -> packed mask
// conversion.
#include "gse_rowctx.h"

namespace gse {

namespace {

constexpr int AT = 256;  // threads of the elementwise kernels

// ---- dist: sampling.py:88-97 -------------------------------------------------------------------------------------------
// out[t] = q_t * keep_t / sum(q * keep) with q = exp(z - z_max) / S; keep_t = packed(key_t, t) >= packed key of the last
// kept rank. Rows whose z holds +inf / NaN or whose maximum is -inf give NaN everywhere, as numpy does.
__global__ __launch_bounds__(AT) void dist_kernel(ScanArgs a, double *probs, int64_t pld) {
  __shared__ uint32_t cnt[CH];
  const int row = blockIdx.y, chunk = blockIdx.x, c0 = chunk * CH;
  const gse_row P = a.params[row];
  const RowCtx c = make_ctx(a, row, P);
  const RowInfo ri = a.info[row];
  double *out = probs + (int64_t)row * pld;
  const bool nan_row = !(ri.flags & R_DONE) || (ri.flags & (R_SPECIAL | R_BAD));
  if (c.pen && !nan_row) build_counts(c, a.hist, c0, cnt);
  const double M = (double)fkey_inv(pk_key(ri.cmax));
  for (int i = threadIdx.x; i < CH; i += AT) {
    const int t = c0 + i;
    if (t >= c.V) break;
    if (nan_row) {
      out[t] = __builtin_nan("");
      continue;
    }
    bool fn = false, ff = false;
    float xm;
    const uint32_t k = elem_key(c, load_one(c, t), c.pen ? cnt[i] : 0u, mask_bit(c, t), fn, ff, xm);
    double v = 0.0;
    if (pack(k, (uint32_t)t) >= ri.kkeep && k > KEY_NEGINF) v = (exp((double)fkey_inv(k) - M) / ri.S) / ri.Z;
    out[t] = v;
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
  hipLaunchKernelGGL(dist_kernel, dim3(a.nch, a.rows), dim3(AT), 0, s, a, probs, probs_ld);
  return hipGetLastError();
}

hipError_t launch_pack(const uint8_t *bools, int64_t bld, int rows, int V, int32_t *words, int64_t wld, hipStream_t s) {
  const int nw = (V + 31) / 32;
  hipLaunchKernelGGL(pack_kernel, dim3((nw + AT - 1) / AT, rows), dim3(AT), 0, s, bools, bld, V, words, wld);
  return hipGetLastError();
}

}  // namespace gse
