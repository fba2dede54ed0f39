// The layers of GCC-A sampling: for every prefix r (a P x m occupation) and mode o the
// probability sum_i w_i |perm(U[r + e_o, s_i])|^2 over the input's substates s_i.
//
// Restates the layer of GeneralizedCliffordsSimulationStrategy
// (theboss/simulation_strategies/generalized_cliffords_simulation_strategy.py:136-247) for
// many prefixes at once: the P m output rows are formed on the device from the prefixes, the
// permanents come from tb_guan_perm_outer_ws, and the weighted squares are summed here.
// w_i holds the substate's weight over its normaliser.
#include <algorithm>

#include "tb_common.hpp"

namespace tb {

// Row p m + o in compact form: the prefix's modes in mode order, one more particle where the
// mode is o; a last slot for o itself, of multiplicity 0 where the prefix holds it. pmf[row] is
// left 0, or NaN where the prefix occupies more modes than width and the row is not whole. One
// thread per row; 4000 rows of 20 modes take 5 us, less than the copy of the rows (they were
// formed on the host, 160 us, and uploaded).
__global__ __launch_bounds__(256) void gcca_rows_kernel(const int *__restrict__ prefixes, int m,
                                                        int64_t rows, int width,
                                                        int *__restrict__ modes,
                                                        int *__restrict__ mult,
                                                        double *__restrict__ pmf) {
  const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (row >= rows) return;
  const int64_t p = row / m;
  const int o = (int)(row - p * m);
  const int *prefix = prefixes + p * m;
  int *mo = modes + row * (width + 1), *mu = mult + row * (width + 1);
  int at = 0;
  for (int j = 0; j < m; ++j) {
    const int c = prefix[j];
    if (c > 0) {
      if (at < width) {
        mo[at] = j;
        mu[at] = c + (j == o);
      }
      ++at;
    }
  }
  pmf[row] = at > width ? NAN : 0.0;
  for (; at < width; ++at) mo[at] = mu[at] = 0;
  mo[width] = o;
  mu[width] = prefix[o] > 0 ? 0 : 1;
}

// pmf[row] += sum_i w_i |perms[row][i]|^2, one wave per row; bound by the read of the
// permanents.
__global__ __launch_bounds__(256) void gcca_pmf_kernel(const cd *__restrict__ perms,
                                                       const double *__restrict__ weights,
                                                       int64_t rows, int n_in,
                                                       double *__restrict__ pmf) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // a whole wave
  const cd *p = perms + row * n_in;
  double sum = 0.0;
  for (int i = threadIdx.x & 63; i < n_in; i += 64) {
    const cd v = p[i];
    sum = fma(weights[i], fma(v.re, v.re, v.im * v.im), sum);
  }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) pmf[row] += sum;
}

}  // namespace tb

namespace {

struct GccaBuffers {
  size_t perms, modes, mult, outer, outer_bytes, bytes;  // offsets in the workspace; sizes
};

GccaBuffers gcca_buffers(int ldu, int64_t rows, int width, int in_max, int n_in, bool common) {
  const auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
  GccaBuffers g{};
  g.modes = align((size_t)rows * n_in * sizeof(tb::cd));
  g.mult = g.modes + align((size_t)rows * (width + 1) * sizeof(int));
  g.outer = g.mult + align((size_t)rows * (width + 1) * sizeof(int));
  g.outer_bytes = common ? tb_guan_outer_workspace_size(ldu, width + 1, (int32_t)rows, in_max, n_in) : 0;
  g.bytes = g.outer + g.outer_bytes;
  return g;
}

bool gcca_sizes_ok(int32_t m, int32_t prefixes_n, int32_t width, int32_t in_max, int32_t n_in) {
  return m >= 1 && prefixes_n >= 1 && width >= 1 && in_max >= 1 && n_in >= 1 &&
         (int64_t)prefixes_n * m <= INT32_MAX && (int64_t)prefixes_n * m * n_in <= INT32_MAX;
}

}  // namespace

extern "C" size_t tb_gcca_layer_workspace_size(int32_t m, int32_t prefixes_n, int32_t width,
                                               int32_t in_max, int32_t n_in, int32_t common) {
  if (!gcca_sizes_ok(m, prefixes_n, width, in_max, n_in)) return 0;
  return gcca_buffers(m, (int64_t)prefixes_n * m, width, in_max, n_in, common != 0).bytes;
}

extern "C" int32_t tb_gcca_layer_pmfs(const tb_complex128 *U, int32_t m, const int32_t *prefixes,
                                      int32_t prefixes_n, int32_t width, const int32_t *in_modes,
                                      const int32_t *in_mult, int32_t in_max, int32_t n_in,
                                      const double *weights, int32_t formula, int32_t common,
                                      double *pmf, void *workspace, size_t workspace_bytes,
                                      void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (m < 1 || prefixes_n < 0 || width < 1 || in_max < 1 || n_in < 1)
    return tbh::fail(TB_EINVAL, "gcca_layer: m=%d prefixes=%d width=%d in_max=%d n_in=%d", m,
                     prefixes_n, width, in_max, n_in);
  if (prefixes_n == 0) return TB_OK;
  if (!gcca_sizes_ok(m, prefixes_n, width, in_max, n_in))
    return tbh::fail(TB_ERANGE, "gcca_layer: %lld rows of %d permanents are more than %d",
                     (long long)prefixes_n * m, n_in, INT32_MAX);
  if (!U || !prefixes || !in_modes || !in_mult || !weights || !pmf || !workspace)
    return tbh::fail(TB_EINVAL, "gcca_layer: NULL pointer");
  const int64_t rows = (int64_t)prefixes_n * m;
  const GccaBuffers g = gcca_buffers(m, rows, width, in_max, n_in, common != 0);
  if (workspace_bytes < g.bytes)
    return tbh::fail(TB_EWORKSPACE, "gcca_layer: workspace %zu bytes < required %zu",
                     workspace_bytes, g.bytes);
  char *ws = (char *)workspace;
  tb_complex128 *perms = (tb_complex128 *)ws;
  int *modes = (int *)(ws + g.modes), *mult = (int *)(ws + g.mult);
  hipLaunchKernelGGL(tb::gcca_rows_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s,
                     prefixes, m, rows, width, modes, mult, pmf);
  if (const int32_t rc = tbh::check_hip(hipGetLastError(), "gcca_rows_kernel")) return rc;
  if (const int32_t rc = tb_guan_perm_outer_ws(U, m, modes, mult, width + 1, (int32_t)rows, in_modes,
                                               in_mult, in_max, n_in, formula, perms,
                                               g.outer_bytes ? ws + g.outer : nullptr,
                                               g.outer_bytes, stream))
    return rc;
  hipLaunchKernelGGL(tb::gcca_pmf_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s,
                     (const tb::cd *)perms, weights, rows, n_in, pmf);
  return tbh::check_hip(hipGetLastError(), "gcca_pmf_kernel");
}
