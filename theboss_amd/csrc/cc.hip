// Entry points of the submatrices calculator (the binary C&C sweep, gathered from U as it stages;
// the mixed-radix fallback lives in guan.hip) and of the permanent gradient.
#include <algorithm>

#include "sweep_impl.hpp"

namespace tbs {
size_t sweep_partial_bytes(int k, int items, int c_override);
int32_t run_sweep(int k, const tb::SweepSource &src, int items, int c_override, tb::cd *partial,
                  const int *in_mult, int in_max, tb::cd *minors, hipStream_t s);
}  // namespace tbs
namespace tbgr {
size_t grad_workspace(int n, int batch, int c_pref);
int32_t run_grad(int n, const tb::cd *A, int64_t mstride, int batch, int c_pref, int conj,
                 tb::cd *partial, tb::cd *grad, tb::cd *perm, hipStream_t s);
}  // namespace tbgr
namespace tbg {
int32_t run_guan(const tb::cd *U, int ldu, const int *out_modes, const int *out_mult, int out_max,
                 const int *in_modes, const int *in_mult, int in_max, int batch, int formula,
                 int mode, tb::cd *out, hipStream_t s, int n_in = 0, int *done = nullptr, int counters = 0);
}  // namespace tbg

namespace tb {

// k == 1: bs_submatrices_permanent_calculator_base.py:156-158 returns s itself.
__global__ void cc_single_kernel(const int *__restrict__ in_mult, int n, cd *__restrict__ minors) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < n) minors[idx] = {(double)in_mult[idx], 0.0};
}

__global__ void grad_small_kernel(const cd *__restrict__ A, int n, int batch, int64_t mstride,
                                  cd *__restrict__ perm, cd *__restrict__ G) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  if (n == 0) {
    perm[b] = {1.0, 0.0};
  } else {  // n == 1
    perm[b] = A[(size_t)b * mstride];
    G[b] = {1.0, 0.0};
  }
}

}  // namespace tb

extern "C" size_t tb_cc_workspace_size(int32_t k, int32_t out_max, int32_t in_max, int32_t batch) {
  (void)out_max;
  (void)in_max;
  if (k < 2 || k > TB_SWEEP_MAX_K) return 0;
  return tbs::sweep_partial_bytes(k, batch, tbh::tuned(TB_TUNE_SWEEP, k, batch));
}

extern "C" int32_t tb_cc_submatrices_batch(const tb_complex128 *U, int32_t ldu,
                                           const int32_t *out_modes, const int32_t *out_mult,
                                           int32_t out_max, const int32_t *in_modes,
                                           const int32_t *in_mult, int32_t in_max, int32_t batch,
                                           int32_t k, int32_t collision_free,
                                           tb_complex128 *minors, void *workspace,
                                           size_t workspace_bytes, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (batch < 0) return tbh::fail(TB_EINVAL, "cc: batch=%d < 0", batch);
  if (batch == 0) return TB_OK;
  if (!in_mult || !minors) return tbh::fail(TB_EINVAL, "cc: NULL pointer");
  if (in_max < 1) return tbh::fail(TB_EINVAL, "cc: in_max=%d < 1", in_max);
  if (k < 1) return tbh::fail(TB_EINVAL, "cc: k=%d < 1", k);
  tb::cd *mo = (tb::cd *)minors;
  if (k == 1) {
    const int n = batch * in_max;
    hipLaunchKernelGGL(tb::cc_single_kernel, dim3((n + 255) / 256), dim3(256), 0, s, in_mult, n, mo);
    return tbh::check_hip(hipGetLastError(), "cc_single_kernel");
  }
  if (!U || !out_modes || !out_mult || !in_modes) return tbh::fail(TB_EINVAL, "cc: NULL pointer");
  if (out_max < 1 || ldu < 1)
    return tbh::fail(TB_EINVAL, "cc: out_max=%d ldu=%d must be >= 1", out_max, ldu);
  if (!collision_free) {
    if (out_max > TB_GUAN_MAX_ROWS || in_max > TB_GUAN_MAX_COLS)
      return tbh::fail(TB_ERANGE, "cc: out_max=%d > %d or in_max=%d > %d", out_max,
                       TB_GUAN_MAX_ROWS, in_max, TB_GUAN_MAX_COLS);
    return tbg::run_guan((const tb::cd *)U, ldu, out_modes, out_mult, out_max, in_modes, in_mult,
                         in_max, batch, TB_FORMULA_RYSER, 1, mo, s);
  }
  if (k > TB_SWEEP_MAX_K)
    return tbh::fail(TB_ERANGE, "cc: k=%d exceeds TB_SWEEP_MAX_K=%d", k, TB_SWEEP_MAX_K);
  const int c = tbh::tuned(TB_TUNE_SWEEP, k, batch);  // read once: size check and launch agree
  const size_t need = tbs::sweep_partial_bytes(k, batch, c);
  if (!workspace || workspace_bytes < need)
    return tbh::fail(TB_EWORKSPACE, "cc: workspace %zu bytes < required %zu", workspace_bytes,
                     need);
  tb::SweepSource src{};
  src.U = (const tb::cd *)U;
  src.ldu = ldu;
  src.out_modes = out_modes;
  src.out_mult = out_mult;
  src.out_max = out_max;
  src.in_modes = in_modes;
  src.in_mult = in_mult;
  src.in_max = in_max;
  return tbs::run_sweep(k, src, batch, c, (tb::cd *)workspace, in_mult, in_max, mo, s);
}

extern "C" size_t tb_perm_grad_workspace_size(int32_t n, int32_t batch) {
  if (n < 2 || n > TB_SWEEP_MAX_K) return 0;
  return tbgr::grad_workspace(n, batch, tbh::tuned(TB_TUNE_GRAD, n, batch));
}

namespace {
int32_t perm_grad(const tb_complex128 *A, int32_t n, int32_t batch, int64_t matrix_stride,
                  int conj, tb_complex128 *perm_out, tb_complex128 *grad_out, void *workspace,
                  size_t workspace_bytes, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (batch < 0) return tbh::fail(TB_EINVAL, "grad: batch=%d < 0", batch);
  if (batch == 0) return TB_OK;
  if (n < 0) return tbh::fail(TB_EINVAL, "grad: n=%d < 0", n);
  if (n > TB_SWEEP_MAX_K)
    return tbh::fail(TB_ERANGE, "grad: n=%d exceeds TB_SWEEP_MAX_K=%d", n, TB_SWEEP_MAX_K);
  if (!perm_out || (n > 0 && (!A || !grad_out))) return tbh::fail(TB_EINVAL, "grad: NULL pointer");
  if (n > 0 && matrix_stride < (int64_t)n * n)
    return tbh::fail(TB_EINVAL, "grad: matrix_stride=%lld < n*n", (long long)matrix_stride);
  if (n < 2) {
    hipLaunchKernelGGL(tb::grad_small_kernel, dim3((batch + 255) / 256), dim3(256), 0, s,
                       (const tb::cd *)A, n, batch, matrix_stride, (tb::cd *)perm_out,
                       (tb::cd *)grad_out);
    return tbh::check_hip(hipGetLastError(), "grad_small_kernel");
  }
  const int c = tbh::tuned(TB_TUNE_GRAD, n, batch);  // read once: size check and launch agree
  const size_t need = tbgr::grad_workspace(n, batch, c);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return tbh::fail(TB_EWORKSPACE, "grad: workspace %zu bytes < required %zu", workspace_bytes,
                     need);
  return tbgr::run_grad(n, (const tb::cd *)A, matrix_stride, batch, c, conj, (tb::cd *)workspace,
                        (tb::cd *)grad_out, (tb::cd *)perm_out, s);
}
}  // namespace

extern "C" int32_t tb_perm_grad_batch(const tb_complex128 *A, int32_t n, int32_t batch,
                                      int64_t matrix_stride, tb_complex128 *perm_out,
                                      tb_complex128 *grad_out, void *workspace,
                                      size_t workspace_bytes, void *stream) {
  return perm_grad(A, n, batch, matrix_stride, 0, perm_out, grad_out, workspace, workspace_bytes,
                   stream);
}

extern "C" int32_t tb_perm_grad_conj_batch(const tb_complex128 *A, int32_t n, int32_t batch,
                                           int64_t matrix_stride, tb_complex128 *perm_out,
                                           tb_complex128 *grad_out, void *workspace,
                                           size_t workspace_bytes, void *stream) {
  return perm_grad(A, n, batch, matrix_stride, 1, perm_out, grad_out, workspace, workspace_bytes,
                   stream);
}
