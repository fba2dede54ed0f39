// Permanent gradient d perm(A) / dA[i][j] = perm(A without row i and column j), all n^2
// entries of a batch of n x n complex128 matrices, in one Gray sweep per matrix.
//
// The reference has no gradients. Row i of the result is what
// BSCCRyserSubmatricesPermanentCalculator.compute_permanents returns with output rows =
// all rows but i (theboss/boson_sampling_utilities/permanent_calculators/
// bs_cc_ryser_submatrices_permanent_calculator.py:73-119).
//
// Formula. Glynn's identity with delta over the rows (delta_{n-1} = +1) and half column
// sums h_j = (1/2) sum_i delta_i A[i][j] gives perm(A) = 2 sum_delta (prod delta) prod_j h_j.
// perm is linear in A[i][j], and d h_l / d A[i][j] = delta_i [l == j] / 2, so
//   G[i][j] = sum_delta (prod delta) delta_i prod_{l != j} h_l.
// A Gray walk over delta keeps, per column j, the running sum T_j of (prod delta) P_j with
// P_j = prod_{l != j} h_l, and for each Gray bit i a corrector E_ij += 2 delta_i(old) T_j
// updated when the bit flips; then sum_t delta_i(t) (prod delta) P_j(t) = E_ij + delta_i(end) T_j.
//
// Columns over lanes. L = 2 or 4 lanes (one per half or per row of 16 lanes of the wave)
// walk the same Gray codes, each holding C = ceil(n / L) columns (padded with columns whose
// sum stays 1). Per code a lane does its C row adds, the product tree of its own columns,
// swaps that product with the other lanes, and walks the tree down with Q = the product of
// the other lanes' columns: 3C - 3 (+ 2 with L = 4) complex multiplies, the last of each
// leaf fused into T_j. All n columns therefore share one walk. The walk in groups of 8
// columns that this replaces redid the row flips and the product of the other n - 8 columns
// in every group: at n = 20 it issued 8.2 FP64 instructions per code and matrix against 4.7.
//
// What bounds it: VALU issue. At n = 20 (L = 4) a step of 16 codes is about 82 VALU
// instructions, 75 of them FP64 (the rest mostly the code-lane sums at block starts): 0.30 ms
// for 64 matrices if issued back to back at 2.2 GHz, 0.39 measured (0.60 before). The products are swapped over the LDS crossbar (ds_swizzle, ds_bpermute)
// because that leaves the VALU alone: with permlane swaps and selects (24 32-bit
// instructions per code) n = 20 took 0.43-0.47 ms. L = 2 needs 4% fewer instructions and pads
// less, L = 4 half the registers: L = 2 is 10-25% faster at n = 10..18 (n = 14, 1000
// matrices: 64 against 84 us), L = 4 from n = 19 on, where L = 2 spills with 3 static bits
// (2 bits: 0.389 against 0.384 ms at n = 20), and at n <= 8, where L = 2 would leave too few
// codes per lane (n = 8, 10000 matrices: 20.8 against 18.6 us; 290 us as n sweeps per matrix).
//
// Work split. A lane group walks an aligned chunk of 2^c Gray ranks. Bits below U flip
// inside the unrolled static block of 2^U steps and keep per-lane correctors in registers.
// Bits U..c-1 flip at block starts in the same direction in every lane (the top one, whose
// direction is bit 0 of the chunk index, takes its sign per lane), so their correctors are
// kept per wave: at such a flip the wave sums T_j over its code lanes (transposed, so
// that each lane ends with one value) and adds it to the row's sums in LDS. Bits above the
// chunk contribute delta_i T_j at the chunk end.
//
// Infinities and NaN. Row i of the result does not depend on row i of the matrix, but every
// column sum holds it. Rows with such an entry are walked as zeros, and the other rows of the
// result, which depend on them, are NaN.
#include <algorithm>
#include <cmath>

#include "flip_common.hpp"

namespace tb {

constexpr int kGradMinN = 6;
constexpr int kGradMaxN = TB_SWEEP_MAX_K;

// Lanes per code, columns per lane, padded columns.
constexpr int grad_l(int n) { return n <= 8 || n > 18 ? 4 : 2; }
constexpr int grad_cols(int n) { return (n + grad_l(n) - 1) / grad_l(n); }
constexpr int grad_np(int n) { return grad_l(n) * grad_cols(n); }
// log2 of the code lanes of a wave.
constexpr int grad_lb(int n) { return grad_l(n) == 4 ? 4 : 5; }
// Static Gray bits: the more, the fewer block starts and their code-lane sums, as far as the
// 2C correctors of each fit 256 VGPRs, but for 2 to 12 values at n = 15..18 and 29..32 that are
// reloaded once a chunk (n = 20: 0.384 ms with 4, 0.396 with 3, 0.424 with 2).
// At n <= 8 a lane group walks 2^3 codes or fewer: 2 bits and 3 take the same time within 4%.
constexpr int grad_u(int n) {
  const int u = grad_l(n) == 2 ? (n <= 16 ? 4 : 3) : n <= 8 ? 2 : n <= 32 ? 4 : 2;
  return n - 1 - grad_lb(n) < u ? n - 1 - grad_lb(n) : u;
}
// LDS: the matrix and one n x np accumulator per wave of the workgroup.
constexpr size_t grad_lds(int n, int w) { return sizeof(cd) * (size_t)n * grad_np(n) * (size_t)(1 + w); }
// log2 of the waves per workgroup: 64 code lanes (at most 64 KiB of LDS).
constexpr int grad_wbits(int n) {
  int w = 6 - grad_lb(n);
  while (w > 0 && grad_lds(n, 1 << w) > 64 * 1024) --w;
  return w;
}

// v of lane ^ 16 and of lane ^ 32, over the LDS crossbar: no VALU issue slots, which the
// FP64 work needs (permlane swaps and their selects: 24 32-bit instructions per code).
__device__ __forceinline__ double xor16_lane(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_ds_swizzle((int)(uint32_t)u, 0x401f);
  const int hi = __builtin_amdgcn_ds_swizzle((int)(uint32_t)(u >> 32), 0x401f);
  return join64((uint32_t)lo, (uint32_t)hi);
}
__device__ __forceinline__ double xor32_lane(double v, int addr) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)u);
  const int hi = __builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)(u >> 32));
  return join64((uint32_t)lo, (uint32_t)hi);
}

// Product tree over columns LO..HI-1 of a lane; inner products are kept in P by the
// node's midpoint.
template <int C, int LO, int HI>
__device__ __forceinline__ cd tree_up(const double (&hr)[C], const double (&hi)[C], cd (&P)[C + 1]) {
  if constexpr (HI - LO == 1) {
    return {hr[LO], hi[LO]};
  } else {
    constexpr int MID = (LO + HI) / 2;
    const cd p = cmul(tree_up<C, LO, MID>(hr, hi, P), tree_up<C, MID, HI>(hr, hi, P));
    P[MID] = p;
    return p;
  }
}
template <int C, int LO, int HI>
__device__ __forceinline__ cd tree_get(const double (&hr)[C], const double (&hi)[C],
                                       const cd (&P)[C + 1]) {
  if constexpr (HI - LO == 1)
    return {hr[LO], hi[LO]};
  else
    return P[(LO + HI) / 2];
}
// T_j += SIGN * (out times the product of the node's other columns) for its columns j.
template <int SIGN, int C, int LO, int HI>
__device__ __forceinline__ void tree_down(cd out, const double (&hr)[C], const double (&hi)[C],
                                          const cd (&P)[C + 1], double (&Tr)[C], double (&Ti)[C]) {
  constexpr int MID = (LO + HI) / 2;
  const cd a = tree_get<C, LO, MID>(hr, hi, P), b = tree_get<C, MID, HI>(hr, hi, P);
  if constexpr (MID - LO == 1)
    cmul_acc<SIGN>(Tr[LO], Ti[LO], out, b);
  else
    tree_down<SIGN, C, LO, MID>(cmul(out, b), hr, hi, P, Tr, Ti);
  if constexpr (HI - MID == 1)
    cmul_acc<SIGN>(Tr[MID], Ti[MID], out, a);
  else
    tree_down<SIGN, C, MID, HI>(cmul(out, a), hr, hi, P, Tr, Ti);
}

// T_j += SIGN * prod_{l != j} h_l for the lane's columns j, l over all columns.
template <int SIGN, int L, int C>
__device__ __forceinline__ void loo_acc(const double (&hr)[C], const double (&hi)[C], double (&Tr)[C],
                                        double (&Ti)[C], int far) {
  cd P[C + 1];
  const cd own = tree_up<C, 0, C>(hr, hi, P);
  cd q;
  if constexpr (L == 4) {
    const cd a = {xor16_lane(own.re), xor16_lane(own.im)};
    const cd half = cmul(own, a);
    const cd b = {xor32_lane(half.re, far), xor32_lane(half.im, far)};
    q = cmul(a, b);
  } else {
    q = {xor32_lane(own.re, far), xor32_lane(own.im, far)};
  }
  if constexpr (C == 1) {
    Tr[0] += SIGN * q.re;
    Ti[0] += SIGN * q.im;
  } else {
    tree_down<SIGN, C, 0, C>(q, hr, hi, P, Tr, Ti);
  }
}

// The lane's slots of its column block of one row, in broadcast form.
template <int C>
__device__ __forceinline__ Bcast<C> grad_row(const cd *block_row, int lane) {
  Bcast<C> b;
#pragma unroll
  for (int p = 0; p < Bcast<C>::P; ++p) {
    const int t = 16 * p + (lane & 15);
    b.v[p] = ((const double *)block_row)[t < 2 * C ? t : 2 * C - 1];
  }
  return b;
}
// Two wait states between whatever wrote the row's registers and its DPP reads.
template <int C>
__device__ __forceinline__ void dpp_ready(Bcast<C> &b) {
  if constexpr (Bcast<C>::P == 1)
    asm volatile("s_nop 1" : "+v"(b.v[0]));
  else
    asm volatile("s_nop 1" : "+v"(b.v[0]), "+v"(b.v[Bcast<C>::P - 1]));
}

// The rows of the matrix in Ms with an infinite or NaN entry, a bit each, and zeros in their place.
// Called by the workgroup where there is one.
template <int N, int NP>
__device__ __attribute__((noinline)) void grad_clear_rows(cd *Ms, uint64_t *bad) {
  if (threadIdx.x == 0) {
    uint64_t rows = 0;
    for (int e = 0; e < N * NP; ++e)
      if (!isfinite(Ms[e].re) || !isfinite(Ms[e].im)) rows |= 1ull << (e / NP);
    *bad = rows;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < N * N; e += blockDim.x)
    if ((*bad >> (e / N)) & 1ull) Ms[e / N * NP + e % N] = {0.0, 0.0};
  __syncthreads();
}

// Workgroup = 2^wb waves of one matrix: chunk q = ((it wpi + wg) 2^wb + wave) 2^lb + code
// lane. wpi workgroups per matrix; direct: wpi == 1 and the results go to grad and perm,
// otherwise to partial[(b wpi + wg)][n][n].
template <int N>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void grad_kernel(
    const cd *__restrict__ A, int64_t mstride, int c, int wpi, int iters, int conj,
    cd *__restrict__ partial, cd *__restrict__ grad, cd *__restrict__ perm) {
  constexpr int L = grad_l(N), C = grad_cols(N), NP = grad_np(N), LB = grad_lb(N), U = grad_u(N);
  constexpr int NB = N - 1;
  extern __shared__ cd smem[];
  cd *Ms = smem;  // [N][NP]
  const int lane = threadIdx.x & 63;
  const int wave = uniform_int(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int b = blockIdx.x / wpi, wg = blockIdx.x - b * wpi;
  cd *acc = smem + (size_t)N * NP * (1 + wave);  // this wave's sums, [N][NP]
  const cd *src = A + (size_t)b * mstride;
  __shared__ uint64_t bad;  // set where `odd` is, per wave: an entry that is not finite
  __shared__ int odd[4];
  bool finite = true;
  for (int e = threadIdx.x; e < N * NP; e += blockDim.x) {
    const int i = e / NP, j = e - i * NP;
    // a padding column's half sum is 1: 2 in the fixed row, 0 in the others
    const cd v = j < N ? src[i * N + j] : cd{i == NB ? 2.0 : 0.0, 0.0};
    Ms[e] = v;
    finite &= isfinite(v.re) && isfinite(v.im);
  }
  for (int e = lane; e < N * NP; e += 64) acc[e] = {0.0, 0.0};
  odd[wave] = __any(!finite);
  __syncthreads();
  const auto any_odd = [&] {
    int any = odd[0];
    for (int w = 1; w < waves; ++w) any |= odd[w];
    return uniform_int(any) != 0;
  };
  if (any_odd()) grad_clear_rows<N, NP>(Ms, &bad);
  const int far = (lane ^ 32) << 2;         // ds_bpermute address of lane ^ 32
  const int blk_col = (lane >> LB) * C;     // first column of the lane's block
  const cd *M = Ms + blk_col;
  const int sum_ix = lane_sums_index<LB>(lane);
  double *acc_l = (double *)(acc + blk_col) + sum_ix;  // + row * 2 NP
  // x (2C values per lane) summed over the code lanes and added to row i of the wave's sums.
  auto row_add = [&](double (&x)[2 * C], int i, double coef) {
    lane_sums<LB, 2 * C>(x, lane);
#pragma unroll
    for (int v = 0; v << LB < 2 * C; ++v)
      if (sum_ix + (v << LB) < 2 * C) {
        double *p = acc_l + i * 2 * NP + (v << LB);
        *p = fma(coef, x[v], *p);
      }
  };
  Bcast<C> rows[U];  // the static rows
#pragma unroll
  for (int u = 0; u < U; ++u) rows[u] = grad_row<C>(M + u * NP, lane);
  const double one = vgpr_one();
#pragma unroll
  for (int u = 0; u < U; ++u) dpp_ready(rows[u]);
  const int nblocks = 1 << (c - U);
  for (int it = 0; it < iters; ++it) {
    const uint64_t qw = ((uint64_t)it * wpi + wg) * waves + wave;  // wave-uniform
    const uint64_t q = (qw << LB) | (uint64_t)(lane & ((1 << LB) - 1));
    const bool q_odd = (lane & 1) != 0;
    const uint64_t t0 = q << c;
    const uint64_t g0 = t0 ^ (t0 >> 1);
    // Half column sums at t0.
    double hr[C], hi[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const cd v = M[NB * NP + j];
      hr[j] = 0.5 * v.re;
      hi[j] = 0.5 * v.im;
    }
#pragma unroll 1
    for (int r = 0; r < NB; ++r) {
      Bcast<C> row = grad_row<C>(M + r * NP, lane);
      const double d = ((g0 >> r) & 1ull) ? -0.5 : 0.5;
      dpp_ready(row);
      flip_bcast<0, C, 0>(hr, hi, row, d);
    }
    double Tr[C], Ti[C];
#pragma unroll
    for (int k = 0; k < C; ++k) {
      Tr[k] = 0.0;
      Ti[k] = 0.0;
    }
    loo_acc<1, L, C>(hr, hi, Tr, Ti, far);  // prod(delta) = (-1)^t0 = +1 (t0 even)
    double Er[U][C], Ei[U][C];
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int k = 0; k < C; ++k) {
        Er[i][k] = 0.0;
        Ei[i][k] = 0.0;
      }
    // Static steps jj = 1 .. 2^U - 1 of block blk: bit i = ctz(jj) flips; its new value
    // is 1 ^ t_{i+1}. t_{i+1} == 0: delta_i +1 -> -1 (h -= row, E += 2T); else h += row,
    // E -= 2T.
    auto static_steps = [&](int blk) {
#pragma unroll
      for (int jj = 1; jj < (1 << U); ++jj) {
        const int i = __builtin_ctz(jj);
        if (i + 1 < U) {
          if ((jj >> (i + 1)) & 1) {
#pragma unroll
            for (int k = 0; k < C; ++k) {
              Er[i][k] = fma(-2.0, Tr[k], Er[i][k]);
              Ei[i][k] = fma(-2.0, Ti[k], Ei[i][k]);
            }
            flip_bcast<0, C, 1>(hr, hi, rows[i], one);
          } else {
#pragma unroll
            for (int k = 0; k < C; ++k) {
              Er[i][k] = fma(2.0, Tr[k], Er[i][k]);
              Ei[i][k] = fma(2.0, Ti[k], Ei[i][k]);
            }
            flip_bcast<0, C, -1>(hr, hi, rows[i], one);
          }
        } else {
          const bool t_next = (U < c) ? ((blk & 1) != 0) : q_odd;
          const double sg = t_next ? 1.0 : -1.0;
#pragma unroll
          for (int k = 0; k < C; ++k) {
            Er[i][k] = fma(-2.0 * sg, Tr[k], Er[i][k]);
            Ei[i][k] = fma(-2.0 * sg, Ti[k], Ei[i][k]);
          }
          flip_bcast<0, C, 0>(hr, hi, rows[i], sg);
        }
        if (jj & 1)
          loo_acc<-1, L, C>(hr, hi, Tr, Ti, far);
        else
          loo_acc<1, L, C>(hr, hi, Tr, Ti, far);
        TB_STEP_FENCE();
      }
    };
    // The row of the next block start is loaded a block ahead.
    Bcast<C> next = grad_row<C>(M + (U < NB ? U : 0) * NP, lane);
    static_steps(0);
    for (int blk = 1; blk < nblocks; ++blk) {
      const int i = U + __builtin_ctz(blk);
      const bool lane_dir = i + 1 == c;  // the top in-chunk bit: direction from the chunk index
      const bool t_next = lane_dir ? q_odd : (((blk >> (i + 1 - U)) & 1) != 0);
      const double sg = t_next ? 1.0 : -1.0;
      {  // wave-level corrector of bit i
        double x[2 * C];
#pragma unroll
        for (int k = 0; k < C; ++k) {
          x[2 * k] = Tr[k];
          x[2 * k + 1] = Ti[k];
        }
        if (lane_dir) {
#pragma unroll
          for (int k = 0; k < 2 * C; ++k) x[k] *= sg;
        }
        row_add(x, i, lane_dir ? -2.0 : -2.0 * sg);
      }
      dpp_ready(next);
      flip_bcast<0, C, 0>(hr, hi, next, sg);
      next = grad_row<C>(M + (U + __builtin_ctz(blk + 1 < nblocks ? blk + 1 : 1)) * NP, lane);
      loo_acc<1, L, C>(hr, hi, Tr, Ti, far);
      TB_STEP_FENCE();
      static_steps(blk);
    }
    // End of the chunk.
    const uint64_t tend = t0 + ((uint64_t)1 << c) - 1;
    const uint64_t gend = tend ^ (tend >> 1);
#pragma unroll
    for (int i = 0; i < U; ++i) {  // static rows: E + delta(end) T per lane
      const double d = ((gend >> i) & 1ull) ? -1.0 : 1.0;
      double x[2 * C];
#pragma unroll
      for (int k = 0; k < C; ++k) {
        x[2 * k] = fma(d, Tr[k], Er[i][k]);
        x[2 * k + 1] = fma(d, Ti[k], Ei[i][k]);
      }
      row_add(x, i, 1.0);
    }
    // Rows whose delta at the chunk end depends on the code lane: the top in-chunk bit and
    // the LB lane bits above it.
    const int lo_lane = c - 1 > U ? c - 1 : U, hi_lane = c + LB < NB ? c + LB : NB;
#pragma unroll 1
    for (int i = lo_lane; i < hi_lane; ++i) {
      const double d = ((gend >> i) & 1ull) ? -1.0 : 1.0;
      double x[2 * C];
#pragma unroll
      for (int k = 0; k < C; ++k) {
        x[2 * k] = d * Tr[k];
        x[2 * k + 1] = d * Ti[k];
      }
      row_add(x, i, 1.0);
    }
    {  // the other rows: in-chunk bits (+1 at the end), bits above the lane bits, the fixed row
      double x[2 * C];
#pragma unroll
      for (int k = 0; k < C; ++k) {
        x[2 * k] = Tr[k];
        x[2 * k + 1] = Ti[k];
      }
      lane_sums<LB, 2 * C>(x, lane);
      const uint64_t gw = gend;  // rows outside the lane range: the same in every lane
      for (int i = U; i < N; ++i) {
        if (i >= lo_lane && i < hi_lane) continue;
        const double d = (i < NB && ((gw >> i) & 1ull)) ? -1.0 : 1.0;
#pragma unroll
        for (int v = 0; v << LB < 2 * C; ++v)
          if (sum_ix + (v << LB) < 2 * C) {
            double *p = acc_l + i * 2 * NP + (v << LB);
            *p = fma(d, x[v], *p);
          }
      }
    }
  }
  __syncthreads();
  const cd *sums = smem + (size_t)N * NP;
  const bool direct = wpi == 1;
  const uint64_t cleared = any_odd() ? bad : 0;
  cd *dst = direct ? grad + (size_t)b * N * N : partial + (size_t)blockIdx.x * N * N;
  for (int e = threadIdx.x; e < N * N; e += blockDim.x) {
    const int i = e / N, j = e - i * N;
    cd v = sums[i * NP + j];
    for (int w = 1; w < waves; ++w) v = cadd(v, sums[(size_t)w * N * NP + i * NP + j]);
    if (cleared != 0 && cleared != 1ull << i) v = {NAN, NAN};
    if (direct && i == 0) {  // perm: the Laplace expansion along row 0
      const cd t = cmul((cleared & 1ull) != 0 ? src[j] : Ms[j], v);
      Ms[j] = t;
    }
    if (direct && conj) v.im = -v.im;
    dst[e] = v;
  }
  if (!direct) return;  // uniform over the workgroup
  __syncthreads();
  if (threadIdx.x == 0) {
    cd p = Ms[0];
    for (int j = 1; j < N; ++j) p = cadd(p, Ms[j]);
    perm[b] = p;
  }
}

// One block per (matrix, row): grad[b][i][j] = sum_w partial[b wpi + w][i][j] in a fixed order
// (256 / n slices of w, then the slices), and perm[b] from row 0 by Laplace expansion.
__global__ __launch_bounds__(256) void grad_reduce_kernel(const cd *__restrict__ partial,
                                                          const cd *__restrict__ A, int64_t mstride,
                                                          int n, int wpi, int conj,
                                                          cd *__restrict__ grad,
                                                          cd *__restrict__ perm) {
  __shared__ cd part[256];
  const int b = blockIdx.x / n, i = blockIdx.x - b * n;
  const int slices = 256 / n;
  const int sl = threadIdx.x / n, j = threadIdx.x - sl * n;
  if (sl < slices) {
    const cd *src = partial + ((size_t)b * wpi * n + i) * n + j;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int w = sl; w < wpi; w += slices) {
      const cd v = src[(size_t)w * n * n];
      re += v.re;
      im += v.im;
    }
    part[threadIdx.x] = {re, im};
  }
  __syncthreads();
  if (threadIdx.x < n) {
    cd v = part[threadIdx.x];
    for (int s = 1; s < slices; ++s) v = cadd(v, part[s * n + threadIdx.x]);
    if (i == 0) part[threadIdx.x] = cmul(A[(size_t)b * mstride + threadIdx.x], v);
    if (conj) v.im = -v.im;
    grad[((size_t)b * n + i) * n + threadIdx.x] = v;
  }
  if (i != 0) return;  // uniform over the block
  __syncthreads();
  if (threadIdx.x == 0) {
    cd p = part[0];
    for (int k = 1; k < n; ++k) p = cadd(p, part[k]);
    perm[b] = p;
  }
}

// Permanent of a K x K matrix in registers, K <= 4 (expansion into 2 x 2 blocks).
template <int K>
__device__ __forceinline__ cd perm_tiny(const cd (&m)[K][K]) {
  auto two = [&](int r, int a, int b) { return cadd(cmul(m[r][a], m[r + 1][b]), cmul(m[r][b], m[r + 1][a])); };
  if constexpr (K == 1) {
    return m[0][0];
  } else if constexpr (K == 2) {
    return two(0, 0, 1);
  } else if constexpr (K == 3) {
    return cadd(cadd(cmul(m[0][0], two(1, 1, 2)), cmul(m[0][1], two(1, 0, 2))), cmul(m[0][2], two(1, 0, 1)));
  } else {
    const cd a = cadd(cmul(two(0, 0, 1), two(2, 2, 3)), cmul(two(0, 2, 3), two(2, 0, 1)));
    const cd b = cadd(cmul(two(0, 0, 2), two(2, 1, 3)), cmul(two(0, 1, 3), two(2, 0, 2)));
    const cd c = cadd(cmul(two(0, 0, 3), two(2, 1, 2)), cmul(two(0, 1, 2), two(2, 0, 3)));
    return cadd(cadd(a, b), c);
  }
}

// n = 2..5: one thread per (matrix, row) expands its n minors directly (fewer than the 32
// codes that fill a wave of the Gray walk); the thread of row 0 also forms the permanent.
template <int N>
__global__ __launch_bounds__(256) void grad_tiny_kernel(const cd *__restrict__ A, int64_t mstride,
                                                        int batch, int conj, cd *__restrict__ grad,
                                                        cd *__restrict__ perm) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)batch * N) return;
  const int b = (int)(idx / N), i = (int)(idx - (int64_t)b * N);
  const cd *src = A + (size_t)b * mstride;
  cd row[N - 1][N];  // the other rows
#pragma unroll
  for (int r = 0; r < N - 1; ++r)
#pragma unroll
    for (int j = 0; j < N; ++j) row[r][j] = src[(r < i ? r : r + 1) * N + j];
  cd p = {0.0, 0.0};
#pragma unroll
  for (int j = 0; j < N; ++j) {
    cd m[N - 1][N - 1];
#pragma unroll
    for (int r = 0; r < N - 1; ++r)
#pragma unroll
      for (int k = 0; k < N - 1; ++k) m[r][k] = row[r][k < j ? k : k + 1];
    cd v = perm_tiny<N - 1>(m);
    if (i == 0) p = cadd(p, cmul(src[j], v));
    if (conj) v.im = -v.im;
    grad[(size_t)idx * N + j] = v;
  }
  if (i == 0) perm[b] = p;
}

}  // namespace tb

namespace tbgr {

struct GradPlan {
  int c, wb, wpi, iters;  // chunk bits, log2 waves per workgroup, workgroups per matrix
};

// Chunks of 2^c ranks per lane group, workgroups of up to 64 code lanes. Built in: among the
// chunks of at most 2^11 ranks, the one with the best product of the fill of the SIMDs (waves
// per SIMD over that rounded up), the share of the issue rate that so many waves reach
// (measured: 0.83 with one, 0.97 with two) and the share of a chunk left after its seed and
// its end, which cost about 10 steps (n = 20, 64 matrices: 2^6 443 us, 2^7 411, 2^8 398,
// 2^9 396, 2^10 405, 2^11 474). A tuned c (c_pref > 0) replaces that choice.
//
// A workgroup writes n^2 partial sums, so with many of them the groups walk several chunks each and
// the partials stay below 2^16 n^2 (n = 30, 1000 matrices: 0.9 GB, not 110). That many groups are
// 64 rounds or more of the resident waves.
constexpr int64_t kGradMaxGroups = 1 << 16;
inline GradPlan grad_plan(int n, int batch, int c_pref) {
  GradPlan p{};
  const int nb = n - 1, lb = tb::grad_lb(n), u = tb::grad_u(n), wfull = tb::grad_wbits(n);
  auto clamp = [&](int c) { return std::min(std::max(c, u), nb - lb); };
  const int top = clamp(11);  // at most one wave per matrix
  int c = top;
  if (c_pref > 0) {
    c = clamp(c_pref);
  } else {
    double best = -1.0;
    for (int cc = top; cc >= u; --cc) {
      const double w = (double)batch * std::ldexp(1.0, nb - cc - lb) / 1024.0;  // per SIMD
      const double up = std::ceil(w), rate = up < 2.0 ? 0.83 : up < 3.0 ? 0.97 : 1.0;
      const double score = w / up * rate / (1.0 + 10.0 / std::ldexp(1.0, cc));
      if (score > best + 1e-9) {
        best = score;
        c = cc;
      }
    }
  }
  p.c = c;
  const int wave_bits = nb - c - lb;  // log2 of the waves per matrix at one chunk per lane group
  p.wb = std::min(wave_bits, wfull);
  int wg_bits = std::min(wave_bits - p.wb, 13);
  while (wg_bits > 0 && ((int64_t)batch << wg_bits) > kGradMaxGroups) --wg_bits;
  p.wpi = 1 << wg_bits;
  p.iters = 1 << (wave_bits - p.wb - wg_bits);
  return p;
}

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t grad_workspace(int n, int batch, int c_pref) {
  if (n < tb::kGradMinN || n > tb::kGradMaxN || batch <= 0) return 0;
  const GradPlan p = grad_plan(n, batch, c_pref);
  return align256((size_t)batch * p.wpi * n * n * sizeof(tb::cd));
}

template <int N>
int32_t launch_grad(const tb::cd *A, int64_t mstride, int batch, const GradPlan &p, int conj,
                    tb::cd *partial, tb::cd *grad, tb::cd *perm, hipStream_t s) {
  hipLaunchKernelGGL((tb::grad_kernel<N>), dim3((unsigned)((int64_t)batch * p.wpi)),
                     dim3(64u << p.wb), tb::grad_lds(N, 1 << p.wb), s, A, mstride, p.c, p.wpi,
                     p.iters, conj, partial, grad, perm);
  return tbh::check_hip(hipGetLastError(), "grad_kernel");
}

template <int N = tb::kGradMinN>
int32_t dispatch_grad(int n, const tb::cd *A, int64_t mstride, int batch, const GradPlan &p,
                      int conj, tb::cd *partial, tb::cd *grad, tb::cd *perm, hipStream_t s) {
  if constexpr (N > tb::kGradMaxN) {
    return tbh::fail(TB_ERANGE, "grad: no kernel for n=%d", n);
  } else {
    if (n == N) return launch_grad<N>(A, mstride, batch, p, conj, partial, grad, perm, s);
    return dispatch_grad<N + 1>(n, A, mstride, batch, p, conj, partial, grad, perm, s);
  }
}

template <int N>
int32_t launch_tiny(const tb::cd *A, int64_t mstride, int batch, int conj, tb::cd *grad,
                    tb::cd *perm, hipStream_t s) {
  hipLaunchKernelGGL((tb::grad_tiny_kernel<N>), dim3((unsigned)(((int64_t)batch * N + 255) / 256)),
                     dim3(256), 0, s, A, mstride, batch, conj, grad, perm);
  return tbh::check_hip(hipGetLastError(), "grad_tiny_kernel");
}

// Permanents and all n^2 minors (conjugated when conj), 2 <= n <= kGradMaxN; the workspace
// holds grad_workspace bytes.
int32_t run_grad(int n, const tb::cd *A, int64_t mstride, int batch, int c_pref, int conj,
                 tb::cd *partial, tb::cd *grad, tb::cd *perm, hipStream_t s) {
  switch (n) {
    case 2: return launch_tiny<2>(A, mstride, batch, conj, grad, perm, s);
    case 3: return launch_tiny<3>(A, mstride, batch, conj, grad, perm, s);
    case 4: return launch_tiny<4>(A, mstride, batch, conj, grad, perm, s);
    case 5: return launch_tiny<5>(A, mstride, batch, conj, grad, perm, s);
    default: break;
  }
  const GradPlan p = grad_plan(n, batch, c_pref);
  int32_t rc = dispatch_grad(n, A, mstride, batch, p, conj, partial, grad, perm, s);
  if (rc || p.wpi == 1) return rc;
  hipLaunchKernelGGL(tb::grad_reduce_kernel, dim3((unsigned)((int64_t)batch * n)), dim3(256), 0, s,
                     partial, A, mstride, n, p.wpi, conj, grad, perm);
  return tbh::check_hip(hipGetLastError(), "grad_reduce_kernel");
}

}  // namespace tbgr
