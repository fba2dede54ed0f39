#pragma once
// Glynn permanents with a reflected Gray code, gfx950 (kernels and launch templates;
// instantiated by glynn_f64.hip and glynn_f32.hip).
//
// Restates GlynnGrayPermanentCalculator.compute_permanent
// (theboss/boson_sampling_utilities/permanent_calculators/glynn_gray_permanent_calculator.py:41-84):
//   perm(M) = 2^-(n-1) * sum_{delta in {+-1}^{n-1} x {+1}} (prod_i delta_i) prod_j sum_i delta_i M[i][j]
// enumerated in Gray order (one delta flip per term).
//
// Work split: the 2^(n-1) Gray ranks are cut into aligned chunks of 2^C ranks. One lane
// owns one chunk: it seeds its column sums at the chunk start in O(n^2) and then walks
// the chunk with O(n) updates per term. Because chunks are aligned, the row flipped at
// local step l is ctz(l) for every lane, so in WIDE mode (all 64 lanes of a wave on one
// matrix) the flipped row is wave-uniform. FP64 keeps the most frequently flipped rows
// (all static ones) in broadcast-form VGPRs (one DPP v_fmac_f64 per value, no LDS read)
// and reads the others from LDS as a broadcast; FP32 holds row 0 in VGPRs.
//
// Half column sums h_j = s_j / 2 are carried so a flip is a plain add/sub of M[i][j];
// perm = 2 * sum_t sign(t) prod_j h_j(t). sign(t) = (-1)^(popcount gray(t)) = (-1)^(t & 1).
#include <algorithm>

#include "flip_common.hpp"

namespace tb {

// FP64 wide kernels keep rows 0..U+1 in broadcast form up to this n, rows 0..U-1 above.
#ifndef TB_GLYNN_BCAST_WIDE_MAX_N
#define TB_GLYNN_BCAST_WIDE_MAX_N 24
#endif

// Occupancy target for the wide kernels: 2 waves per SIMD (<= 256 VGPRs).
#ifndef TB_WIDE_ATTR
#define TB_WIDE_ATTR(N) __attribute__((amdgpu_waves_per_eu((N) <= 40 ? 2 : 1)))
#endif

// Values of row 0 held in SGPRs by the WIDE kernels that keep no row in VGPRs (20
// complex values = 80 SGPRs; more spills SGPRs).
#ifndef TB_GLYNN_SROW
#define TB_GLYNN_SROW 20
#endif

// FP64 SMALL kernels from this n on give a matrix at least 16 lanes and hold its rows in
// broadcast form.
constexpr int kSmallBcastMinN = 7;

// Rows 0..R0-1 (the most frequently flipped: row i flips on 2^-(i+1) of all steps) are
// held in VGPRs; the rest are read from memory at each flip.
template <int N, int R0, typename F>
struct RegRows {
  F re[R0 > 0 ? R0 : 1][N], im[R0 > 0 ? R0 : 1][N];
};

// Rows 0..B-1 in broadcast form (FP64 only): every static flip and 3/4 of the
// block-start flips read no LDS.
template <int N, int B>
struct BcastRows {
  Bcast<N> r[B > 0 ? B : 1];
  double one;
};

template <int N, int R0, int S, int MODE, typename F, typename P, int B = 0>
__device__ __forceinline__ void flip_row(F (&hr)[N], F (&hi)[N], const RegRows<N, R0, F> &rr,
                                         const SRow<S, F> &sr, P M, int i, F sg,
                                         const BcastRows<N, B> *bs = nullptr) {
  if constexpr (B > 0) {
    if (i < B) {  // compile-time at the static flip sites, uniform at block starts
#pragma unroll
      for (int u = 0; u < B; ++u)
        if (u == i) flip_bcast<0, N, MODE>(hr, hi, bs->r[u], MODE == 0 ? sg : bs->one);
      return;
    }
  }
  if constexpr (S > 0) {
    if (i == 0) {
      flip_srow<N, S, MODE, F>(hr, hi, sr, M, sg);
      return;
    }
  }
  if constexpr (R0 > 0) {
    if (i < R0) {
      // i is a compile-time constant at every static flip site after unrolling.
#pragma unroll
      for (int r = 0; r < R0; ++r)
        if (r == i) flip_reg<N, MODE, F>(hr, hi, rr.re[r], rr.im[r], sg);
      return;
    }
  }
  flip_mem<N, MODE, F>(hr, hi, M + (size_t)i * N, sg);
}

// One lane walks `iters` chunks q = q0 + it*qstride of 2^C Gray ranks each; M is the
// n x n matrix as complex rows. `topbit_fixed` means C == N-1 (the whole enumeration in
// one chunk), so the Gray bit above the chunk is 0.
template <int N, int U, int R0, typename F, typename P, int S = 0, int B = 0>
__device__ __forceinline__ void glynn_lane(P M, int C, uint64_t q0, uint64_t qstride, int iters,
                                           double &acc_re, double &acc_im) {
  constexpr int NB = N - 1;  // Gray bits
  const bool topbit_fixed = (C == NB);
  SRow<S, F> sr;
  if constexpr (S > 0) load_srow(sr, M);
  BcastRows<N, B> bs;
  if constexpr (B > 0) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < B; ++u) load_bcast(bs.r[u], (const double *)(M + (size_t)u * N), lane);
    bs.one = vgpr_one();
    asm volatile("s_nop 4");  // VALU writes of the store before its first DPP read
  }
  RegRows<N, R0, F> rr;
  if constexpr (R0 > 0) {
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const cpx<F> v = M[(size_t)r * N + j];
        rr.re[r][j] = v.re;
        rr.im[r][j] = v.im;
      }
  }
  for (int it = 0; it < iters; ++it) {
    const uint64_t q = q0 + (uint64_t)it * qstride;
    const uint64_t t0 = q << C;
    const uint64_t g0 = t0 ^ (t0 >> 1);
    F hr[N], hi[N];
    if constexpr (B > 0) {
      seed_half_sums<N>(hr, hi, (const double *)(M + (size_t)(N - 1) * N), (const double *)M, NB, C, g0);
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const cpx<F> v = M[(size_t)(N - 1) * N + j];
        hr[j] = v.re;
        hi[j] = v.im;
      }
#pragma unroll 1
      for (int i = 0; i < NB; ++i) {
        const F sg = ((g0 >> i) & 1ull) ? F(-1) : F(1);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const cpx<F> v = M[(size_t)i * N + j];
          hr[j] = fma(sg, v.re, hr[j]);
          hi[j] = fma(sg, v.im, hi[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < N; ++j) {
        hr[j] *= F(0.5);
        hi[j] *= F(0.5);
      }
    }
    const bool q_odd = (q & 1ull) != 0;
    double cre, cim;
    {
      cpx<F> p = TreeProdT<F, 0, N>::run(hr, hi);
      cre = (double)p.re;
      cim = (double)p.im;
    }
    const int nblocks = 1 << (C - U);
    // Static steps j = 1 .. 2^U - 1 of block blk (row ctz(j) < U flips).
    auto static_steps = [&](int blk) {
#pragma unroll
      for (int j = 1; j < (1 << U); ++j) {
        const int i = __builtin_ctz(j);
        if (i + 1 < U) {
          // Direction fixed by the local bit i+1 of j.
          if ((j >> (i + 1)) & 1)
            flip_row<N, R0, S, 1, F, P, B>(hr, hi, rr, sr, M, i, F(1), &bs);
          else
            flip_row<N, R0, S, -1, F, P, B>(hr, hi, rr, sr, M, i, F(-1), &bs);
        } else {
          bool add;
          if (U < C)
            add = (blk & 1) != 0;
          else
            add = topbit_fixed ? false : q_odd;
          flip_row<N, R0, S, 0, F, P, B>(hr, hi, rr, sr, M, i, add ? F(1) : F(-1), &bs);
        }
        if constexpr (sizeof(F) == 8) {  // last multiply fused into the accumulation
          if (j & 1)
            tree_prod_acc<-1, 0, N>(cre, cim, (const double *)hr, (const double *)hi);
          else
            tree_prod_acc<1, 0, N>(cre, cim, (const double *)hr, (const double *)hi);
        } else {
          cpx<F> p = TreeProdT<F, 0, N>::run(hr, hi);
          if (j & 1) {
            cre -= (double)p.re;
            cim -= (double)p.im;
          } else {
            cre += (double)p.re;
            cim += (double)p.im;
          }
        }
        TB_STEP_FENCE();
      }
    };
    // Block 0 is peeled so the loop body is branch-free (no phi copies of h).
    static_steps(0);
    for (int blk = 1; blk < nblocks; ++blk) {
      const int i = U + __builtin_ctz(blk);
      bool add;
      if (i + 1 < C)
        add = ((blk >> (i + 1 - U)) & 1) != 0;
      else
        add = topbit_fixed ? false : q_odd;
      if constexpr (B > U) {
        if (i < B)
          flip_row<N, 0, 0, 0, F, P, B>(hr, hi, rr, sr, M, i, add ? F(1) : F(-1), &bs);
        else
          flip_mem<N, 0, F>(hr, hi, M + (size_t)i * N, add ? F(1) : F(-1));
      } else {
        flip_mem<N, 0, F>(hr, hi, M + (size_t)i * N, add ? F(1) : F(-1));
      }
      if constexpr (sizeof(F) == 8) {
        tree_prod_acc<1, 0, N>(cre, cim, (const double *)hr, (const double *)hi);
      } else {
        cpx<F> p = TreeProdT<F, 0, N>::run(hr, hi);
        cre += (double)p.re;
        cim += (double)p.im;
      }
      TB_STEP_FENCE();
      static_steps(blk);
    }
    acc_re += cre;
    acc_im += cim;
  }
}

// Wave of the workgroup, in an SGPR.
__device__ __forceinline__ int wave_in_block() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// The plain walk of one wave (wq of wpm) over the matrix in LDS.
template <int N, int U, int R0, typename F>
__device__ __forceinline__ void glynn_wide_walk(const cpx<F> *Ms, int C, int wq, int wpm, int iters,
                                                double &are, double &aim) {
  // R0 = 0: row 0's first values in SGPRs; 1: row 0 in VGPRs; 2 (FP64): rows 0..U+1
  // (n <= TB_GLYNN_BCAST_WIDE_MAX_N) or 0..U-1 in broadcast form; 3: rows 0..U-1 (every
  // static flip) in VGPRs.
  constexpr int S = (R0 == 0) ? TB_GLYNN_SROW : 0;
  constexpr int BW = (N <= TB_GLYNN_BCAST_WIDE_MAX_N) ? U + 2 : U;  // rows in broadcast form
  constexpr int B = (R0 == 2) ? (BW < N - 1 ? BW : N - 1) : 0;
  constexpr int RR = (R0 == 2) ? 0 : (R0 == 3 ? U : R0);  // rows in plain VGPRs
  glynn_lane<N, U, RR, F, const cpx<F> *, (S < N ? S : N), B>(
      Ms, C, (uint64_t)wq * 64 + (threadIdx.x & 63), (uint64_t)wpm * 64, iters, are, aim);
}

// A wave's sum goes to its partial; a matrix of one workgroup (wpm = 4) is summed here and
// needs no second launch. With the matrices that the paired walk cannot take walked in the same
// kernel that is one launch instead of three: 256 matrices of n = 14 take 14 us, not 28.
__device__ __forceinline__ void glynn_store(double re, double im, int b, int wq, int wpm, cd *sums,
                                            cd *__restrict__ partial, cd *__restrict__ out) {
  const bool first = (threadIdx.x & 63) == 0;
  if (wpm > 4) {
    if (first) partial[(size_t)b * wpm + wq] = {re, im};
    return;
  }
  if (first) sums[wq & 3] = {re, im};
  __syncthreads();
  if (threadIdx.x == 0) {
    const cd t = cadd(cadd(sums[0], sums[1]), cadd(sums[2], sums[3]));
    out[b] = {2.0 * t.re, 2.0 * t.im};
  }
}

// WIDE: the 4 waves of a workgroup share one matrix, staged once into LDS (and converted on
// the way for FP32 column sums); every flip is a broadcast LDS read. Grid: batch * (wpm/4)
// workgroups; wave wq of matrix b covers chunks q = (wq + it*wpm)*64 + lane. Strides count
// complex elements. `handled` (may be null): matrices the paired kernel already did.
template <int N, int U, int R0, typename F>
__global__ __launch_bounds__(256) TB_WIDE_ATTR(N) void glynn_wide_kernel(const cd *__restrict__ A,
                                                         int64_t mstride, int C, int wpm, int iters,
                                                         cd *__restrict__ partial,
                                                         const int *__restrict__ handled,
                                                         cd *__restrict__ out) {
  __shared__ cpx<F> Ms[N * N];
  __shared__ cd sums[4];
  const int wgs_per_matrix = wpm >> 2;
  const int b = blockIdx.x / wgs_per_matrix;
  if (handled != nullptr && handled[b] != 0) return;
  const int wq = (blockIdx.x - b * wgs_per_matrix) * 4 + wave_in_block();
  const cd *src = A + (size_t)b * mstride;
  for (int e = threadIdx.x; e < N * N; e += 256) Ms[e] = {(F)src[e].re, (F)src[e].im};
  __syncthreads();
  double are = 0.0, aim = 0.0;
  glynn_wide_walk<N, U, R0, F>(Ms, C, wq, wpm, iters, are, aim);
  glynn_store(wave_sum(are), wave_sum(aim), b, wq, wpm, sums, partial, out);
}

// ------------------------------------------------------------------------------------
// Paired Gray walk (FP64 WIDE). Gray codes 2t and 2t+1 differ only in row 0. With row
// N-1 fixed (delta = +1) and u_j = sum_{i >= 1} delta_i M[i][j] / M[0][j], their half
// column sums are h_j = (M[0][j] / 2)(u_j + 1) and (M[0][j] / 2)(u_j - 1), so
//   perm = 2 K sum_t (-1)^t [prod_j (u_j + 1) - prod_j (u_j - 1)],  K = prod_j M[0][j] / 2,
// over the 2^(N-2) Gray ranks t of rows 1..N-2. A flip of row i adds +-2 M[i][j] / M[0][j]
// to every u_j (one update for both codes), and a factor (u_j +- 1) enters a running
// product x as x u_j +- x: four FMAs with the +-1 folded into their addends. A pair of
// codes costs 2N flip instructions and 2 (4N - 2) product instructions (each product two
// chains of N/2 factors, joined by a multiply fused into the accumulation) against
// 2 (6N - 4) for two plain steps. The row whose smallest entry is largest becomes row 0
// (a row permutation leaves the permanent unchanged); a matrix none of whose rows has all
// entries above 2^-16 of its largest entry (zeros included) is left to the plain kernel.
// ------------------------------------------------------------------------------------

// acc += SIGN * (prod (u + 1) - prod (u - 1)).
template <int SIGN, int N>
__device__ __forceinline__ void pair_acc(double &ar, double &ai, const double (&ur)[N],
                                         const double (&ui)[N]) {
  constexpr int H = N / 2;
  const cd ap = fold_chain<1, 0, H>(ur, ui), bp = fold_chain<1, H, N>(ur, ui);
  const cd am = fold_chain<-1, 0, H>(ur, ui), bm = fold_chain<-1, H, N>(ur, ui);
  cmul_acc<SIGN>(ar, ai, ap, bp);
  cmul_acc<-SIGN>(ar, ai, am, bm);
}

// u += sg * row i + 1 of S2 (rows 1..B in broadcast form, the others from LDS).
template <int N, int MODE, int B>
__device__ __forceinline__ void pair_flip(double (&ur)[N], double (&ui)[N], const BcastRows<N, B> &bs,
                                          const cpx<double> *S2, int i, double sg) {
  if constexpr (B > 0) {
    if (i < B) {  // compile-time at the static flip sites, uniform at block starts
#pragma unroll
      for (int u = 0; u < B; ++u)
        if (u == i) flip_bcast<0, N, MODE>(ur, ui, bs.r[u], MODE == 0 ? sg : bs.one);
      return;
    }
  }
  flip_mem<N, MODE, double>(ur, ui, S2 + (size_t)(i + 1) * N, sg);
}

// One lane walks `iters` chunks q = q0 + it*qstride of 2^C super-steps (Gray ranks of rows
// 1..N-2) each; S2 holds 2 M[i][j] / M[0][j] in rows 1..N-1. Same chunk, block and
// direction structure as glynn_lane with row i + 1 at Gray bit i.
template <int N, int U, int B>
__device__ __forceinline__ void glynn_pair_lane(const cpx<double> *S2, int C, uint64_t q0,
                                                uint64_t qstride, int iters, double &acc_re,
                                                double &acc_im) {
  constexpr int NB = N - 2;  // Gray bits
  const bool topbit_fixed = (C == NB);
  BcastRows<N, B> bs;
  if constexpr (B > 0) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < B; ++u)
      load_bcast(bs.r[u], (const double *)(S2 + (size_t)(u + 1) * N), lane);
    bs.one = vgpr_one();
    asm volatile("s_nop 4");  // VALU writes of the store before its first DPP read
  }
  for (int it = 0; it < iters; ++it) {
    const uint64_t q = q0 + (uint64_t)it * qstride;
    const uint64_t t0 = q << C;
    const uint64_t g0 = t0 ^ (t0 >> 1);
    double ur[N], ui[N];
    seed_half_sums<N>(ur, ui, (const double *)(S2 + (size_t)(N - 1) * N), (const double *)(S2 + N), NB,
                      C, g0);
    const bool q_odd = (q & 1ull) != 0;
    double cre = 0.0, cim = 0.0;
    pair_acc<1>(cre, cim, ur, ui);
    const int nblocks = 1 << (C - U);
    auto static_steps = [&](int blk) {
#pragma unroll
      for (int j = 1; j < (1 << U); ++j) {
        const int i = __builtin_ctz(j);
        if (i + 1 < U) {
          if ((j >> (i + 1)) & 1)
            pair_flip<N, 1, B>(ur, ui, bs, S2, i, 1.0);
          else
            pair_flip<N, -1, B>(ur, ui, bs, S2, i, -1.0);
        } else {
          bool add;
          if (U < C)
            add = (blk & 1) != 0;
          else
            add = topbit_fixed ? false : q_odd;
          pair_flip<N, 0, B>(ur, ui, bs, S2, i, add ? 1.0 : -1.0);
        }
        if (j & 1)
          pair_acc<-1>(cre, cim, ur, ui);
        else
          pair_acc<1>(cre, cim, ur, ui);
        TB_STEP_FENCE();
      }
    };
    static_steps(0);
    for (int blk = 1; blk < nblocks; ++blk) {
      const int i = U + __builtin_ctz(blk);
      bool add;
      if (i + 1 < C)
        add = ((blk >> (i + 1 - U)) & 1) != 0;
      else
        add = topbit_fixed ? false : q_odd;
      if constexpr (B > U) {
        if (i < B)
          pair_flip<N, 0, B>(ur, ui, bs, S2, i, add ? 1.0 : -1.0);
        else
          flip_mem<N, 0, double>(ur, ui, S2 + (size_t)(i + 1) * N, add ? 1.0 : -1.0);
      } else {
        flip_mem<N, 0, double>(ur, ui, S2 + (size_t)(i + 1) * N, add ? 1.0 : -1.0);
      }
      pair_acc<1>(cre, cim, ur, ui);
      TB_STEP_FENCE();
      static_steps(blk);
    }
    acc_re += cre;
    acc_im += cim;
  }
}

// The pair row of the matrix in Ms (its row with the largest smallest entry, row r), or -1
// where that is too small against the largest entry of all: the same value in every wave.
// Four lanes look at each row, and every wave then compares the rows itself. rmin, rmax: N
// values each. Ends with the barrier between the looks and the compare only.
template <int N>
__device__ __forceinline__ int pair_row(const cd *Ms, double *rmin, double *rmax) {
  if (threadIdx.x < 4 * N) {
    const int row = threadIdx.x >> 2;
    double lo = INFINITY, hi = 0.0;  // of the squared magnitudes
    for (int j = threadIdx.x & 3; j < N; j += 4) {
      const cd v = Ms[row * N + j];
      const double a = fma(v.re, v.re, v.im * v.im);
      lo = fmin(lo, a);
      hi = fmax(hi, a);
    }
    lo = fmin(lo, dpp_perm<0xb1>(lo));  // quad_perm 1,0,3,2 and 2,3,0,1
    hi = fmax(hi, dpp_perm<0xb1>(hi));
    lo = fmin(lo, dpp_perm<0x4e>(lo));
    hi = fmax(hi, dpp_perm<0x4e>(hi));
    if ((threadIdx.x & 3) == 0) {
      rmin[row] = lo;
      rmax[row] = hi;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const double mn = lane < N ? rmin[lane] : -1.0, mx = lane < N ? rmax[lane] : 0.0;
  const double top = wave_allmax(mx), best = wave_allmax(mn);
  if (!(top > 0.0 && top <= 1.7976931348623157e308 && best >= kPairMinRel2 * top)) return -1;
  return __ffsll((unsigned long long)__ballot(mn == best)) - 1;  // the first such row
}

// Wave 0: swaps row r with row 0, whose old entries go to row r, and leaves the reciprocals
// of the new row 0 in inv0 (scaled by a power of two so that the square stays in range) and
// K = prod_j M[0][j] / 2 as Km 2^Ke. Row 0 itself is not written back.
template <int N>
__device__ __forceinline__ void pair_divisors(cd *Ms, int r, cd *inv0, cd *Km, int *Ke) {
  const int lane = threadIdx.x;
  cd m = {1.0, 0.0};
  double e = 0.0;
  if (lane < N) {
    const cd v = Ms[r * N + lane];
    if (r != 0) Ms[r * N + lane] = Ms[lane];
    const int ex = ilogb(fmax(fabs(v.re), fabs(v.im)));
    m = {ldexp(v.re, -ex), ldexp(v.im, -ex)};
    const double d = fma(m.re, m.re, m.im * m.im);
    inv0[lane] = {ldexp(m.re / d, -ex), ldexp(-m.im / d, -ex)};
    e = (double)ex;
  }
  const cd k = wave_prod(m);  // below 2^60: each mantissa is at most 2 sqrt 2
  const double ke = wave_allsum(e);
  if (lane == 0) {
    *Km = k;
    *Ke = (int)ke - N;
  }
}

// PAIRED WIDE kernel: grid, chunks and partial layout of glynn_wide_kernel with C Gray
// bits per chunk of codes (C - 1 super-step bits). A matrix without a pair row takes the
// plain walk (U0 static bits) in the same workgroups.
template <int N, int U, int B, int U0, int R0>
__global__ __launch_bounds__(256) TB_WIDE_ATTR(N) void glynn_pair_kernel(
    const cd *__restrict__ A, int64_t mstride, int C, int wpm, int iters, cd *__restrict__ partial,
    cd *__restrict__ out) {
  __shared__ cd Ms[N * N];
  __shared__ cd inv0[N];
  __shared__ double rmin[N], rmax[N];
  __shared__ int Ke;
  __shared__ cd Km;
  __shared__ cd sums[4];
  const int lane = threadIdx.x & 63;
  const int wgs_per_matrix = wpm >> 2;
  const int b = blockIdx.x / wgs_per_matrix;
  const int wq = (blockIdx.x - b * wgs_per_matrix) * 4 + wave_in_block();
  const cd *src = A + (size_t)b * mstride;
  for (int e = threadIdx.x; e < N * N; e += 256) Ms[e] = src[e];
  __syncthreads();
  const int r = pair_row<N>(Ms, rmin, rmax);
  double are = 0.0, aim = 0.0;
  if (r < 0) {  // uniform over the workgroup
    glynn_wide_walk<N, U0, R0, double>((const cpx<double> *)Ms, C, wq, wpm, iters, are, aim);
    glynn_store(wave_sum(are), wave_sum(aim), b, wq, wpm, sums, partial, out);
    return;
  }
  if (threadIdx.x < 64) pair_divisors<N>(Ms, r, inv0, &Km, &Ke);
  __syncthreads();
  for (int e = N + threadIdx.x; e < N * N; e += 256) {
    const cd v = cmul(Ms[e], inv0[e % N]);
    Ms[e] = {2.0 * v.re, 2.0 * v.im};
  }
  __syncthreads();
  glynn_pair_lane<N, U, B>((const cpx<double> *)Ms, C - 1, (uint64_t)wq * 64 + lane,
                           (uint64_t)wpm * 64, iters, are, aim);
  are = wave_sum(are);
  aim = wave_sum(aim);
  const cd k = Km;
  glynn_store(ldexp(k.re * are - k.im * aim, Ke), ldexp(k.re * aim + k.im * are, Ke), b, wq, wpm,
              sums, partial, out);
}

// ------------------------------------------------------------------------------------
// Paired walk with FP32 column sums and products (14 <= n <= TB_FP32_COLSUM_MAX_N): the
// walk of glynn_pair_lane in float, the quotients 2 M[i][j] / M[0][j] formed in FP64 and
// rounded once; static row 1 in SGPRs (SR = 1), rows SR + 1..U in plain VGPRs. Each pair's
// difference prod(u + 1) - prod(u - 1) is formed in FP32, summed in FP32 over the 2^U
// pairs of a block and accumulated in FP64 once per block.
// ------------------------------------------------------------------------------------
// Complex values per LDS read group of the paired FP32 kernel's memory flips (two
// groups in flight).
#ifndef TB_GLYNN_F32_PAIR_FLIP_G
#define TB_GLYNN_F32_PAIR_FLIP_G 4
#endif
// One step of the chain x <- x (u + PM), split in its two FMA levels.
template <int PM>
__device__ __forceinline__ void chain_lvl1(float xr, float xi, float u_r, float u_i, float &tr,
                                           float &ti) {
  tr = fmaf(xr, u_r, (float)PM * xr);
  ti = fmaf(xr, u_i, (float)PM * xi);
}
__device__ __forceinline__ void chain_lvl2(float &xr, float &xi, float u_r, float u_i, float tr,
                                           float ti) {
  const float nr = fmaf(-xi, u_i, tr);
  xi = fmaf(xi, u_r, ti);
  xr = nr;
}

// SIGN * (Π(u + 1) - Π(u - 1)) added to the FP32 block sums (ar, ai). Four chains run side by side, Π(u ± 1)
// over columns [0, H) and [H, N): a chain step is two dependent FMA levels, and FP32
// issues fast enough that one chain alone waits on its own results; with the four
// interleaved level by level, each FMA's operand was produced eight instructions earlier.
template <int SIGN, int N>
__device__ __forceinline__ void pair_acc_f32(float &ar, float &ai, const float (&ur)[N],
                                             const float (&ui)[N]) {
  constexpr int H = N / 2;  // the upper half is the longer one for odd N
  float pr = ur[0] + 1.f, pi = ui[0];  // (u + 1), columns [0, H)
  float qr = ur[H] + 1.f, qi = ui[H];  // (u + 1), columns [H, N)
  float mr = ur[0] - 1.f, mi = ui[0];  // (u - 1), columns [0, H)
  float wr = ur[H] - 1.f, wi = ui[H];  // (u - 1), columns [H, N)
#pragma unroll
  for (int k = 1; k < N - H; ++k) {
    float t[8];
    if (k < H) {
      chain_lvl1<1>(pr, pi, ur[k], ui[k], t[0], t[1]);
      chain_lvl1<-1>(mr, mi, ur[k], ui[k], t[4], t[5]);
    }
    chain_lvl1<1>(qr, qi, ur[H + k], ui[H + k], t[2], t[3]);
    chain_lvl1<-1>(wr, wi, ur[H + k], ui[H + k], t[6], t[7]);
    if (k < H) {
      chain_lvl2(pr, pi, ur[k], ui[k], t[0], t[1]);
      chain_lvl2(mr, mi, ur[k], ui[k], t[4], t[5]);
    }
    chain_lvl2(qr, qi, ur[H + k], ui[H + k], t[2], t[3]);
    chain_lvl2(wr, wi, ur[H + k], ui[H + k], t[6], t[7]);
  }
  // (p q) - (m w) with the difference folded into the FMAs
  const float mwr = fmaf(-mi, wi, mr * wr), mwi = fmaf(mi, wr, mr * wi);
  const float dr = fmaf(pr, qr, -fmaf(pi, qi, mwr));
  const float di = fmaf(pr, qi, fmaf(pi, qr, -mwi));
  if constexpr (SIGN > 0) {
    ar += dr;
    ai += di;
  } else {
    ar -= dr;
    ai -= di;
  }
}

// h += v, h -= v or h += sg v for the static row whose first S values sit in SGPRs (s)
// and the rest in VGPRs (rr, ri; entries below S unused).
template <int N, int MODE, int S>
__device__ __forceinline__ void flip_split_f32(float (&hr)[N], float (&hi)[N],
                                               const SRow<S, float> &s, const float (&rr)[N],
                                               const float (&ri)[N], float sg) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float vr = j < S ? s.re[j < S ? j : 0] : rr[j];
    const float vi = j < S ? s.im[j < S ? j : 0] : ri[j];
    if constexpr (MODE == 1) {
      hr[j] += vr;
      hi[j] += vi;
    } else if constexpr (MODE == -1) {
      hr[j] -= vr;
      hi[j] -= vi;
    } else {
      hr[j] = fmaf(sg, vr, hr[j]);
      hi[j] = fmaf(sg, vi, hi[j]);
    }
  }
}

template <int N, int U, int SR, int S2P>
__device__ __forceinline__ void glynn_pair_lane_f32(const cpx<float> *S2, int C, uint64_t q0,
                                                    uint64_t qstride, int iters, double &acc_re,
                                                    double &acc_im) {
  constexpr int NB = N - 2;  // Gray bits: row i + 1 at bit i
  const bool topbit_fixed = (C == NB);
  // Static row SR (row 1 flips on half of all pairs, row 2 on a quarter) in SGPRs when
  // SR > 0, as the scalar operand of the adds (an FP32 instruction with an SGPR operand
  // does not dual-issue, so the register it frees costs issue rate); the other static
  // rows in VGPRs, except the first S2P values of row 2 beside an SGPR row 1.
  static_assert(SR <= U, "the SGPR row is a static row");
  static_assert(S2P == 0 || (SR == 1 && U >= 2), "row 2 splits only beside an SGPR row 1");
  constexpr int NR = U - (SR ? 1 : 0);  // static rows in VGPRs
  SRow<SR ? N : 0, float> sr;
  if constexpr (SR) load_srow<N>(sr, S2 + (size_t)SR * N);
  SRow<S2P, float> sr2;
  if constexpr (S2P > 0) load_srow<S2P>(sr2, S2 + 2 * N);
  RegRows<N, NR, float> rr;  // rr[r]: static row index r, skipping SR - 1
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (r == 0 && j < S2P) continue;
      const int i = (SR && r >= SR - 1) ? r + 1 : r;
      const cpx<float> v = S2[(size_t)(i + 1) * N + j];
      rr.re[r][j] = v.re;
      rr.im[r][j] = v.im;
    }
  for (int it = 0; it < iters; ++it) {
    const uint64_t q = q0 + (uint64_t)it * qstride;
    const uint64_t t0 = q << C;
    const uint64_t g0 = t0 ^ (t0 >> 1);
    float ur[N], ui[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const cpx<float> v = S2[(size_t)(N - 1) * N + j];
      ur[j] = v.re;
      ui[j] = v.im;
    }
#pragma unroll 1
    for (int i = 0; i < NB; ++i) {
      const float sg = ((g0 >> i) & 1ull) ? -1.0f : 1.0f;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const cpx<float> v = S2[(size_t)(i + 1) * N + j];
        ur[j] = fmaf(sg, v.re, ur[j]);
        ui[j] = fmaf(sg, v.im, ui[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      ur[j] *= 0.5f;
      ui[j] *= 0.5f;
    }
    const bool q_odd = (q & 1ull) != 0;
    // Each block's pair terms (the block-start pair and the 2^U - 1 static ones) are
    // summed in FP32, then added to the FP64 lane sums: one conversion and one FP64 add
    // per block and component.
    float bre = 0.f, bim = 0.f;
    pair_acc_f32<1>(bre, bim, ur, ui);
    const int nblocks = 1 << (C - U);
    // row i + 1: mode +1 / -1 (fixed direction) or 0 (direction sg); every call site
    // passes constants, so the branches fold away after unrolling
    auto do_flip = [&](int i, int mode, float sg) {
      if (SR && i == SR - 1) {
        if constexpr (SR) {
          if (mode == 1)
            flip_reg<N, 1, float>(ur, ui, sr.re, sr.im, sg);
          else if (mode == -1)
            flip_reg<N, -1, float>(ur, ui, sr.re, sr.im, sg);
          else
            flip_reg<N, 0, float>(ur, ui, sr.re, sr.im, sg);
        }
        return;
      }
      if (S2P > 0 && i == 1) {
        if constexpr (S2P > 0) {
          if (mode == 1)
            flip_split_f32<N, 1, S2P>(ur, ui, sr2, rr.re[0], rr.im[0], sg);
          else if (mode == -1)
            flip_split_f32<N, -1, S2P>(ur, ui, sr2, rr.re[0], rr.im[0], sg);
          else
            flip_split_f32<N, 0, S2P>(ur, ui, sr2, rr.re[0], rr.im[0], sg);
        }
        return;
      }
      if (i < U) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (((SR && r >= SR - 1) ? r + 1 : r) == i) {
            if (mode == 1)
              flip_reg<N, 1, float>(ur, ui, rr.re[r], rr.im[r], sg);
            else if (mode == -1)
              flip_reg<N, -1, float>(ur, ui, rr.re[r], rr.im[r], sg);
            else
              flip_reg<N, 0, float>(ur, ui, rr.re[r], rr.im[r], sg);
          }
        return;
      }
      flip_mem<N, 0, float, const cpx<float> *, 0, TB_GLYNN_F32_PAIR_FLIP_G>(ur, ui, S2 + (size_t)(i + 1) * N, sg);
    };
    auto static_steps = [&](int blk) {
#pragma unroll
      for (int j = 1; j < (1 << U); ++j) {
        const int i = __builtin_ctz(j);
        if (i + 1 < U) {
          if ((j >> (i + 1)) & 1)
            do_flip(i, 1, 1.0f);
          else
            do_flip(i, -1, -1.0f);
        } else {
          bool add;
          if (U < C)
            add = (blk & 1) != 0;
          else
            add = topbit_fixed ? false : q_odd;
          do_flip(i, 0, add ? 1.0f : -1.0f);
        }
        if (j & 1)
          pair_acc_f32<-1>(bre, bim, ur, ui);
        else
          pair_acc_f32<1>(bre, bim, ur, ui);
        TB_STEP_FENCE();
      }
      acc_re += (double)bre;
      acc_im += (double)bim;
      bre = 0.f;
      bim = 0.f;
    };
    static_steps(0);
    for (int blk = 1; blk < nblocks; ++blk) {
      const int i = U + __builtin_ctz(blk);
      bool add;
      if (i + 1 < C)
        add = ((blk >> (i + 1 - U)) & 1) != 0;
      else
        add = topbit_fixed ? false : q_odd;
      flip_mem<N, 0, float, const cpx<float> *, 0, TB_GLYNN_F32_PAIR_FLIP_G>(ur, ui, S2 + (size_t)(i + 1) * N, add ? 1.0f : -1.0f);
      pair_acc_f32<1>(bre, bim, ur, ui);
      TB_STEP_FENCE();
      static_steps(blk);
    }
  }
}

// PAIRED WIDE kernel, FP32 column sums: reads the FP64 matrices (the quotients and the
// row-0 product are formed in FP64). A matrix without a pair row is left to the plain kernel
// (handled[b] = 0, else 1), whose rows need more registers than this kernel's waves have.
template <int N, int U, int SR, int S2P, int WPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void glynn_pair_kernel_f32(
    const cd *__restrict__ A, int64_t mstride, int C, int wpm, int iters,
    cd *__restrict__ partial, int *__restrict__ handled, cd *__restrict__ out) {
  __shared__ cd Ms[N * N];
  __shared__ cpx<float> Sf[N * N];
  __shared__ cd inv0[N];
  __shared__ double rmin[N], rmax[N];
  __shared__ int Ke;
  __shared__ cd Km;
  __shared__ cd sums[4];
  const int lane = threadIdx.x & 63;
  const int wgs_per_matrix = wpm >> 2;
  const int b = blockIdx.x / wgs_per_matrix;
  const int wg = blockIdx.x - b * wgs_per_matrix;
  const int wq = wg * 4 + wave_in_block();
  const cd *src = A + (size_t)b * mstride;
  for (int e = threadIdx.x; e < N * N; e += 256) Ms[e] = src[e];
  __syncthreads();
  const int r = pair_row<N>(Ms, rmin, rmax);
  if (wg == 0 && threadIdx.x == 0) handled[b] = r < 0 ? 0 : 1;
  if (r < 0) return;  // uniform over the workgroup
  if (threadIdx.x < 64) pair_divisors<N>(Ms, r, inv0, &Km, &Ke);
  __syncthreads();
  for (int e = N + threadIdx.x; e < N * N; e += 256) {
    const cd v = cmul(Ms[e], inv0[e % N]);
    Sf[e] = {(float)(2.0 * v.re), (float)(2.0 * v.im)};
  }
  __syncthreads();
  double are = 0.0, aim = 0.0;
  glynn_pair_lane_f32<N, U, SR, S2P>(Sf, C - 1, (uint64_t)wq * 64 + lane, (uint64_t)wpm * 64, iters, are, aim);
  are = wave_sum(are);
  aim = wave_sum(aim);
  const cd k = Km;
  glynn_store(ldexp(k.re * are - k.im * aim, Ke), ldexp(k.re * aim + k.im * are, Ke), b, wq, wpm,
              sums, partial, out);
}

// One row of a matrix in LDS in broadcast form, each 16-lane row of the wave from its own M.
template <int N>
__device__ __forceinline__ Bcast<N> row_bcast(const cpx<double> *M, int i) {
  const int lane = threadIdx.x & 15;
  Bcast<N> b;
#pragma unroll
  for (int p = 0; p < Bcast<N>::P; ++p) {
    const int t = 16 * p + lane;
    b.v[p] = ((const double *)(M + i * N))[t < 2 * N ? t : 2 * N - 1];
  }
  return b;
}
// Two wait states between whatever wrote the row's registers and its DPP reads (N <= 16).
template <int N>
__device__ __forceinline__ void bcast_ready(Bcast<N> &b) {
  asm volatile("s_nop 1" : "+v"(b.v[0]), "+v"(b.v[Bcast<N>::P - 1]));
}

// glynn_lane with every row in broadcast form, for matrices that own whole 16-lane rows: the
// U static rows stay in registers, the others are loaded (2 values per lane instead of N
// complex ones) a row ahead of the flip that adds them.
template <int N, int U>
__device__ __forceinline__ void glynn_bcast_lane(const cpx<double> *M, int C, uint32_t q,
                                                 double &acc_re, double &acc_im) {
  constexpr int NB = N - 1;
  const uint32_t t0 = q << C, g0 = t0 ^ (t0 >> 1);
  const bool q_odd = (q & 1u) != 0;  // the Gray bit above the chunk
  Bcast<N> rows[U];
#pragma unroll
  for (int u = 0; u < U; ++u) rows[u] = row_bcast<N>(M, u);
  const double one = vgpr_one();
  double hr[N], hi[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    hr[j] = 0.0;
    hi[j] = 0.0;
  }
  Bcast<N> next = row_bcast<N>(M, NB);
#pragma unroll 1
  for (int i = NB; i >= 0; --i) {  // half column sums at t0, the fixed row first
    Bcast<N> row = next;
    next = row_bcast<N>(M, i > 0 ? i - 1 : (U < NB ? U : 0));
    const double d = (i < NB && ((g0 >> i) & 1u)) ? -0.5 : 0.5;
    bcast_ready(row);
    flip_bcast<0, N, 0>(hr, hi, row, d);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) bcast_ready(rows[u]);
  const cd p0 = TreeProd<0, N>::run(hr, hi);
  double cre = p0.re, cim = p0.im;
  const int nblocks = 1 << (C - U);
  auto static_steps = [&](int blk) {
#pragma unroll
    for (int j = 1; j < (1 << U); ++j) {
      const int i = __builtin_ctz(j);
      if (i + 1 < U) {
        if ((j >> (i + 1)) & 1)
          flip_bcast<0, N, 1>(hr, hi, rows[i], one);
        else
          flip_bcast<0, N, -1>(hr, hi, rows[i], one);
      } else {
        const bool add = (U < C) ? (blk & 1) != 0 : q_odd;
        flip_bcast<0, N, 0>(hr, hi, rows[i], add ? 1.0 : -1.0);
      }
      if (j & 1)
        tree_prod_acc<-1, 0, N>(cre, cim, hr, hi);
      else
        tree_prod_acc<1, 0, N>(cre, cim, hr, hi);
      TB_STEP_FENCE();
    }
  };
  static_steps(0);
  for (int blk = 1; blk < nblocks; ++blk) {
    const int i = U + __builtin_ctz(blk);
    const bool add = i + 1 < C ? ((blk >> (i + 1 - U)) & 1) != 0 : q_odd;
    Bcast<N> row = next;
    next = row_bcast<N>(M, U + __builtin_ctz(blk + 1 < nblocks ? blk + 1 : 1));
    bcast_ready(row);
    flip_bcast<0, N, 0>(hr, hi, row, add ? 1.0 : -1.0);
    tree_prod_acc<1, 0, N>(cre, cim, hr, hi);
    TB_STEP_FENCE();
    static_steps(blk);
  }
  acc_re += cre;
  acc_im += cim;
}

// SMALL (n < kWideMinN): 2^(N-1-C) lanes per matrix, each walking one chunk of 2^C ranks, 256
// lanes per workgroup; the matrices are staged in LDS (one complex value of padding each, so
// that the groups of a wave read different banks) and the lanes' sums added up by shuffles,
// beyond a wave through LDS. One launch, no partial sums in memory.
// What bounds it: latency and, in large batches, VALU issue. Against one lane per matrix with
// its rows in global memory (n <= 10) and 4 waves per matrix, an idle fallback launch and a
// finishing one (n = 11..13), times from Python, where an empty call takes 9 us: one n = 10
// matrix 76 -> 9 us, 20,000 of them 140 -> 29; one n = 12 matrix 14 -> 9, 20,000: 203 -> 112.
// From LDS rows instead of broadcast ones, 1000 n = 13 matrices took 28 us (15; 21 before):
// the seeds' N^2 16-byte broadcast reads per lane held the LDS return path.
template <int N, int U, typename F>
__global__ __launch_bounds__(256) void glynn_small_kernel(const cd *__restrict__ A, int64_t mstride,
                                                          int batch, int C, cd *__restrict__ out) {
  constexpr int NB = N - 1, MS = N * N + 1;
  extern __shared__ char small_lds[];
  cpx<F> *Ms = (cpx<F> *)small_lds;
  __shared__ double wave_re[4], wave_im[4];
  const int tid = threadIdx.x;
  const int wbits = NB - C, W = 1 << wbits;  // lanes per matrix, 1..256
  const int mats = 256 >> wbits;
  const int b0 = blockIdx.x * mats;
  const int here = min(mats, batch - b0);
  for (int e = tid; e < here * N * N; e += 256) {
    const int k = e / (N * N), r = e - k * (N * N);
    const cd v = A[(size_t)(b0 + k) * mstride + r];
    Ms[k * MS + r] = {(F)v.re, (F)v.im};
  }
  __syncthreads();
  const int g = min(tid >> wbits, here - 1);  // idle groups repeat the last matrix
  const int q = tid & (W - 1);
  double are = 0.0, aim = 0.0;
  if constexpr (sizeof(F) == 8 && N >= kSmallBcastMinN)
    glynn_bcast_lane<N, U>((const cpx<double> *)(Ms + g * MS), C, (uint32_t)q, are, aim);
  else
    glynn_lane<N, U, 1, F>((const cpx<F> *)(Ms + g * MS), C, (uint64_t)q, 0, 1, are, aim);
  for (int off = min(W, 64) >> 1; off >= 1; off >>= 1) {
    are += __shfl_xor(are, off, 64);
    aim += __shfl_xor(aim, off, 64);
  }
  if (W > 64) {  // uniform over the launch
    if ((tid & 63) == 0) {
      wave_re[tid >> 6] = are;
      wave_im[tid >> 6] = aim;
    }
    __syncthreads();
    if (q == 0)
      for (int w = 1; w < W >> 6; ++w) {
        are += wave_re[(tid >> 6) + w];
        aim += wave_im[(tid >> 6) + w];
      }
  }
  if (q == 0 && (tid >> wbits) < here) out[b0 + g] = {2.0 * are, 2.0 * aim};
}

namespace {  // internal linkage: each translation unit keeps its own copy

// Sum the wpm wave partials of each matrix in a fixed order: deterministic results.
__global__ __launch_bounds__(256) void glynn_finish_kernel(const cd *__restrict__ partial, int wpm,
                                                           int batch, cd *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= batch) return;
  double re = 0.0, im = 0.0;
  for (int w = lane; w < wpm; w += 64) {
    re += partial[(size_t)b * wpm + w].re;
    im += partial[(size_t)b * wpm + w].im;
  }
  re = wave_sum(re);
  im = wave_sum(im);
  if (lane == 0) out[b] = {2.0 * re, 2.0 * im};
}

__global__ void fill_one_kernel(cd *out, int batch) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < batch) out[b] = {1.0, 0.0};
}

__global__ void copy_scalar_kernel(const cd *A, int64_t mstride, int batch, cd *out) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < batch) out[b] = A[(size_t)b * mstride];
}

}  // namespace

}  // namespace tb

// ------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------
namespace tbgl {

// Rows held in VGPRs by the WIDE kernel: row 0 (flipped on half of all steps) when the
// register budget of 2 waves per SIMD allows it -- FP32 always, FP64 up to n = 24.
#ifndef TB_GLYNN_F64_R0_MAX_N
#define TB_GLYNN_F64_R0_MAX_N 24
#endif
// Up to n = 40 the broadcast rows stay in VGPRs; above, the compiler parks them in AGPRs
// and copies them back right before the DPP reads (a VALU write the DPP read must not
// follow within 2 wait states), so larger n keep row 0 in SGPRs instead.
#ifndef TB_GLYNN_F64_BCAST_MAX_N
#define TB_GLYNN_F64_BCAST_MAX_N 40
#endif
// FP32 rows cost half the registers: up to TB_GLYNN_F32_ROWS_MAX_N the FP32 kernels keep
// every static row (0..U-1) in VGPRs, so only block-start flips read LDS.
#ifndef TB_GLYNN_F32_ROWS_MAX_N
#define TB_GLYNN_F32_ROWS_MAX_N 24
#endif
template <int N, typename F>
constexpr int glynn_reg_rows() {
  if (sizeof(F) == 8 && N <= TB_GLYNN_F64_BCAST_MAX_N) return 2;
  if (sizeof(F) == 4) return N <= TB_GLYNN_F32_ROWS_MAX_N ? 3 : 1;
  return N <= TB_GLYNN_F64_R0_MAX_N ? 1 : 0;
}

// Static Gray bits (unrolled block of 2^U steps) of the WIDE kernels: FP64 at n >= 25,
// whose static rows are all in broadcast form, unrolls TB_GLYNN_U_LARGE bits.
#ifndef TB_GLYNN_U_LARGE
#define TB_GLYNN_U_LARGE 3
#endif
// Static Gray bits of the FP32 kernels that keep their static rows in VGPRs: 3 (7/8 of
// the flips from registers; measured 1.05x at n = 20, 1.11x at n = 23 over row 0 alone).
// The plan keeps at least 2^8 chunks per matrix (C <= n - 9) and needs C >= U, so U = 3
// starts at n = 12.
#ifndef TB_GLYNN_F32_U
#define TB_GLYNN_F32_U 3
#endif
// The paired FP32 kernel: 2 static Gray bits, static row SR in SGPRs (row 1 by default)
// and the other in VGPRs. A SIMD issues two FP32 instructions per 4-cycle slot only from
// two different waves, so the kernel wants 4 resident waves (<= 128 VGPRs): row 1 in
// SGPRs and, at n = 19..22, the first values of row 2 too (glynn_f32_pair_s2) give 4 waves
// up to n = 22 and 3 at n = 23. 3 static bits with every row in VGPRs need 217 VGPRs
// (2 waves) at n = 20. SR = 2 (row 2 in SGPRs, so the row-1 flips dual-issue) fits 4
// waves at every n and measured the same time at n = 20 and 5% slower at n = 23: at
// n = 20 the launch runs the clock down to 1.9 GHz whichever rows dual-issue.
#ifndef TB_GLYNN_F32_PAIR_U
#define TB_GLYNN_F32_PAIR_U 2
#endif
#ifndef TB_GLYNN_F32_PAIR_SR
#define TB_GLYNN_F32_PAIR_SR 1
#endif
#ifndef TB_GLYNN_F32_PAIR_WPE
#define TB_GLYNN_F32_PAIR_WPE 3
#endif
template <int N, typename F>
constexpr int glynn_u() {
  if (sizeof(F) == 4)
    return (N <= TB_GLYNN_F32_ROWS_MAX_N && N - 9 >= TB_GLYNN_F32_U) ? TB_GLYNN_F32_U : 2;
  return N >= 25 ? TB_GLYNN_U_LARGE : 2;
}
inline int glynn_u_max(int n) {
  const int u32 = (n <= TB_GLYNN_F32_ROWS_MAX_N && n - 9 >= TB_GLYNN_F32_U) ? TB_GLYNN_F32_U : 2;
  return std::max({2, n >= 25 ? TB_GLYNN_U_LARGE : 2, u32});
}

constexpr int kWideMinN = 14;  // below this the SMALL kernel

// Sizes that run the paired walk (FP64: matrices it cannot take walk plainly in the same
// kernel; FP32: in a second one): from where a chunk holds the static block plus one bit up to the
// largest n that fits 256 VGPRs without spills (n = 40 spills).
#ifndef TB_GLYNN_PAIR_MIN_N
#define TB_GLYNN_PAIR_MIN_N 14
#endif
#ifndef TB_GLYNN_PAIR_MAX_N
#define TB_GLYNN_PAIR_MAX_N 39
#endif
template <int N, typename F>
constexpr bool glynn_paired() {
  if constexpr (sizeof(F) == 8) return N >= TB_GLYNN_PAIR_MIN_N && N <= TB_GLYNN_PAIR_MAX_N;
  // FP32 column sums: where the FP32 kernel is in use (larger n, run only to measure its
  // error, keep the plain FP32 walk)
  return N >= TB_GLYNN_PAIR_MIN_N && N <= TB_FP32_COLSUM_MAX_N;
}
// Static super-step bits of the paired walk and its rows in broadcast form (rows 1..B).
// Static super-step bits: 3 at every paired n (a block of 8 pairs between block-start
// flips; 172..256 VGPRs; n = 23 and 24 spill 1 and 10 values, of which the walk reloads one a
// block, and are 1-7% faster than the three launches without spills were). Measured against
// 2 bits below n = 25: 3.7% faster at n = 16 and 3.6-4% at n = 20..24.
template <int N>
constexpr int glynn_pair_u() {
  return 3;
}
template <int N>
constexpr int glynn_pair_b() {
  constexpr int b = (N <= TB_GLYNN_BCAST_WIDE_MAX_N) ? glynn_pair_u<N>() + 2 : glynn_pair_u<N>();
  return b < N - 2 ? b : N - 2;
}
// Lower bound on C of a launch of n: the static bits, and for the paired walk its static
// super-step bits plus the pair bit.
template <int N, typename F>
constexpr int glynn_pair_u_of() {
  return sizeof(F) == 8 ? glynn_pair_u<N>() : TB_GLYNN_F32_PAIR_U;
}
// Values of row 2 the paired FP32 kernel also keeps in SGPRs, so that it fits 4 waves
// per SIMD (<= 128 VGPRs): about 6n + 15 VGPRs without them, 2 fewer per value; up to 11
// values (row 1 takes 2n SGPRs; n = 23 would need 14 and exceed the 102 SGPRs).
#ifndef TB_GLYNN_F32_PAIR_S2_MAX
#define TB_GLYNN_F32_PAIR_S2_MAX 11
#endif
template <int N>
constexpr int glynn_f32_pair_s2() {
  if (TB_GLYNN_F32_PAIR_SR != 1 || TB_GLYNN_F32_PAIR_U < 2) return 0;
  constexpr int over = 6 * N + 15 - 128;
  constexpr int need = over <= 0 ? 0 : (over + 1) / 2 + 1;  // one value of margin
  return (over <= 0 || need > TB_GLYNN_F32_PAIR_S2_MAX) ? 0 : need;
}
// Waves per SIMD the launch is resident at.
template <int N, typename F>
constexpr int glynn_wave_slots() {
  if constexpr (sizeof(F) == 4 && glynn_paired<N, F>()) {
    if constexpr (TB_GLYNN_F32_PAIR_SR == 1)
      return (6 * N + 15 <= 128 || glynn_f32_pair_s2<N>() > 0) ? 4 : TB_GLYNN_F32_PAIR_WPE;
    if constexpr (TB_GLYNN_F32_PAIR_SR == 2) return 4;
    return TB_GLYNN_F32_PAIR_WPE;
  }
  return 2;
}
// Waves per SIMD of the plan's bound on C: the residency, but 3 at n = 22, the one size whose fourth
// wave came with the present register count. With 3 no batch measured is slower than at 3 resident
// waves. With 4 some are 5-20% faster (8, 16, 150, 500 matrices: 67 -> 54, 102 -> 88, 736 -> 685,
// 2255 -> 2152 us) and some 12-23% slower (4, 24, 100: 31 -> 38, 126 -> 145, 493 -> 556), as the
// plan's score takes 2^6 ranks for 2^7.
template <int N, typename F>
constexpr int glynn_plan_slots() {
  return N == 22 ? std::min(glynn_wave_slots<N, F>(), 3) : glynn_wave_slots<N, F>();
}
template <int N, typename F>
constexpr int glynn_min_c() {
  constexpr int u = glynn_u<N, F>();
  if constexpr (glynn_paired<N, F>())
    return u > glynn_pair_u_of<N, F>() + 1 ? u : glynn_pair_u_of<N, F>() + 1;
  return u;
}
constexpr int kMaxC = 12;      // Gray bits per lane chunk
constexpr int kMaxWpmBits = 13;  // waves per matrix before lanes iterate over chunks

struct GlynnPlan {
  int C, wpm, iters;
};

// WIDE plan: chunks of 2^C ranks, one per lane.
//
// Upper bound: the sums drift with the length of a chunk (FP32 sums at n = 20 are off by 5e-6
// with C = 8 and 1.1e-5 with C = 10), so C is at most what gives the batch ~8192 waves, or 7,
// moved by up to two towards fuller rounds of waves: kernels resident at more than 2 waves per
// SIMD (wave_slots) compare it with C - 1 and C - 2, FP64 ones with C + 1 and C + 2 (grow), by
// how full the last round of wave_slots x 1024 waves is, times the share of a chunk left after
// seeding ((n - 2) 2 / (5 2^C) of its instructions). Ties keep the candidate tried first.
//
// Below that bound the plan takes the C with the least ceil(waves / 1024) (2^C + 1.1 n): a
// launch lasts as long as the SIMD with the most waves, and a wave costs its chunk and a fixed
// part (staging the matrix, the quotients, seeding the sums) worth about 1.1 n ranks (0.85 n with
// the FP64 seeds of seed_half_sums, which moves no choice below). One FP64
// wave alone on a SIMD issues 2% slower than two, one FP32 wave at half the rate (dual issue
// takes two). FP64, C = 4, 5, 6, 7, 8 and the rule's choice, with the bound taken before:
//   one matrix of n = 20      15.2   16.5   21.5   33.5   57.1 us    4   (C = 7)
//   16 of n = 20                67     48     39     36     56       7   (C = 7)
//   16 of n = 22               249    178    146    132    125       8   (C = 8)
// and FP32, 16 of n = 22: 178, 129, 100, 94 us, choice 7.
//
// A tuned C (c_pref > 0) replaces the choice. Always: U <= C <= 12 and a matrix gets at least 4
// waves (one workgroup).
constexpr int kPlanSimds = 1024;
inline int glynn_plan_clamp(int C, int nb, int u) {
  return std::min(std::max(std::min(C, kMaxC), u), nb - 8);
}
inline GlynnPlan glynn_plan(int n, int batch, int c_pref, int u = 2, int wave_slots = 2,
                            int grow = 0) {
  GlynnPlan p{};
  const int nb = n - 1;
  const auto waves = [&](int c) { return (double)batch * std::ldexp(1.0, nb - c - 6); };
  int C;
  if (c_pref > 0) {
    C = glynn_plan_clamp(c_pref, nb, u);
  } else {
    int want_bits = 0;  // log2(waves per matrix needed for ~8192 waves in total)
    while (((int64_t)batch << want_bits) < 8192 && want_bits < 30) ++want_bits;
    C = glynn_plan_clamp(std::max(nb - 6 - want_bits, std::min(7, nb - 8)), nb, u);
    const int step = wave_slots > 2 ? -1 : 1, count = wave_slots > 2 ? 3 : 1 + grow;
    double best = -1.0;
    for (int k = 0, c = C, c0 = C; k < count; ++k, c = c0 + k * step) {
      if (glynn_plan_clamp(c, nb, u) != c) continue;
      const double rounds = waves(c) / ((double)kPlanSimds * wave_slots);
      const double seed = (double)(n - 2) * 2.0 / (5.0 * std::ldexp(1.0, c));
      const double score = rounds / std::ceil(rounds) * (1.0 - seed);
      if (score > best + 1e-9) {
        best = score;
        C = c;
      }
    }
    const double alone = grow > 0 ? 1.02 : 2.0;
    double least = INFINITY;
    for (int c = C, low = glynn_plan_clamp(0, nb, u); c >= low; --c) {
      const double cost =
          std::max(std::ceil(waves(c) / kPlanSimds), alone) * (std::ldexp(1.0, c) + 1.1 * n);
      if (cost < least) {
        least = cost;
        C = c;
      }
    }
  }
  p.C = C;
  const int wave_bits = nb - p.C - 6;  // log2(waves needed at one chunk per lane), >= 2
  const int wpm_bits = std::min(wave_bits, kMaxWpmBits);
  p.wpm = 1 << wpm_bits;
  p.iters = 1 << (wave_bits - wpm_bits);
  return p;
}

// SMALL plan: the longest chunk (less seeding) that still gives the launch a wave per SIMD (2
// or 4 measured up to 10% slower, 12 and 13 columns, 1000 to 4000 matrices), at least U bits,
// at most 256 lanes per matrix and 48 KiB of matrices per workgroup; 16 lanes or more where the
// rows are in broadcast form.
#ifndef TB_SMALL_WAVES
#define TB_SMALL_WAVES 1024
#endif
inline size_t glynn_small_lds(int n, int C, size_t elem) {
  return (size_t)(256 >> (n - 1 - C)) * (n * n + 1) * elem;
}
inline int glynn_small_plan(int n, int batch, int c_pref, int u, size_t elem) {
  const int nb = n - 1;
  const int lo = std::max(u, nb - 8);
  int hi = elem == sizeof(tb::cpx<double>) && n >= tb::kSmallBcastMinN ? nb - 4 : nb;
  while (hi > lo && glynn_small_lds(n, hi, elem) > 48 * 1024) --hi;
  if (c_pref > 0) return std::min(std::max(c_pref, lo), hi);
  int C = hi;
  while (C > lo && ((int64_t)batch << (nb - C)) < TB_SMALL_WAVES * 64) --C;
  return C;
}

// wpm_cap: partials per matrix the workspace holds; a plan that needs more fails with
// TB_EWORKSPACE instead of writing past them.
template <int N, typename F>
inline int32_t launch_glynn_n(const tb::cd *A, int64_t mstride, int batch, tb::cd *out,
                              tb::cd *partial, int *handled, int wpm_cap, int c_pref,
                              hipStream_t s) {
  if constexpr (N < kWideMinN) {
    constexpr int U = (N - 1) < 2 ? (N - 1) : 2;
    const int C = glynn_small_plan(N, batch, c_pref, U, sizeof(tb::cpx<F>));
    const int mats = 256 >> (N - 1 - C);
    hipLaunchKernelGGL((tb::glynn_small_kernel<N, U, F>), dim3((batch + mats - 1) / mats), dim3(256),
                       glynn_small_lds(N, C, sizeof(tb::cpx<F>)), s, A, mstride, batch, C, out);
    (void)partial;
    (void)handled;
    (void)wpm_cap;
    return tbh::check_hip(hipGetLastError(), "glynn_small_kernel");
  } else {
    constexpr int U = glynn_u<N, F>(), R0 = glynn_reg_rows<N, F>();
    constexpr int CMIN = glynn_min_c<N, F>();
    constexpr bool paired = glynn_paired<N, F>(), fp32 = sizeof(F) == 4;
    static_assert(CMIN <= N - 9, "the static block must fit the smallest chunk (C <= n - 9)");
    const GlynnPlan p = glynn_plan(N, batch, c_pref, CMIN, glynn_plan_slots<N, F>(), fp32 ? 0 : 2);
    if (p.wpm > wpm_cap)
      return tbh::fail(TB_EWORKSPACE,
                       "glynn: the plan for n=%d batch=%d needs %d partials per matrix, the "
                       "workspace holds %d", N, batch, p.wpm, wpm_cap);
    const dim3 blocks((unsigned)batch * (unsigned)(p.wpm / 4));
    if constexpr (paired && fp32) {
      hipLaunchKernelGGL((tb::glynn_pair_kernel_f32<N, TB_GLYNN_F32_PAIR_U, TB_GLYNN_F32_PAIR_SR,
                                                    glynn_f32_pair_s2<N>(), glynn_wave_slots<N, F>()>),
                         blocks, dim3(256), 0, s, A, mstride, p.C, p.wpm, p.iters, partial, handled,
                         out);
      if (const int32_t rc = tbh::check_hip(hipGetLastError(), "glynn_pair_kernel_f32")) return rc;
    }
    if constexpr (paired && !fp32)
      hipLaunchKernelGGL((tb::glynn_pair_kernel<N, glynn_pair_u<N>(), glynn_pair_b<N>(), U, R0>),
                         blocks, dim3(256), 0, s, A, mstride, p.C, p.wpm, p.iters, partial, out);
    else
      hipLaunchKernelGGL((tb::glynn_wide_kernel<N, U, R0, F>), blocks, dim3(256), 0, s, A, mstride,
                         p.C, p.wpm, p.iters, partial, paired ? handled : nullptr, out);
    const int32_t rc = tbh::check_hip(hipGetLastError(), "glynn walk");
    if (rc || p.wpm == 4) return rc;
    hipLaunchKernelGGL(tb::glynn_finish_kernel, dim3((batch + 3) / 4), dim3(256), 0, s, partial,
                       p.wpm, batch, out);
    return tbh::check_hip(hipGetLastError(), "glynn_finish_kernel");
  }
}

template <typename F, int N = 2>
inline int32_t dispatch_glynn(int n, const tb::cd *A, int64_t mstride, int batch, tb::cd *out,
                              tb::cd *partial, int *handled, int wpm_cap, int c_pref,
                              hipStream_t s) {
  if constexpr (N > TB_GLYNN_MAX_N) {
    return tbh::fail(TB_ERANGE, "glynn: n=%d exceeds TB_GLYNN_MAX_N=%d", n, TB_GLYNN_MAX_N);
  } else {
    if (n == N)
      return launch_glynn_n<N, F>(A, mstride, batch, out, partial, handled, wpm_cap, c_pref, s);
    return dispatch_glynn<F, N + 1>(n, A, mstride, batch, out, partial, handled, wpm_cap, c_pref, s);
  }
}

// `handled`: batch ints of workspace for the paired FP32 walk; `wpm_cap`: partials per matrix
// after them. Both take the FP64 matrices.
int32_t glynn_dispatch_f64(int n, const tb::cd *A, int64_t mstride, int batch, tb::cd *out,
                           tb::cd *partial, int *handled, int wpm_cap, int c_pref, hipStream_t s);
int32_t glynn_dispatch_f32(int n, const tb::cd *A, int64_t mstride, int batch, tb::cd *out,
                           tb::cd *partial, int *handled, int wpm_cap, int c_pref, hipStream_t s);

}  // namespace tbgl
