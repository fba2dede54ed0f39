#pragma once
// Gray-walk building blocks shared by the Glynn, sweep and gradient kernels: complex values
// of either precision, balanced product trees, and the flip of one matrix row into the
// half column sums (from LDS/global rows, VGPR rows, SGPR-held values or broadcast-form
// VGPR vectors).
#include "tb_common.hpp"

namespace tb {

// Keeps the scheduler from hoisting the next Gray step's row reads above the current
// step (which otherwise multiplies live registers by the unroll factor and spills).
#ifndef TB_STEP_FENCE
#define TB_STEP_FENCE() __builtin_amdgcn_sched_barrier(0)
#endif

template <typename F>
struct cpx {
  F re, im;
};

template <typename F>
__device__ __forceinline__ cpx<F> cmulT(cpx<F> a, cpx<F> b) {
  cpx<F> r;
  r.re = fma(a.re, b.re, -(a.im * b.im));
  r.im = fma(a.re, b.im, a.im * b.re);
  return r;
}

template <typename F, int LO, int HI>
struct TreeProdT {
  static __device__ __forceinline__ cpx<F> run(const F *re, const F *im) {
    constexpr int MID = (LO + HI) / 2;
    return cmulT<F>(TreeProdT<F, LO, MID>::run(re, im), TreeProdT<F, MID, HI>::run(re, im));
  }
};
template <typename F, int LO>
struct TreeProdT<F, LO, LO + 1> {
  static __device__ __forceinline__ cpx<F> run(const F *re, const F *im) { return {re[LO], im[LO]}; }
};

// h += row (add) or h -= row; `row` is an LDS row shared by the lanes of a matrix (broadcast
// reads). The row is consumed in groups of G complex values
// with the reads of group g+1 issued before the adds of group g, and a scheduling
// barrier per group, so at most 2*G loaded values are live at once.
#ifndef TB_FLIP_GROUP
#define TB_FLIP_GROUP 4
#endif

// MODE 1: h += row, MODE -1: h -= row, MODE 0: h += sg * row (runtime direction, one
// FMA per component with sg = +-1 held per lane).
// Columns J0..N-1 only (J0 > 0 when the first J0 values of the row are held in SGPRs).
template <int N, int MODE, typename F, typename P, int J0 = 0, int G = TB_FLIP_GROUP>
__device__ __forceinline__ void flip_mem(F (&hr)[N], F (&hi)[N], P row, F sg) {
  constexpr int NG = (N - J0 + G - 1) / G;
  cpx<F> cur[G], nxt[G];
#pragma unroll
  for (int e = 0; e < G; ++e)
    if (J0 + e < N) cur[e] = row[J0 + e];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g + 1 < NG) {
#pragma unroll
      for (int e = 0; e < G; ++e)
        if (J0 + (g + 1) * G + e < N) nxt[e] = row[J0 + (g + 1) * G + e];
    }
#pragma unroll
    for (int e = 0; e < G; ++e) {
      const int j = J0 + g * G + e;
      if (j < N) {
        if constexpr (MODE == 1) {
          hr[j] += cur[e].re;
          hi[j] += cur[e].im;
        } else if constexpr (MODE == -1) {
          hr[j] -= cur[e].re;
          hi[j] -= cur[e].im;
        } else {
          hr[j] = fma(sg, cur[e].re, hr[j]);
          hi[j] = fma(sg, cur[e].im, hi[j]);
        }
      }
    }
    TB_STEP_FENCE();
#pragma unroll
    for (int e = 0; e < G; ++e) cur[e] = nxt[e];
  }
}

template <int N, int MODE, typename F>
__device__ __forceinline__ void flip_reg(F (&hr)[N], F (&hi)[N], const F (&rr)[N], const F (&ri)[N],
                                         F sg) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if constexpr (MODE == 1) {
      hr[j] += rr[j];
      hi[j] += ri[j];
    } else if constexpr (MODE == -1) {
      hr[j] -= rr[j];
      hi[j] -= ri[j];
    } else {
      hr[j] = fma(sg, rr[j], hr[j]);
      hi[j] = fma(sg, ri[j], hi[j]);
    }
  }
}

// The first S values of row 0 held in SGPRs (wave-uniform): a flip of row 0 reads them
// as scalar operands and only the rest from LDS, which unloads the LDS return path.
template <int S, typename F>
struct SRow {
  F re[S > 0 ? S : 1], im[S > 0 ? S : 1];
};

__device__ __forceinline__ double uniform_value(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float uniform_value(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// Flip of row 0: its first S values from SGPRs, the rest from `row`.
template <int N, int S, int MODE, typename F, typename P>
__device__ __forceinline__ void flip_srow(F (&hr)[N], F (&hi)[N], const SRow<S, F> &sr, P row,
                                          F sg) {
#pragma unroll
  for (int j = 0; j < S; ++j) {
    if constexpr (MODE == 1) {
      hr[j] += sr.re[j];
      hi[j] += sr.im[j];
    } else if constexpr (MODE == -1) {
      hr[j] -= sr.re[j];
      hi[j] -= sr.im[j];
    } else {
      hr[j] = fma(sg, sr.re[j], hr[j]);
      hi[j] = fma(sg, sr.im[j], hi[j]);
    }
  }
  flip_mem<N, MODE, F, P, S>(hr, hi, row, sg);
}

// Load the first S values of a wave-uniform row into SGPRs.
template <int S, typename F, typename P>
__device__ __forceinline__ void load_srow(SRow<S, F> &sr, P row) {
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const cpx<F> v = row[j];
    sr.re[j] = uniform_value(v.re);
    sr.im[j] = uniform_value(v.im);
  }
}

// A row (or column) of N complex values in broadcast form: value t (re/im interleaved)
// sits in lane t mod 16 of every 16-lane row of VGPR pair t / 16, i.e. 2 ceil(2N/16) VGPRs
// per vector. A flip adds it to the half sums with one v_fmac_f64 per value whose first
// operand is taken from that lane by DPP row_newbcast, with no LDS read. Every lane of
// the wave must be active at a flip (DPP reads other lanes' registers).
template <int N>
struct Bcast {
  static constexpr int P = (2 * N + 15) / 16;
  double v[P];
};

// Lane `lane` of the wave loads its slots of the vector `src` (N complex values).
template <int N>
__device__ __forceinline__ void load_bcast(Bcast<N> &b, const double *src, int lane) {
#pragma unroll
  for (int p = 0; p < Bcast<N>::P; ++p) {
    const int t = 16 * p + (lane & 15);
    b.v[p] = t < 2 * N ? src[t] : 0.0;
  }
}

// h += s * v[L] (L = lane within each 16-lane row), and the same with -v[L].
template <int L>
__device__ __forceinline__ void fmac_bcast(double &h, double v, double s) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(h)
      : "v"(v), "v"(s), "i"(L));
}
template <int L>
__device__ __forceinline__ void fmac_bcast_neg(double &h, double v, double s) {
  asm("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
      : "+v"(h)
      : "v"(v), "v"(s), "i"(L));
}

// h += sg * vector (MODE 0), h += vector (MODE 1, s = 1) or h -= vector (MODE -1, s = 1).
template <int T, int N, int MODE>
__device__ __forceinline__ void flip_bcast(double (&hr)[N], double (&hi)[N], const Bcast<N> &b,
                                           double s) {
  if constexpr (T < 2 * N) {
    double &h = (T & 1) ? hi[T / 2] : hr[T / 2];
    if constexpr (MODE == -1)
      fmac_bcast_neg<T % 16>(h, b.v[T / 16], s);
    else
      fmac_bcast<T % 16>(h, b.v[T / 16], s);
    flip_bcast<T + 1, N, MODE>(hr, hi, b, s);
  }
}

// ------------------------------------------------------------------------------------
// Paired walks. Two Gray codes that differ only in one row (particle) r have column sums
// c_j (u_j + 1) and c_j (u_j - 1) once every other row is divided by row r
// (u_j = sum_{i != r} delta_i M[i][j] / M[r][j]), so one update of u serves both codes
// and each factor (u_j +- 1) enters a running product x as x u_j +- x: four FMAs with
// the +-1 folded into their addends.
// ------------------------------------------------------------------------------------

// prod_{j in [LO, HI)} (u_j + PM), PM = +-1: the first factor formed by one add, each
// further one folded into x u_j + PM x.
template <int PM, int LO, int HI, int N>
__device__ __forceinline__ cd fold_chain(const double (&ur)[N], const double (&ui)[N]) {
  double xr = ur[LO] + (double)PM, xi = ui[LO];
#pragma unroll
  for (int j = LO + 1; j < HI; ++j) {
    const double nr = fma(-xi, ui[j], fma(xr, ur[j], (double)PM * xr));
    const double ni = fma(xi, ur[j], fma(xr, ui[j], (double)PM * xi));
    xr = nr;
    xi = ni;
  }
  return {xr, xi};
}

// X += SIGN prod(u + 1), Y += SIGN prod(u - 1); each product is two chains of N/2
// factors joined by a multiply fused into the accumulation.
template <int SIGN, int N>
__device__ __forceinline__ void pair_acc2(double &xr, double &xi, double &yr, double &yi,
                                          const double (&ur)[N], const double (&ui)[N]) {
  constexpr int H = N / 2;
  cmul_acc<SIGN>(xr, xi, fold_chain<1, 0, H>(ur, ui), fold_chain<1, H, N>(ur, ui));
  cmul_acc<SIGN>(yr, yi, fold_chain<-1, 0, H>(ur, ui), fold_chain<-1, H, N>(ur, ui));
}

// A pair row must have every entry above 2^-16 of the matrix's largest entry (squared
// magnitudes compared): far from zero, its quotients stay in range and well rounded.
constexpr double kPairMinRel2 = 0x1p-32;

// ------------------------------------------------------------------------------------
// Sums of several values over 2^LB lanes (LB = 4: each row of 16 lanes; 5: the rows 0, 1 and
// 2, 3; 6: the wave), transposed: every stage halves the number of values a lane carries, so
// CNT sums cost about CNT additions and swaps in all instead of CNT LB shuffles, and use no
// LDS (permlane swaps for lane distances 32 and 16, DPP inside a row).
// ------------------------------------------------------------------------------------
__device__ __forceinline__ double select_f64(bool c, double a, double b) { return c ? a : b; }

template <int CTRL>
__device__ __forceinline__ double dpp_perm(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
  return join64(lo, hi);
}

// (a, b) -> lanes < 32: a + a[lane ^ 32]; lanes >= 32: b + b[lane ^ 32].
__device__ __forceinline__ double swap32_pair_sum(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)ua, (uint32_t)ub, false, false);
  const auto hi =
      __builtin_amdgcn_permlane32_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
  return join64(lo[0], hi[0]) + join64(lo[1], hi[1]);
}
// (a, b) -> rows 0, 2: a + a[lane ^ 16]; rows 1, 3: b + b[lane ^ 16].
__device__ __forceinline__ double swap16_pair_sum(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)ua, (uint32_t)ub, false, false);
  const auto hi =
      __builtin_amdgcn_permlane16_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
  return join64(lo[0], hi[0]) + join64(lo[1], hi[1]);
}
// (a, b) -> lanes with `odd` clear: a + a[partner], set: b + b[partner].
template <int CTRL>
__device__ __forceinline__ double dpp_pair_sum(double a, double b, bool odd) {
  const double keep = select_f64(odd, b, a), send = select_f64(odd, a, b);
  return keep + dpp_perm<CTRL>(send);
}
// Halves `x` (CNT values) by one stage.
template <int CTRL, int CNT>
__device__ __forceinline__ void dpp_stage(double *x, bool odd) {
#pragma unroll
  for (int k = 0; k < CNT / 2; ++k) x[k] = dpp_pair_sum<CTRL>(x[2 * k], x[2 * k + 1], odd);
  if (CNT & 1) x[CNT / 2] = x[CNT - 1] + dpp_perm<CTRL>(x[CNT - 1]);
}

// Ends with ceil(CNT / 2^LB) values in x: value v of a lane is the total of input
// lane_sums_index(lane) + v 2^LB (meaningless where that is CNT or more).
template <int LB, int CNT>
__device__ __forceinline__ void lane_sums(double *x, int lane) {
  constexpr int H32 = LB == 6 ? (CNT + 1) / 2 : CNT, H16 = LB >= 5 ? (H32 + 1) / 2 : H32;
  if constexpr (LB == 6) {
#pragma unroll
    for (int k = 0; k < CNT / 2; ++k) x[k] = swap32_pair_sum(x[2 * k], x[2 * k + 1]);
    if (CNT & 1) x[CNT / 2] = swap32_pair_sum(x[CNT - 1], x[CNT - 1]);
  }
  if constexpr (LB >= 5) {
#pragma unroll
    for (int k = 0; k < H32 / 2; ++k) x[k] = swap16_pair_sum(x[2 * k], x[2 * k + 1]);
    if (H32 & 1) x[H32 / 2] = swap16_pair_sum(x[H32 - 1], x[H32 - 1]);
  }
  constexpr int H8 = (H16 + 1) / 2, H4 = (H8 + 1) / 2, H2 = (H4 + 1) / 2;
  dpp_stage<0x128, H16>(x, (lane & 8) != 0);  // row_ror:8
  dpp_stage<0x141, H8>(x, (lane & 4) != 0);   // row_half_mirror
  dpp_stage<0x4E, H4>(x, (lane & 2) != 0);    // quad_perm [2,3,0,1]
  dpp_stage<0xB1, H2>(x, (lane & 1) != 0);    // quad_perm [1,0,3,2]
}
template <int LB>
__device__ __forceinline__ int lane_sums_index(int lane) {
  const int a = ((lane & 1) << 3) | ((lane & 2) << 1) | ((lane & 4) >> 1) | ((lane & 8) >> 3);
  const int b = 2 * a + ((lane >> 4) & 1);
  return LB == 4 ? a : LB == 5 ? b : 2 * b + ((lane >> 5) & 1);
}

// 1.0 in a VGPR the compiler cannot fold away (second operand of fixed-direction flips).
__device__ __forceinline__ double vgpr_one() {
  double one = 1.0;
  asm volatile("" : "+v"(one));
  return one;
}

// Two wait states between whatever wrote a broadcast-form row's registers and its DPP reads.
template <int N>
__device__ __forceinline__ void bcast_settle(Bcast<N> &b) {
#pragma unroll
  for (int p = 0; p < Bcast<N>::P; ++p) asm volatile("s_nop 1" : "+v"(b.v[p]));
}

// The half sums at the start of a chunk of 2^c ranks, h = (fixed + sum_b d_b row_b) / 2 with
// d_b = -1 where bit b of g0 is set, row b at rows + 2 N b, for lanes on consecutive chunks:
// only bits c - 1 .. c + 5 differ between the lanes of a wave. The rows of the other bits are
// added up once per wave, each lane keeping the components it holds in broadcast form, and the
// sum and the seven others enter every lane's sums from there by DPP: at n = 20, 16 N FMAs and
// 3 reads per row instead of 2 N FMAs and N 16-byte reads for each of 19 rows. That took the
// fixed cost of a wave of the k = 20 sweep from about 38 codes to 20 (one item 28.7 -> 18.8 us,
// 16 items 67 -> 47), of a Glynn wave at n = 20 from 22 to 17 (20 matrices 53 -> 48 us). Reading
// the seven rows ahead of their use gains nothing more, and FP32 sums, which issue two FMAs in
// the time of one of these, are 1-20% slower this way.
template <int N>
__device__ __forceinline__ void seed_half_sums(double (&hr)[N], double (&hi)[N], const double *fixed,
                                               const double *rows, int bits, int c, uint64_t g0) {
  constexpr int P = Bcast<N>::P;
  int lane = threadIdx.x;
  asm volatile("" : "+v"(lane));  // the slots are worked out here, not kept from chunk to chunk
  const uint64_t g = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)g0) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(g0 >> 32)) << 32;
  int at[P];
#pragma unroll
  for (int p = 0; p < P; ++p) at[p] = min(16 * p + (lane & 15), 2 * N - 1);
  Bcast<N> sum;
#pragma unroll
  for (int p = 0; p < P; ++p) sum.v[p] = 0.5 * fixed[at[p]];
  const int lo = max(c - 1, 0), end = min(c + 6, bits);
  const auto add = [&](int b) {
    const double d = ((g >> b) & 1ull) ? -0.5 : 0.5;
#pragma unroll
    for (int p = 0; p < P; ++p) sum.v[p] = fma(d, rows[2 * N * b + at[p]], sum.v[p]);
  };
#pragma unroll 2
  for (int b = 0; b < lo; ++b) add(b);
#pragma unroll 2
  for (int b = end; b < bits; ++b) add(b);
#pragma unroll
  for (int j = 0; j < N; ++j) hr[j] = hi[j] = 0.0;
  bcast_settle(sum);
  flip_bcast<0, N, 1>(hr, hi, sum, vgpr_one());
#pragma unroll 1
  for (int b = lo; b < end; ++b) {
    Bcast<N> row;
#pragma unroll
    for (int p = 0; p < P; ++p) row.v[p] = rows[2 * N * b + at[p]];
    bcast_settle(row);
    flip_bcast<0, N, 0>(hr, hi, row, ((g0 >> b) & 1ull) ? -0.5 : 0.5);
  }
}

// Largest of one value per lane, in every lane.
__device__ __forceinline__ double wave_allmax(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const auto l32 = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto h32 = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  v = fmax(join64(l32[0], h32[0]), join64(l32[1], h32[1]));
  const uint64_t t = __builtin_bit_cast(uint64_t, v);
  const auto l16 = __builtin_amdgcn_permlane16_swap((uint32_t)t, (uint32_t)t, false, false);
  const auto h16 = __builtin_amdgcn_permlane16_swap((uint32_t)(t >> 32), (uint32_t)(t >> 32), false, false);
  v = fmax(join64(l16[0], h16[0]), join64(l16[1], h16[1]));
  v = fmax(v, dpp_perm<0x128>(v));
  v = fmax(v, dpp_perm<0x124>(v));
  v = fmax(v, dpp_perm<0x122>(v));
  return fmax(v, dpp_perm<0x121>(v));
}

// Both halves' value of a lane pair at distance 32: {low lane's, high lane's}, in both.
__device__ __forceinline__ void both32(double v, double &lo, double &hi) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const auto a = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  lo = join64(a[0], b[0]);
  hi = join64(a[1], b[1]);
}

// Product of one complex value per lane over the wave (wave-uniform).
__device__ __forceinline__ cd wave_prod(cd v) {
  cd a, b;
  both32(v.re, a.re, b.re);
  both32(v.im, a.im, b.im);
  v = cmul(a, b);
  v = cmul(v, {__shfl_xor(v.re, 16, 64), __shfl_xor(v.im, 16, 64)});
  v = cmul(v, {dpp_perm<0x128>(v.re), dpp_perm<0x128>(v.im)});
  v = cmul(v, {dpp_perm<0x124>(v.re), dpp_perm<0x124>(v.im)});
  v = cmul(v, {dpp_perm<0x122>(v.re), dpp_perm<0x122>(v.im)});
  v = cmul(v, {dpp_perm<0x121>(v.re), dpp_perm<0x121>(v.im)});
  return {uniform_value(v.re), uniform_value(v.im)};
}

}  // namespace tb
