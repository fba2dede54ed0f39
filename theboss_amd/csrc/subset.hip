// All pairs of output rows t and input rows s by the subset recurrence: with t_l the l-th
// output particle and k particles on both sides,
//   perm(U[t_1..t_l, s]) = sum_d s_d U[t_l][d] perm(U[t_1..t_{l-1}, s - e_d])
// (expansion along the last row; s_d the multiplicity of mode d). Every input row of a call
// is a point of the lattice of occupations below their entrywise maximum, so one pass over the
// lattice's levels 1..k yields every pair of an output row: GCC-A's layers (all k-particle
// substates of one input) and the exact distributions (all lossy inputs of one state).
//
// Replaces, for those calls, one walk of prod (s_d + 1) Guan codes per pair (the permanent
// loop of generalized_cliffords_simulation_strategy.py:162-171 over :224-247 calls
// compute_permanent per pair). For n input modes of one particle each the lattice costs
// sum_{l <= k} l C(n, l) complex multiply-adds per output row, against C(n, k) 2^k codes of k
// multiplies: n = 10, k = 5: 2560 against 40,000. No term cancels another by construction, so the
// result is at least as accurate as the alternating sums.
//
// What bounds it: latency (GCC-A layer of 200 prefixes x 20 outputs x C(10, 5) inputs, 1.0M
// pairs: 42 us, 4 of them the 16 MB written; the walk 351). A workgroup first builds the lattice from the input rows (in LDS, for
// itself: a plan kernel with predecessor lists in global memory took 20 us more per call),
// then a wave per output row walks the levels (the whole workgroup where the levels are wide
// or the rows few). The Guan walk follows in stream order over the rows whose done flag is 0:
// all of them when the lattice is too large, or a row whose particle number differs.
#include <algorithm>

#include "tb_common.hpp"

namespace tb {

constexpr int kSubModes = 12;      // modes of the lattice
constexpr int kSubCodes = 4096;    // points of the lattice
constexpr int kSubK = 12;          // particles
constexpr int kSubMaxLdu = 1024;   // mode indices the plan can hold
constexpr int kSubMaxIn = 2048;    // input rows
constexpr int kSubEntries = 2048;  // complex values of two adjacent levels in LDS
constexpr int kSubWaveEntries = kSubEntries / 4;  // ... when a wave works alone
// Output rows from which on a wave each is better than a workgroup each.
constexpr int kSubWaveRows = 2048;

struct SubsetPlan {
  int ok, k, D, width, multi, total;
  int modes[kSubModes], radix[kSubModes], stride[kSubModes];
  int cnt[kSubK + 1], off[kSubK + 1];
};

struct SubsetLds {
  union {
    cd F[kSubEntries];    // two levels of up to 4 output rows
    int top[kSubMaxLdu];  // while planning, per mode: largest multiplicity, then its index
  };
  cd Ul[4][kSubK * kSubModes];  // U[t_l][mode d] of a wave's output row
  unsigned short order[kSubCodes], pos[kSubCodes];  // points by level; place in its level
  unsigned short in_pos[kSubMaxIn];
  int rl[4][kSubK];
  int binom[kSubModes + 1][kSubModes + 1];
  int bad;
  SubsetPlan p;
};

// Fills S.p, S.order, S.pos and S.in_pos; S.p.ok = 0 when the rows have no small lattice.
__device__ __forceinline__ void subset_plan(SubsetLds &S, const int *__restrict__ in_modes,
                                            const int *__restrict__ in_mult, int in_max, int n_in,
                                            int ldu) {
  const int tid = threadIdx.x;
  SubsetPlan &p = S.p;
  for (int e = tid; e < ldu; e += 256) S.top[e] = 0;
  if (tid < (kSubModes + 1) * (kSubModes + 1)) {
    const int n = tid / (kSubModes + 1), r = tid % (kSubModes + 1);
    int c = r > n ? 0 : 1;
    for (int i = 1; i <= r && r <= n; ++i) c = c * (n - r + i) / i;
    S.binom[n][r] = c;
  }
  if (tid <= kSubK) p.cnt[tid] = 0;
  if (tid == 0) S.bad = 0;
  // multiplicities above kSubK are refused below, so capped sums cannot wrap
  int k = 0;
  for (int q = 0; q < in_max; ++q) k += min(max(in_mult[q], 0), kSubK + 1);
  __syncthreads();
  for (int i = tid; i < n_in; i += 256) {
    const int *sm = in_modes + (size_t)i * in_max, *su = in_mult + (size_t)i * in_max;
    int sum = 0;
    bool refuse = false;
    for (int q = 0; q < in_max; ++q) {
      const int m = su[q], d = sm[q];
      if (m <= 0) continue;
      sum += min(m, kSubK + 1);
      if (d < 0 || d >= ldu || m > kSubK) {
        refuse = true;
        continue;
      }
      int all = m;  // a mode may fill several slots
      for (int r = 0; r < q; ++r)
        if (su[r] > 0 && sm[r] == d) all += min(su[r], kSubK + 1);
      atomicMax(&S.top[d], all);
    }
    if (refuse || sum != k) S.bad = 1;
  }
  __syncthreads();
  if (tid < 64) {  // the occupied modes, in mode order
    int D = 0;
    for (int e0 = 0; e0 < ldu; e0 += 64) {
      const int v = e0 + tid < ldu ? S.top[e0 + tid] : 0;
      const uint64_t bal = __ballot(v > 0);
      const int at = D + __popcll(bal & ((1ull << tid) - 1ull));
      if (v > 0 && at < kSubModes) {
        p.modes[at] = e0 + tid;
        p.radix[at] = v + 1;
      }
      D += __popcll(bal);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (tid == 0) {
      bool ok = !S.bad && D <= kSubModes && k <= kSubK;
      int points = 1, multi = 0;
      for (int d = 0; ok && d < D; ++d) {
        p.stride[d] = points;
        points *= p.radix[d];  // at most 4096 * 13: no overflow
        multi |= p.radix[d] > 2;
        ok = points <= kSubCodes;
      }
      p.ok = ok ? 1 : 0;
      p.k = k;
      p.D = D;
      p.multi = multi;
      p.total = points;
    }
  }
  __syncthreads();
  if (!p.ok) return;
  if (tid < p.D) S.top[p.modes[tid]] = tid;
  __syncthreads();
  for (int i = tid; i < n_in; i += 256) {
    const int *sm = in_modes + (size_t)i * in_max, *su = in_mult + (size_t)i * in_max;
    int code = 0;
    for (int q = 0; q < in_max; ++q)
      if (su[q] > 0) code += su[q] * p.stride[S.top[sm[q]]];
    S.in_pos[i] = (unsigned short)code;
  }
  if (p.multi) {
    for (int c = tid; c < p.total; c += 256) {
      int l = 0;
      for (int d = 0; d < p.D; ++d) l += (c / p.stride[d]) % p.radix[d];
      if (l <= p.k) S.pos[c] = (unsigned short)atomicAdd(&p.cnt[l], 1);
    }
  } else {  // one particle per mode: the rank among the subsets of the same size
    if (tid <= min(p.k, p.D)) p.cnt[tid] = S.binom[p.D][tid];
    for (int c = tid; c < p.total; c += 256) {
      int r = 0, i = 1;
      for (int m = c; m; m &= m - 1, ++i) r += S.binom[__ffs(m) - 1][i];
      S.pos[c] = (unsigned short)r;
    }
  }
  __syncthreads();
  if (tid == 0) {
    int at = 0, width = 1;
    for (int l = 0; l <= p.k; ++l) {
      p.off[l] = at;
      at += p.cnt[l];
      width = max(width, p.cnt[l]);
    }
    p.width = width;
    if (2 * width > kSubEntries) p.ok = 0;
  }
  __syncthreads();
  if (!p.ok) return;
  for (int c = tid; c < p.total; c += 256) {
    int l = __popc(c);
    if (p.multi) {
      l = 0;
      for (int d = 0; d < p.D; ++d) l += (c / p.stride[d]) % p.radix[d];
    }
    if (l <= p.k) S.order[p.off[l] + S.pos[c]] = (unsigned short)c;
  }
  for (int i = tid; i < n_in; i += 256) S.in_pos[i] = S.pos[S.in_pos[i]];
  __syncthreads();
}

__device__ __forceinline__ void cfma(double &re, double &im, cd a, cd b) {
  re = fma(a.re, b.re, re);
  re = fma(-a.im, b.im, re);
  im = fma(a.re, b.im, im);
  im = fma(a.im, b.re, im);
}

// Level l from level l - 1 by the T threads of a group (t inside it).
template <int T, bool MULTI>
__device__ __forceinline__ void subset_level(const SubsetLds &S, const cd *src, cd *dst, const cd *u,
                                             int l, int t) {
  const SubsetPlan &p = S.p;
  const int cnt = p.cnt[l];
  const unsigned short *order = S.order + p.off[l];
  for (int i = t; i < cnt; i += T) {
    const int c = order[i];
    double re = 0.0, im = 0.0;
    if constexpr (MULTI) {
      for (int d = 0; d < p.D; ++d) {
        const int st = p.stride[d];
        const int s = (c / st) % p.radix[d];
        if (s == 0) continue;
        const cd w = u[d];
        cfma(re, im, {(double)s * w.re, (double)s * w.im}, src[S.pos[c - st]]);
      }
    } else {
      int m = c;
#pragma unroll 4
      for (int j = 0; j < l; ++j) {  // every point of level l has l bits
        const int bit = m & -m;
        m ^= bit;
        cfma(re, im, u[__ffs(bit) - 1], src[S.pos[c ^ bit]]);
      }
    }
    dst[i] = {re, im};
  }
}

// Output row j by the T threads of a group; F holds two levels of p.width values.
template <int T>
__device__ __forceinline__ void subset_row(SubsetLds &S, const cd *__restrict__ U, int ldu,
                                           const int *__restrict__ out_modes,
                                           const int *__restrict__ out_mult, int out_max, int j,
                                           int n_in, cd *F, cd *Ul, int *rl, int *__restrict__ done,
                                           cd *__restrict__ out) {
  const SubsetPlan &p = S.p;
  const int lane = threadIdx.x & 63, t = T == 64 ? lane : (int)threadIdx.x;
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto sync = [&] {
    if constexpr (T == 64)
      wave_sync();
    else
      __syncthreads();
  };
  // The row's particles, one after the other: a lane per slot (out_max <= 64).
  int m = 0, md = 0;
  if (lane < out_max) {
    m = max(out_mult[(size_t)j * out_max + lane], 0);
    md = out_modes[(size_t)j * out_max + lane];
  }
  int incl = m;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, 64);
    if (lane >= off) incl += v;
  }
  // the same in every wave of the group (slots above p.k could wrap the sum)
  const bool mine = !__any(m > p.k) && __shfl(incl, 63, 64) == p.k;
  if (t == 0) done[j] = mine ? 1 : 0;
  if (!mine) return;
  for (int e = incl - m; e < incl; ++e) rl[e] = md;
  wave_sync();
  for (int e = lane; e < p.k * p.D; e += 64) {
    const int l = e / p.D, d = e - l * p.D;
    Ul[e] = U[(size_t)rl[l] * ldu + p.modes[d]];
  }
  if (t == 0) F[0] = {1.0, 0.0};
  sync();
  for (int l = 1; l <= p.k; ++l) {
    const cd *src = F + ((l & 1) ? 0 : p.width);
    cd *dst = F + ((l & 1) ? p.width : 0);
    if (p.multi)
      subset_level<T, true>(S, src, dst, Ul + (l - 1) * p.D, l, t);
    else
      subset_level<T, false>(S, src, dst, Ul + (l - 1) * p.D, l, t);
    sync();
  }
  const cd *last = F + ((p.k & 1) ? p.width : 0);
  for (int i = t; i < n_in; i += T) out[(size_t)j * n_in + i] = last[S.in_pos[i]];
  sync();
}

__global__ __launch_bounds__(256) void subset_rows_kernel(
    const int *__restrict__ in_modes, const int *__restrict__ in_mult, int in_max, int n_in,
    const cd *__restrict__ U, int ldu, const int *__restrict__ out_modes,
    const int *__restrict__ out_mult, int out_max, int n_out, int *__restrict__ done,
    cd *__restrict__ out) {
  __shared__ SubsetLds S;
  subset_plan(S, in_modes, in_mult, in_max, n_in, ldu);
  const int wave = threadIdx.x >> 6;
  if (!S.p.ok) {
    for (int j = blockIdx.x * 256 + threadIdx.x; j < n_out; j += gridDim.x * 256) done[j] = 0;
    return;
  }
  if (n_out >= kSubWaveRows && 2 * S.p.width <= kSubWaveEntries) {
    for (int j = blockIdx.x * 4 + wave; j < n_out; j += gridDim.x * 4)
      subset_row<64>(S, U, ldu, out_modes, out_mult, out_max, j, n_in,
                     S.F + wave * kSubWaveEntries, S.Ul[wave], S.rl[wave], done, out);
  } else {
    for (int j = blockIdx.x; j < n_out; j += gridDim.x)
      subset_row<256>(S, U, ldu, out_modes, out_mult, out_max, j, n_in, S.F, S.Ul[wave],
                      S.rl[wave], done, out);
  }
}

}  // namespace tb

namespace tbsub {

// Whether a call may use the recurrence (the lattice itself is only known on the device) and is
// large enough to gain: pairs times the 2^in_max codes of a pair's walk of at least 2^20. The
// recurrence takes 14-28 us plus its share of the rows, the walk 9 us plus its pairs; they cross
// near that line (20 modes, 10 photons: k = 3, 24,000 pairs 9 us walked, 15 by recurrence;
// k = 4, 42,000: 16, 16; k = 6, 42,000: 40, 20; k = 8, 9000: 39, 26; k = 5, 1,008,000: 351, 42).
constexpr int64_t kSubMinCodes = 1 << 20;
bool attempt(int ldu, int out_max, int n_out, int in_max, int n_in) {
  if (n_out < 1 || n_in < 1 || in_max < 1 || out_max < 1 || ldu < 1) return false;
  if (ldu > tb::kSubMaxLdu || in_max > tb::kSubModes || n_in > tb::kSubMaxIn || out_max > 64)
    return false;
  return ((int64_t)n_out * n_in) << in_max >= kSubMinCodes;
}

size_t workspace(int n_out) { return (sizeof(int) * (size_t)n_out + 255) & ~(size_t)255; }

// 512 workgroups: two per CU, what their LDS allows.
int32_t run(const tb::cd *U, int ldu, const int *out_modes, const int *out_mult, int out_max,
            int n_out, const int *in_modes, const int *in_mult, int in_max, int n_in, int *done,
            tb::cd *out, hipStream_t s) {
  hipLaunchKernelGGL(tb::subset_rows_kernel, dim3(std::min(n_out, 512)), dim3(256), 0, s, in_modes,
                     in_mult, in_max, n_in, U, ldu, out_modes, out_mult, out_max, n_out, done, out);
  return tbh::check_hip(hipGetLastError(), "subset_rows_kernel");
}

}  // namespace tbsub
