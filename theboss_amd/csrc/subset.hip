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
// multiplies: n = 10, k = 5: 2560 against 40,000. No inclusion-exclusion signs enter: the terms
// are products of entries, so the error is bounded by the permanent of the entries' moduli, where
// the alternating sums start from terms up to 2^k times larger (not by |perm|: entries of any
// phase still cancel). Measured on 200 prefixes of 10 modes, k = 5: 2.7e-16 against 2.8e-15.
//
// What bounds it (GCC-A layer of 200 prefixes x 20 outputs x C(10, 5) inputs, 1.0M pairs: 30 us a
// call, 4 of them the 16 MB written; the walk 351): a workgroup first builds the lattice from
// the input rows, 19,000 cycles of latency (in LDS, for itself: a plan kernel with predecessor
// lists in global memory took 20 us more per call); then a wave per output row walks the levels
// (the whole workgroup where the levels are wide or the rows few), 17,000 cycles a row with the
// eight waves of a CU sharing its LDS reads. Slots loaded all at once and a row ahead, levels
// unrolled, and ranks that share their low bits: 42 us before, with the walk's flags (below); 12
// modes, k = 6, 1200 rows: 77 -> 54. The Guan walk follows in stream order over the rows whose
// done flag is 0, whose particle number differs, or over all of them when the lattice is too large.
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

// An input row in registers, all its slots loaded at once (in_max <= kSubModes); slots past
// in_max are empty. Slot by slot the loads of the plan came one latency after the other.
struct SubsetIn {
  int d[kSubModes], m[kSubModes];
};
__device__ __forceinline__ SubsetIn subset_in(const int *__restrict__ in_modes,
                                              const int *__restrict__ in_mult, int in_max, int i) {
  SubsetIn r;
  const int *sm = in_modes + (size_t)i * in_max, *su = in_mult + (size_t)i * in_max;
#pragma unroll
  for (int q = 0; q < kSubModes; ++q) {
    const int at = min(q, in_max - 1);
    r.d[q] = sm[at];
    r.m[q] = su[at];
  }
#pragma unroll
  for (int q = 0; q < kSubModes; ++q) r.m[q] = q < in_max ? max(r.m[q], 0) : 0;
  return r;
}

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
  const SubsetIn first = subset_in(in_modes, in_mult, in_max, 0);
  SubsetIn in = subset_in(in_modes, in_mult, in_max, min(tid, n_in - 1));
#pragma unroll
  for (int q = 0; q < kSubModes; ++q) k += min(first.m[q], kSubK + 1);
  __syncthreads();
  for (int i = tid; i < n_in; i += 256) {
    if (i != tid) in = subset_in(in_modes, in_mult, in_max, i);
    int sum = 0;
    bool refuse = false;
#pragma unroll
    for (int q = 0; q < kSubModes; ++q) {
      const int m = in.m[q], d = in.d[q];
      if (m == 0) continue;
      sum += min(m, kSubK + 1);
      if (d < 0 || d >= ldu || m > kSubK) {
        refuse = true;
        continue;
      }
      int all = m;  // a mode may fill several slots
#pragma unroll
      for (int r = 0; r < q; ++r) all += in.d[r] == d ? min(in.m[r], kSubK + 1) : 0;
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
    if (n_in > 256) in = subset_in(in_modes, in_mult, in_max, i);
    int code = 0;
#pragma unroll
    for (int q = 0; q < kSubModes; ++q)
      if (in.m[q] > 0) code += in.m[q] * p.stride[S.top[in.d[q]]];
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
    int low = 0, n_low = 0;  // of the eight bits that a thread's points share
    for (int m = min(tid, p.total - 1); m; m &= m - 1) low += S.binom[__ffs(m) - 1][++n_low];
    for (int c = tid; c < p.total; c += 256) {
      int r = low, i = n_low;
      for (int m = c >> 8; m; m &= m - 1) r += S.binom[7 + __ffs(m)][++i];
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

// Level L from level L - 1 by the T threads of a group (t inside it), one particle per mode:
// every point of the level has L bits. Unrolled, so that the reads of a point are all in flight.
template <int T, int L>
__device__ __forceinline__ void subset_level_bits(const SubsetLds &S, const cd *src, cd *dst,
                                                  const cd *u, int t) {
  const int cnt = S.p.cnt[L];
  const unsigned short *order = S.order + S.p.off[L];
  for (int i = t; i < cnt; i += T) {
    const int c = order[i];
    double re = 0.0, im = 0.0;
    int m = c;
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int bit = m & -m;
      m ^= bit;
      cfma(re, im, u[__ffs(bit) - 1], src[S.pos[c ^ bit]]);
    }
    dst[i] = {re, im};
  }
}

// The same with several particles per mode.
template <int T>
__device__ __forceinline__ void subset_level_multi(const SubsetLds &S, const cd *src, cd *dst,
                                                   const cd *u, int l, int t) {
  const SubsetPlan &p = S.p;
  const int cnt = p.cnt[l];
  const unsigned short *order = S.order + p.off[l];
  for (int i = t; i < cnt; i += T) {
    const int c = order[i];
    double re = 0.0, im = 0.0;
    for (int d = 0; d < p.D; ++d) {
      const int st = p.stride[d];
      const int s = (c / st) % p.radix[d];
      if (s == 0) continue;
      const cd w = u[d];
      cfma(re, im, {(double)s * w.re, (double)s * w.im}, src[S.pos[c - st]]);
    }
    dst[i] = {re, im};
  }
}

template <int T>
__device__ __forceinline__ void subset_level(const SubsetLds &S, const cd *src, cd *dst, const cd *u,
                                             int l, int t) {
  if (S.p.multi) {
    subset_level_multi<T>(S, src, dst, u, l, t);
    return;
  }
  static_assert(kSubK == 12, "a case for each level");
  switch (l) {
    case 1: subset_level_bits<T, 1>(S, src, dst, u, t); break;
    case 2: subset_level_bits<T, 2>(S, src, dst, u, t); break;
    case 3: subset_level_bits<T, 3>(S, src, dst, u, t); break;
    case 4: subset_level_bits<T, 4>(S, src, dst, u, t); break;
    case 5: subset_level_bits<T, 5>(S, src, dst, u, t); break;
    case 6: subset_level_bits<T, 6>(S, src, dst, u, t); break;
    case 7: subset_level_bits<T, 7>(S, src, dst, u, t); break;
    case 8: subset_level_bits<T, 8>(S, src, dst, u, t); break;
    case 9: subset_level_bits<T, 9>(S, src, dst, u, t); break;
    case 10: subset_level_bits<T, 10>(S, src, dst, u, t); break;
    case 11: subset_level_bits<T, 11>(S, src, dst, u, t); break;
    case 12: subset_level_bits<T, 12>(S, src, dst, u, t); break;
  }
}

// A lane's slot of an output row (out_max <= 64); empty past the row's slots and past the rows.
struct SubsetSlot {
  int m, d;
};
__device__ __forceinline__ SubsetSlot subset_slot(const int *__restrict__ out_modes,
                                                  const int *__restrict__ out_mult, int out_max,
                                                  int n_out, int64_t j) {
  const int lane = threadIdx.x & 63;
  if (lane >= out_max || j >= n_out) return {0, 0};
  return {max(out_mult[j * out_max + lane], 0), out_modes[j * out_max + lane]};
}

// Output row j, of these slots, by the T threads of a group; F holds two levels of p.width
// values.
template <int T>
__device__ __forceinline__ void subset_row(SubsetLds &S, const cd *__restrict__ U, int ldu,
                                           SubsetSlot slot, int j, int n_in, cd *F, cd *Ul, int *rl,
                                           int *__restrict__ done, cd *__restrict__ out) {
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
  // The row's particles, one after the other.
  const int m = slot.m, md = slot.d;
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
    subset_level<T>(S, src, dst, Ul + (l - 1) * p.D, l, t);
    sync();
  }
  const cd *last = F + ((p.k & 1) ? p.width : 0);
  for (int i = t; i < n_in; i += T) out[(size_t)j * n_in + i] = last[S.in_pos[i]];
  sync();
}

__global__ __launch_bounds__(256) void subset_rows_kernel(
    const int *__restrict__ in_modes, const int *__restrict__ in_mult, int in_max, int n_in,
    const cd *__restrict__ U, int ldu, const int *__restrict__ out_modes,
    const int *__restrict__ out_mult, int out_max, int n_out, int *__restrict__ done, int counters,
    cd *__restrict__ out) {
  __shared__ SubsetLds S;
  const int wave = threadIdx.x >> 6;
  // A row per wave or per workgroup, its slots loaded while the plan is made or the row before
  // it is done; which of the two is known for most calls before the plan.
  const bool many = n_out >= kSubWaveRows;
  int64_t j = many ? blockIdx.x * 4 + wave : blockIdx.x;
  SubsetSlot slot = subset_slot(out_modes, out_mult, out_max, n_out, j);
  subset_plan(S, in_modes, in_mult, in_max, n_in, ldu);
  if (!S.p.ok) {  // nothing is done: counters for the walk that follows, in place of the flags
    if (blockIdx.x == 0 && (int)threadIdx.x < counters)
      done[threadIdx.x * kSubCounterStride] = INT32_MIN;
    return;
  }
  const bool waves = many && 2 * S.p.width <= kSubWaveEntries;
  if (many && !waves) {
    j = blockIdx.x;
    slot = subset_slot(out_modes, out_mult, out_max, n_out, j);
  }
  const int64_t step = (int64_t)gridDim.x * (waves ? 4 : 1);
  for (; j < n_out; j += step) {
    const SubsetSlot next = subset_slot(out_modes, out_mult, out_max, n_out, j + step);
    if (waves)
      subset_row<64>(S, U, ldu, slot, (int)j, n_in, S.F + wave * kSubWaveEntries, S.Ul[wave],
                     S.rl[wave], done, out);
    else
      subset_row<256>(S, U, ldu, slot, (int)j, n_in, S.F, S.Ul[wave], S.rl[wave], done, out);
    slot = next;
  }
}

}  // namespace tb

namespace tbsub {

// Whether a call may use the recurrence (the lattice itself is only known on the device) and is
// large enough to gain: pairs times the 2^in_max codes of a pair's walk of at least 2^20. The
// recurrence takes 14-28 us plus its share of the rows, the walk 9 us plus its pairs; they cross
// near that line (20 modes, 10 photons: k = 3, 24,000 pairs 9 us walked, 15 by recurrence;
// k = 4, 42,000: 16, 16; k = 6, 42,000: 40, 19; k = 8, 9000: 39, 26; k = 5, 1,008,000: 351, 32).
constexpr int64_t kSubMinCodes = 1 << 20;
bool attempt(int ldu, int out_max, int n_out, int in_max, int n_in) {
  if (n_out < 1 || n_in < 1 || in_max < 1 || out_max < 1 || ldu < 1) return false;
  if (ldu > tb::kSubMaxLdu || in_max > tb::kSubModes || n_in > tb::kSubMaxIn || out_max > 64)
    return false;
  return ((int64_t)n_out * n_in) << in_max >= kSubMinCodes;
}

// Bytes of the flags, the least a workspace may hold, and with all the counters.
size_t flag_bytes(int n_out) { return (sizeof(int) * (size_t)n_out + 255) & ~(size_t)255; }
size_t workspace(int n_out) {
  return std::max(flag_bytes(n_out), sizeof(int) * tb::kSubCounters * tb::kSubCounterStride);
}

// 512 workgroups: two per CU, what their LDS allows.
int32_t run(const tb::cd *U, int ldu, const int *out_modes, const int *out_mult, int out_max,
            int n_out, const int *in_modes, const int *in_mult, int in_max, int n_in, int *done,
            int counters, tb::cd *out, hipStream_t s) {
  hipLaunchKernelGGL(tb::subset_rows_kernel, dim3(std::min(n_out, 512)), dim3(256), 0, s, in_modes,
                     in_mult, in_max, n_in, U, ldu, out_modes, out_mult, out_max, n_out, done, counters, out);
  return tbh::check_hip(hipGetLastError(), "subset_rows_kernel");
}

}  // namespace tbsub
