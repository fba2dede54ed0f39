// Clifford & Clifford submatrices sweep kernels and their host launch (the Gray-walk
// building blocks and the formula are in sweep_impl.hpp).
#include "sweep_impl.hpp"

namespace tb {

// Stages item `item` as Vs[nu][j] = V[nu][j]: copied from gathered columns, or gathered from U
// by the item's slots (particles: the occupied input slots in order; rows: the output slots,
// repeated by multiplicity; entries past either list are 0). With fewer than K particles every
// minor has a column of zeros, so the item is all 0: its minors are then exactly 0 at whatever slot
// they are written. lists: 2K - 1 ints of LDS.
template <int K>
__device__ __forceinline__ void sweep_stage(const SweepSource &src, int item, cd *Vs, int *lists,
                                            int lane) {
  constexpr int R = K - 1;
  if (src.U == nullptr) {
    const cd *v = src.Vt + (size_t)item * src.item_stride;
    for (int e = lane; e < K * R; e += 64) {
      const int nu = e / R, j = e - nu * R;
      Vs[e] = v[(size_t)nu * src.ldv + j];
    }
    return;
  }
  int *cols = lists, *rows = lists + K;
  for (int e = lane; e < K + R; e += 64) lists[e] = -1;
  __syncthreads();
  int base = 0;
  for (int q0 = 0; q0 < src.in_max; q0 += 64) {
    const size_t q = (size_t)item * src.in_max + q0 + lane;
    const bool on = q0 + lane < src.in_max && src.in_mult[q] > 0;
    const uint64_t bal = __ballot(on);
    const int at = base + __popcll(bal & ((1ull << lane) - 1ull));
    if (on && at < K) cols[at] = src.in_modes[q];
    base += __popcll(bal);
  }
  if (base < K)
    for (int e = lane; e < K; e += 64) cols[e] = -1;
  base = 0;
  for (int q0 = 0; q0 < src.out_max; q0 += 64) {
    const size_t q = (size_t)item * src.out_max + q0 + lane;
    const int m = q0 + lane < src.out_max ? min(max(src.out_mult[q], 0), R) : 0;
    int incl = m;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    for (int e = base + incl - m; e < min(base + incl, R); ++e) rows[e] = src.out_modes[q];
    base = min(base + __shfl(incl, 63, 64), R);
  }
  __syncthreads();
  for (int e = lane; e < K * R; e += 64) {
    const int nu = e / R, j = e - nu * R;
    const int row = rows[j], col = cols[nu];
    Vs[e] = row >= 0 && col >= 0 ? src.U[(size_t)row * src.ldu + col] : cd{0.0, 0.0};
  }
}

// The tasks of a workgroup. Workgroups go round-robin over the XCDs; an XCD takes consecutive
// tasks, as many as its share of the workgroups, so with a workgroup for every task each has
// one (an eighth of the tasks, rounded up, gave some workgroups two and others none where 8 does
// not divide them: 500 k = 12 items in 500 workgroups 11.6 us instead of 19.7).
struct SweepTasks {
  int64_t first, end;
  int step;
  __device__ __forceinline__ explicit SweepTasks(int64_t total) {
    constexpr int kXcd = 8;
    const int G = gridDim.x, x = blockIdx.x % kXcd;
    const int before = x * (G / kXcd) + min(x, G % kXcd);  // workgroups of the XCDs before
    step = G / kXcd + (x < G % kXcd ? 1 : 0);
    first = total * before / G + blockIdx.x / kXcd;
    end = total * (before + step) / G;
  }
};

// Persistent grid: G one-wave blocks loop over the tasks (slot, w), slot < active
// items, w < wpi. Blocks are dispatched round-robin over the 8 XCDs (each with its own
// L2); each XCD takes a contiguous task range (SweepTasks) so that the waves of one
// item run on one XCD and its columns are fetched into one L2 only. The active item
// count may come from device memory, so a captured graph launches the same grid for
// any number of active items and idle tasks cost nothing.
template <int K, int U, int R0>
__global__ __launch_bounds__(64) TB_SWEEP_ATTR(K) void sweep_kernel(
    SweepSource src, const int *__restrict__ item_map, const int *__restrict__ item_count,
    int items, int c, int wpi, int iters, cd *__restrict__ partial) {
  constexpr int R = K - 1;
  extern __shared__ cd smem[];
  cd *Vs = smem;          // K*R
  cd *Ed = smem + K * R;  // (c - U) * 64 corrector slots
  int *lists = (int *)(Ed + (size_t)(c > U ? c - U : 0) * 64);  // 2K - 1
  const int lane = threadIdx.x;
  int nitems = items;
  if (item_count) nitems = min(items, *item_count);
  const SweepTasks own((int64_t)nitems * wpi);
  for (int64_t task = own.first; task < own.end; task += own.step) {
    const int slot = (int)(task / wpi);
    const int w = (int)(task - (int64_t)slot * wpi);
    __syncthreads();  // previous task's reads of Vs are done
    sweep_stage<K>(src, item_map ? item_map[slot] : slot, Vs, lists, lane);
    __syncthreads();
    const SweepSums<K> acc = sweep_wave<K, U, R0>(Vs, Ed, lane, c, w, wpi, iters);
    double *dst = (double *)(partial + ((size_t)slot * wpi + w) * K);
#pragma unroll
    for (int v = 0; v < SweepSums<K>::V; ++v) {
      const int e = lane_sums_index<6>(lane) + 64 * v;
      if (e < 2 * K) dst[e] = acc.v[v];
    }
  }
}

// Paired variant of sweep_kernel (same grid, tasks and partial layout). Per task the wave
// stages the item, picks the particle whose smallest column entry is largest (relative to
// the item's largest entry, at least 2^-16), swaps it into particle 1, divides the other
// columns by it and runs the paired walk; an item without such a particle takes the plain
// walk. The swap is undone when the minors are written. The pick, the column product and the
// sums of the minors are wave operations without LDS round trips (one lane multiplying the 19
// entries one after the other, one lane scanning the particles and 6 shuffles per minor
// component took 7 of the 34 us of one k = 20 item on 256 waves; the k = 13..16 sweeps of the
// sampler are 2-8% faster and its fused steps 1..12 260 -> 200 us).
// LDS: Vs | Ed | inv[R] | lists.
template <int K, int U>
__global__ __launch_bounds__(64) TB_SWEEP_PAIR_ATTR(K) void sweep_pair_kernel(
    SweepSource src, const int *__restrict__ item_map, const int *__restrict__ item_count,
    int items, int c, int wpi, int iters, cd *__restrict__ partial) {
  constexpr int R = K - 1;
  extern __shared__ cd smem[];
  cd *Vs = smem;                                       // K*R
  cd *Ed = smem + K * R;                               // (c - U) * 64
  cd *inv = Ed + (size_t)(c > U ? c - U : 0) * 64;     // R
  int *lists = (int *)(inv + R);                       // 2K - 1
  const int lane = threadIdx.x;
  int nitems = items;
  if (item_count) nitems = min(items, *item_count);
  const SweepTasks own((int64_t)nitems * wpi);
  for (int64_t task = own.first; task < own.end; task += own.step) {
    const int slot = (int)(task / wpi);
    const int w = (int)(task - (int64_t)slot * wpi);
    __syncthreads();  // previous task's reads of LDS are done
    sweep_stage<K>(src, item_map ? item_map[slot] : slot, Vs, lists, lane);
    __syncthreads();
    double mn = -1.0, mx = 0.0;  // squared magnitudes of particle `lane`'s entries
    if (lane < K) {
      mn = INFINITY;
      for (int j = 0; j < R; ++j) {
        const cd v = Vs[lane * R + j];
        const double a = fma(v.re, v.re, v.im * v.im);
        mn = fmin(mn, a);
        mx = fmax(mx, a);
      }
    }
    const double top = wave_allmax(mx), best = wave_allmax(mn);
    const bool ok = top > 0.0 && top <= 1.7976931348623157e308 && best >= kPairMinRel2 * top;
    const int pick = __ffsll((unsigned long long)__ballot(mn == best)) - 1;  // the first such particle
    SweepSums<K> acc;
    double *dst = (double *)(partial + ((size_t)slot * wpi + w) * K);
    if (!ok) {
      acc = sweep_wave<K, U, 3>(Vs, Ed, lane, c, w, wpi, iters);
    } else {
      if (pick != 1 && lane < R) {
        const cd t = Vs[R + lane];
        Vs[R + lane] = Vs[pick * R + lane];
        Vs[pick * R + lane] = t;
      }
      // Per lane < R the reciprocal of particle 1's entry, scaled by a power of two so that
      // its square stays in range, and the entry's mantissa of magnitude 1 to 2 sqrt 2.
      cd m = {1.0, 0.0};
      double e = 0.0;
      if (lane < R) {
        const cd v = Vs[R + lane];
        const int ex = ilogb(fmax(fabs(v.re), fabs(v.im)));
        m = {ldexp(v.re, -ex), ldexp(v.im, -ex)};
        const double d = fma(m.re, m.re, m.im * m.im);
        inv[lane] = {ldexp(m.re / d, -ex), ldexp(-m.im / d, -ex)};
        e = (double)ex;
      }
      __syncthreads();
      for (int q = lane; q < K * R; q += 64) {
        const int nu = q / R, j = q - nu * R;
        if (nu != 1) {
          const cd v = cmul(Vs[q], inv[j]);
          Vs[q] = {2.0 * v.re, 2.0 * v.im};
        }
      }
      // K = prod_j V[1][j] / 2 as mantissa (below 2^60) and power of two
      const cd km = wave_prod(m);
      const int ke = (int)uniform_value(wave_allsum(e)) - R;
      __syncthreads();
      acc = sweep_pair_wave<K, U>(Vs, Ed, lane, c, w, wpi, iters);
#pragma unroll
      for (int v = 0; v < SweepSums<K>::V; ++v) {
        double re, im;  // lanes < 32 hold real parts, their partners the imaginary ones
        both32(acc.v[v], re, im);
        acc.v[v] = ldexp(lane < 32 ? km.re * re - km.im * im : km.re * im + km.im * re, ke);
      }
    }
#pragma unroll
    for (int v = 0; v < SweepSums<K>::V; ++v) {
      const int q = lane_sums_index<6>(lane) + 64 * v;
      int i = q >> 1;
      if (ok && i == 1)
        i = pick;
      else if (ok && i == pick)
        i = 1;
      if (q < 2 * K) dst[2 * i + (q & 1)] = acc.v[v];
    }
  }
}

// Output d of item b: minor nu of the item, nu = d, or with in_mult the rank of slot d among the
// occupied slots (0 where it is empty).
__device__ __forceinline__ int sweep_output_minor(const int *in_mult, int in_max, int b, int d,
                                                  int K) {
  if (in_mult == nullptr) return d;
  if (in_mult[(size_t)b * in_max + d] <= 0) return -1;
  int nu = 0;
  for (int e = 0; e < d; ++e) nu += in_mult[(size_t)b * in_max + e] > 0;
  return nu < K ? nu : -1;
}

// minors[b*in_max + d] = sum_w partial[(b*wpi + w)*K + nu(d)], in w order.
__global__ void sweep_reduce_kernel(const cd *__restrict__ partial, int K, int wpi, int items,
                                    const int *__restrict__ in_mult, int in_max,
                                    cd *__restrict__ minors) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= items * in_max) return;
  const int b = idx / in_max;
  const int nu = sweep_output_minor(in_mult, in_max, b, idx - b * in_max, K);
  double re = 0.0, im = 0.0;
  if (nu >= 0) {
#pragma unroll 8
    for (int w = 0; w < wpi; ++w) {  // unrolled: the loads are in flight together
      const cd v = partial[((size_t)b * wpi + w) * K + nu];
      re += v.re;
      im += v.im;
    }
  }
  minors[idx] = {re, im};
}

// The same for many partials per item, one block per item: 256 / K slices of w, then the
// slices in order (one thread per minor took 11 us over the 256 partials of a single item).
__global__ __launch_bounds__(256) void sweep_reduce_wide_kernel(
    const cd *__restrict__ partial, int K, int wpi, const int *__restrict__ in_mult, int in_max,
    cd *__restrict__ minors) {
  __shared__ cd part[256];
  const int b = blockIdx.x;
  const int slices = 256 / K, sl = threadIdx.x / K, nu = threadIdx.x - sl * K;
  if (sl < slices) {
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int w = sl; w < wpi; w += slices) {
      const cd v = partial[((size_t)b * wpi + w) * K + nu];
      re += v.re;
      im += v.im;
    }
    part[threadIdx.x] = {re, im};
  }
  __syncthreads();
  if (threadIdx.x < K) {
    cd v = part[threadIdx.x];
    for (int s = 1; s < slices; ++s) v = cadd(v, part[s * K + threadIdx.x]);
    part[threadIdx.x] = v;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < in_max; d += 256) {
    const int i = sweep_output_minor(in_mult, in_max, b, d, K);
    minors[(size_t)b * in_max + d] = i >= 0 ? part[i] : cd{0.0, 0.0};
  }
}

}  // namespace tb

// ------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------
namespace tbs {

struct SweepPlan {
  int c, wpi, iters;
};

#ifndef TB_SWEEP_BUILTIN_MAX_C
#define TB_SWEEP_BUILTIN_MAX_C 11
#endif
// Shortest built-in walk per lane between re-seeds (bits): below it the O(k^2) seed and the
// per-chunk wave sums of the k minors outweigh the walk itself.
#ifndef TB_SWEEP_BUILTIN_MIN_C
#define TB_SWEEP_BUILTIN_MIN_C 5
#endif
constexpr int64_t kSweepMaxBlocks = 8192;  // 4 one-wave blocks per SIMD of 256 CUs x 4 SIMDs x 2
// Waves a launch should provide before the built-in plan stops shortening the chunks: 4
// per SIMD (one-wave blocks, 2 resident per SIMD, so two rounds and a short tail).
constexpr int64_t kSweepWaveTarget = 4096;

// What a wave of the sweep costs besides walking, in codes: seeding a chunk; staging and the sums.
constexpr int64_t kSweepSeedCodes = 10, kSweepWaveCodes = 10;

// Built-in chunk: the longest walk (at most 2^11 Gray steps per lane) that still gives the
// launch kSweepWaveTarget waves, but not below 2^5 steps. A batch of 4096 k = 20 items
// keeps 2^11 (4 waves per item); one k = 20 item gets 2^5 (256 waves) instead of a
// 4-wave launch. A launch that would leave SIMDs idle all the same goes on down to 2^3 steps,
// up to 1024 waves and 256 partials per item to add (us at 2^5, 2^4, 2^3, with the seeds as they
// were: one k = 14 item 17.5, 15.5, 15.0; one k = 18 item 23.4, 21.3, 20.1; 16 k = 16 items 20.8,
// 19.7, 17.2; past the lines 100 k = 16 items 28, 41, 52 and one k = 20 item 28.5, 28.1, 30.4),
// unless one wave is an item. The tuner may choose
// otherwise per (k, batch bucket).
//
// all_items: the launch sweeps all `items`, not a part of them that only the device knows, so its
// waves share the SIMDs evenly and a launch lasts as long as the SIMD with the most waves. A wave
// then walks as many chunks as make ceil(waves / 1024) times its cost least, where that is less by
// a tenth (fewer waves per SIMD hide less latency: 200 k = 15 items, less by 0.096, took 26 us
// instead of 24), or a twentieth where it saves the reduction: 2000 k = 14 items 71 -> 57 us, 1000 of
// k = 15 76 -> 65, 4 of k = 22 67 -> 60. Longer chunks in place of more of them gain up to twice that, but
// the half sums drift: 200 k = 18 items from 4e-15 to 2e-14. The partials are never more than the
// workspace, which is sized without this, holds.
inline SweepPlan sweep_plan(int k, int64_t items, int c_override, bool all_items = false) {
  SweepPlan p{};
  const int nb = k - 1;                      // Gray bits (particle 0 is fixed)
  const int u = std::min(tb::kSweepU, nb);   // static bits of the kernel for this k
  int c;
  if (c_override > 0) {
    c = c_override;
  } else {
    int want_bits = 0;  // log2(waves per item that bring the launch to the target)
    while (std::max<int64_t>(items, 1) << want_bits < kSweepWaveTarget && want_bits < 30)
      ++want_bits;
    c = std::min(TB_SWEEP_BUILTIN_MAX_C, nb - 6 - want_bits);
    c = std::max(c, std::min(TB_SWEEP_BUILTIN_MIN_C, nb - 6));
    const auto wpi = [&](int bits) { return (int64_t)1 << std::max(0, nb - bits - 6); };
    while (c > u && wpi(c) > 1 && wpi(c - 1) <= 256 && items * wpi(c - 1) <= 1024) --c;
  }
  c = std::max(c, u);
  c = std::min(c, std::min(nb, tb::kSweepMaxC));
  p.c = c;
  const int chunk_bits = nb - c;                      // log2(chunks per item)
  const int wave_bits = std::max(0, chunk_bits - 6);  // log2(waves at one chunk per lane)
  int wpi_bits = std::min(wave_bits, 13);
  if (all_items && c_override <= 0) {
    const auto cost = [&](int bits) {
      return ((items << bits) + 1023) / 1024 *
             ((((int64_t)1 << c) + kSweepSeedCodes) * ((int64_t)1 << (wave_bits - bits)) + kSweepWaveCodes);
    };
    for (int bits = wpi_bits - 1; bits >= 0; --bits)
      if (100 * cost(bits) < (bits == 0 ? 95 : 90) * cost(wpi_bits)) wpi_bits = bits;
  }
  p.wpi = 1 << wpi_bits;
  p.iters = 1 << (wave_bits - wpi_bits);
  return p;
}

// LDS per wave: the item's k(k-1) columns, 64 lanes x (c - U) corrector slots and the particle
// and row lists; the paired kernel adds the quotients' reciprocals.
inline size_t sweep_lds_bytes(int k, int c) {
  const int u = std::min(tb::kSweepU, k - 1);
  return sizeof(tb::cd) * ((size_t)k * (k - 1) + (size_t)std::max(c - u, 0) * 64) +
         sizeof(int) * (size_t)(2 * k);
}
inline size_t sweep_pair_lds_bytes(int k, int c) {
  return sweep_lds_bytes(k, c) + sizeof(tb::cd) * (size_t)(k - 1);
}
// Sizes that run the paired sweep (with a chunk holding the static block plus the pair
// bit), at 2 waves per SIMD: up to k = 21 with five particles in broadcast form, from
// k = 22 with the three static ones (206..256 VGPRs; 1, 3 and 4 values are spilled around the
// walk at k = 21, 30 and 31, and the SGPRs that staging needs, 24 bytes a lane at every k; k = 30
// and 31 are 3-7% faster than when nothing was spilled). Five broadcast particles
// spill from k = 22, and at one wave per SIMD the compiler parks broadcast columns in
// AGPRs and reloads them right before their DPP reads, a hazard that
// tests/test_dpp_hazards.py looks for. k = 31 is the largest broadcast-column sweep.
#ifndef TB_SWEEP_PAIR_MAX_K
#define TB_SWEEP_PAIR_MAX_K 31
#endif
template <int K>
constexpr bool sweep_paired() {
  return K >= tb::kSweepPairMinK && K <= TB_SWEEP_PAIR_MAX_K;
}

template <int K>
int32_t launch_sweep_k(const tb::SweepSource &src, const int *item_map, const int *item_count,
                       int items, const SweepPlan &p, tb::cd *partial,
                       hipStream_t s) {
  // Persistent grid: enough one-wave blocks to fill every SIMD a few times over.
  const int64_t tasks = (int64_t)items * p.wpi;
  const unsigned grid = (unsigned)std::min<int64_t>(tasks, tbs::kSweepMaxBlocks);
  constexpr int R0 = (K <= TB_SWEEP_BCAST_MAX_K) ? 3 : 2;
  constexpr int U = (K - 1 < tb::kSweepU) ? K - 1 : tb::kSweepU;
  if constexpr (sweep_paired<K>()) {
    if (p.c >= U + 1) {
      hipLaunchKernelGGL((tb::sweep_pair_kernel<K, U>), dim3(grid), dim3(64),
                         sweep_pair_lds_bytes(K, p.c), s, src, item_map, item_count, items,
                         p.c, p.wpi, p.iters, partial);
      return tbh::check_hip(hipGetLastError(), "sweep_pair_kernel");
    }
  }
  hipLaunchKernelGGL((tb::sweep_kernel<K, U, R0>), dim3(grid), dim3(64), sweep_lds_bytes(K, p.c), s,
                     src, item_map, item_count, items, p.c, p.wpi, p.iters,
                     partial);
  return tbh::check_hip(hipGetLastError(), "sweep_kernel");
}

template <int K = 2>
int32_t dispatch_sweep(int k, const tb::SweepSource &src, const int *item_map,
                       const int *item_count, int items, const SweepPlan &p, tb::cd *partial,
                       hipStream_t s) {
  if constexpr (K > TB_SWEEP_MAX_K) {
    return tbh::fail(TB_ERANGE, "sweep: k=%d exceeds TB_SWEEP_MAX_K=%d", k, TB_SWEEP_MAX_K);
  } else {
    if (k == K) return launch_sweep_k<K>(src, item_map, item_count, items, p, partial, s);
    return dispatch_sweep<K + 1>(k, src, item_map, item_count, items, p, partial, s);
  }
}

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t sweep_partial_bytes(int k, int items, int c_override) {
  if (k < 2 || items <= 0) return 0;
  const SweepPlan p = sweep_plan(k, items, c_override);
  return align256((size_t)items * p.wpi * k * sizeof(tb::cd));
}

void sweep_plan_of(int k, int items, int c_override, int *c, int *wpi, int *iters) {
  const SweepPlan p = sweep_plan(k, items, c_override);
  *c = p.c;
  *wpi = p.wpi;
  *iters = p.iters;
}

tb::SweepSource gathered(const tb::cd *Vt, int ldv, int64_t item_stride) {
  tb::SweepSource src{};
  src.Vt = Vt;
  src.ldv = ldv;
  src.item_stride = item_stride;
  return src;
}

// Partial sums only: partial[(item * wpi + w) * k + nu], w < *wpi. A consumer that sums
// them in w order gets the same minors as run_sweep with the same plan and up to kReduceInOrder
// of them.
int32_t run_sweep_partial(int k, const tb::cd *Vt, int ldv, int64_t item_stride,
                          const int *item_map, const int *item_count, int items, int c_override,
                          tb::cd *partial, int *wpi, hipStream_t s) {
  const SweepPlan p = sweep_plan(k, items, c_override);
  *wpi = p.wpi;
  return dispatch_sweep(k, gathered(Vt, ldv, item_stride), item_map, item_count, items, p, partial, s);
}

// Full sweep: partial sums then the fixed-order reduction into minors[items][k], or with
// in_mult into minors[items][in_max] by input slot (0 at empty ones).
constexpr int kReduceInOrder = 32;
int32_t run_sweep(int k, const tb::SweepSource &src, int items, int c_override, tb::cd *partial,
                  const int *in_mult, int in_max, tb::cd *minors, hipStream_t s) {
  const SweepPlan p = sweep_plan(k, items, c_override, true);
  const int outs = in_mult ? in_max : k;
  // One wave per item and no more slots than particles: the sums are the minors, with nothing to
  // add or place (an item with an empty slot after all is short of a particle, so all 0)
  // (one launch of two saved: 14.6 us a call instead of 17.4 up to k = 12).
  const bool direct = p.wpi == 1 && outs == k;
  int32_t rc = dispatch_sweep(k, src, nullptr, nullptr, items, p, direct ? minors : partial, s);
  if (rc || direct) return rc;
  if (p.wpi > kReduceInOrder) {
    hipLaunchKernelGGL(tb::sweep_reduce_wide_kernel, dim3(items), dim3(256), 0, s, partial, k, p.wpi,
                       in_mult, outs, minors);
  } else {
    const int total = items * outs;
    hipLaunchKernelGGL(tb::sweep_reduce_kernel, dim3((total + 255) / 256), dim3(256), 0, s, partial,
                       k, p.wpi, items, in_mult, outs, minors);
  }
  return tbh::check_hip(hipGetLastError(), "sweep_reduce_kernel");
}

}  // namespace tbs

extern "C" size_t tb_sweep_workspace_size(int32_t k, int32_t batch) {
  if (k > TB_SWEEP_MAX_K) return 0;
  return tbs::sweep_partial_bytes(k, batch, tbh::tuned(TB_TUNE_SWEEP, k, batch));
}

extern "C" int32_t tb_sweep_minors_batch(const tb_complex128 *Vt, int32_t k, int32_t ldv,
                                         int64_t item_stride, int32_t batch,
                                         tb_complex128 *minors, void *workspace,
                                         size_t workspace_bytes, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (batch < 0) return tbh::fail(TB_EINVAL, "sweep: batch=%d < 0", batch);
  if (batch == 0) return TB_OK;
  if (k < 2) return tbh::fail(TB_EINVAL, "sweep: k=%d < 2 (k == 1 has no sweep)", k);
  if (k > TB_SWEEP_MAX_K)
    return tbh::fail(TB_ERANGE, "sweep: k=%d exceeds TB_SWEEP_MAX_K=%d", k, TB_SWEEP_MAX_K);
  if (!Vt || !minors) return tbh::fail(TB_EINVAL, "sweep: NULL pointer");
  if (ldv < k - 1) return tbh::fail(TB_EINVAL, "sweep: ldv=%d < k-1=%d", ldv, k - 1);
  if (item_stride < (int64_t)k * ldv)
    return tbh::fail(TB_EINVAL, "sweep: item_stride=%lld < k*ldv", (long long)item_stride);
  const int c = tbh::tuned(TB_TUNE_SWEEP, k, batch);  // read once: size check and launch agree
  const size_t need = tbs::sweep_partial_bytes(k, batch, c);
  if (!workspace || workspace_bytes < need)
    return tbh::fail(TB_EWORKSPACE, "sweep: workspace %zu bytes < required %zu", workspace_bytes,
                     need);
  return tbs::run_sweep(k, tbs::gathered((const tb::cd *)Vt, ldv, item_stride), batch, c,
                        (tb::cd *)workspace, nullptr, 0, (tb::cd *)minors, s);
}
