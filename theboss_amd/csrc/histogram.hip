// Histogram of output samples over the reference's outcome order.
//
// Replaces the counting loop of BSSampleBasedDistributionCalculator
// (theboss/distribution_calculators/bs_sample_based_distribution_calculator.py:92-106),
// which scans the outcome list for every sample, by a direct rank: the index of an
// occupation vector in generate_possible_states(n, m, losses)
// (theboss/boson_sampling_utilities/boson_sampling_utilities.py:81-152). That list holds
// one block per particle number l (ascending; only l = n without losses), each block in
// reverse lexicographic order. Within a block, the states ranked before s are those that
// agree with s on modes < i and hold more particles in mode i; with r particles left for
// modes i..m-1 they number
//   sum_{v = s_i + 1}^{r} C(r - v + m - i - 2, m - i - 2) = C(r - s_i - 1 + m - i - 1, m - i - 1)
// (hockey stick), so the rank is a sum of m table lookups. Block l starts at
// sum_{l' < l} C(l' + m - 1, m - 1) = C(l - 1 + m, m).
//
// Every rank lies below the number of outcomes, which is below 2^31, so the table and the
// sums are 32-bit.
#include <algorithm>

#include "tb_common.hpp"

namespace tb {

// The rank's table and the samples of one tile in LDS. The table is shifted by one particle:
// row y, column r holds C(r - 1 + y, y), and 0 at r = 0, which is the term of a mode with r
// particles and y modes after it; row m gives the start of block r. A tile has one row per
// thread at an odd stride, so the lanes of a read cover all banks.
struct HistShape {
  int m, n, ld, losses;
};

template <int TH>
__device__ __forceinline__ void hist_table(unsigned *T, const HistShape &h) {
  const int W = h.n + 1, entries = (h.m + 1) * W;
  for (int d = 0; d <= h.m + h.n; ++d) {
    for (int e = threadIdx.x; e < entries; e += TH) {
      const int y = e / W, r = e - y * W;
      if (y + r != d) continue;
      T[e] = r == 0 ? 0u : (y == 0 || r == 1) ? 1u : T[e - W] + T[e - 1];
    }
    __syncthreads();
  }
}

// Four values of a tile whose rows follow each other, from value 4 e on, which is of row r and
// mode c.
__device__ __forceinline__ void hist_put(int *tile, int e, int r, int c, int4 q, int m) {
  int *d = tile + 4 * e;
  if (!(m & 1)) d += r;  // the stride is m + 1
  d[0] = q.x, d[1] = q.y;
  if (!(m & 1)) d += c + 2 >= m;  // a row may end after the first two values, and only there
  d[2] = q.z, d[3] = q.w;
}

// The values `from` on of `rows` samples, one by one: rows of any stride and start.
template <int TH>
__device__ __forceinline__ void hist_stage_each(int *tile, const int *__restrict__ src, int from,
                                                int rows, const HistShape &h) {
  const int m = h.m, pad = m | 1;
  for (int e = from + threadIdx.x; e < rows * m; e += TH) {
    const int r = e / m, c = e - r * m;
    tile[r * pad + c] = src[(int64_t)r * h.ld + c];
  }
}

// Whether rows follow each other without a gap and start on 16 bytes (a tile's first row is a
// multiple of 256 rows from the samples' first). Those are read four values per lane: 62 us for
// 2^22 samples of 20 modes, 5.4 TB/s, where one value per lane, and the lanes then walking
// rows of stride m, took 172.
__device__ __forceinline__ bool hist_wide(const int *src, const HistShape &h) {
  return h.ld == h.m && ((uintptr_t)src & 15) == 0;
}

// The `rows` samples from `src` on.
template <int TH>
__device__ __forceinline__ void hist_stage(int *tile, const int *__restrict__ src, int rows,
                                           const HistShape &h) {
  const int n4 = hist_wide(src, h) ? rows * h.m / 4 : 0;
  for (int e = threadIdx.x; e < n4; e += TH) {
    const int r = 4 * e / h.m;
    hist_put(tile, e, r, 4 * e - r * h.m, ((const int4 *)src)[e], h.m);
  }
  hist_stage_each<TH>(tile, src, 4 * n4, rows, h);
}

// The same a tile ahead: the next tile's loads are in flight while one is ranked. Up to
// 4 kHistAhead modes, what the registers hold beside a chunk's ranks.
constexpr int kHistAhead = 8;
template <int TH>
struct HistTile {
  int4 v[kHistAhead];
  bool ahead;
  int r0, c0, dr, dc;  // row and mode of the lane's first value, and of TH lanes further on

  __device__ __forceinline__ void init(const int *samples, const HistShape &h) {
    ahead = hist_wide(samples, h) && h.m <= 4 * kHistAhead;
    r0 = 4 * (int)threadIdx.x / h.m;
    c0 = 4 * (int)threadIdx.x - r0 * h.m;
    dr = 4 * TH / h.m;
    dc = 4 * TH - dr * h.m;
  }
  __device__ __forceinline__ void load(const int *__restrict__ src, int rows, const HistShape &h) {
    if (!ahead) return;
    const int n4 = rows * h.m / 4;
#pragma unroll
    for (int k = 0; k < kHistAhead; ++k) {
      const int e = k * TH + (int)threadIdx.x;
      if (e < n4) v[k] = ((const int4 *)src)[e];
    }
  }
  __device__ __forceinline__ void stage(int *tile, const int *__restrict__ src, int rows,
                                        const HistShape &h) const {
    if (!ahead) {
      hist_stage<TH>(tile, src, rows, h);
      return;
    }
    const int n4 = rows * h.m / 4;
    int r = r0, c = c0;
#pragma unroll
    for (int k = 0; k < kHistAhead; ++k) {
      const int e = k * TH + (int)threadIdx.x;
      if (e < n4) hist_put(tile, e, r, c, v[k], h.m);
      r += dr;
      c += dc;
      if (c >= h.m) {
        c -= h.m;
        ++r;
      }
    }
    hist_stage_each<TH>(tile, src, 4 * n4, rows, h);
  }
};

constexpr unsigned kHistOutside = ~0u;

// Rank of the sample in `row`, or kHistOutside. The modes are taken from the last, so the
// particles after a mode are a running sum, and the table's index is held to its row. Entries
// all of 0..n sum up to m n at most; with any other the sample is outside, whatever the sum.
__device__ __forceinline__ unsigned hist_rank(const int *row, const unsigned *T,
                                              const HistShape &h) {
  const int W = h.n + 1;
  unsigned after = 0, most = 0, rank = 0;
  const unsigned *t = T;
  for (int i = h.m - 1; i >= 0; --i, t += W) {
    rank += t[min(after, (unsigned)h.n)];
    const unsigned v = (unsigned)row[i];
    most = max(most, v);
    after += v;
  }
  if (most > (unsigned)h.n || after > (unsigned)h.n || (!h.losses && after != (unsigned)h.n))
    return kHistOutside;
  return rank + (h.losses ? t[after] : 0u);  // row m: where the block begins
}

// Adds a wave's number of samples outside the list: one atomic per wave.
__device__ __forceinline__ void hist_add_outside(bool out, unsigned *outside) {
  const uint64_t who = __ballot(out);
  if (who && outside && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)who) - 1))
    atomicAdd(outside, (unsigned)__popcll(who));
}

// Counting straight into the counters, or into LDS first where all of them fit there.
// Counter `rank` is the word counts[rank * words]: 1 for 32-bit counters, 2 for the low word
// of 64-bit ones, which no more than 2^31 - 1 samples carry out of.
//
// The atomics bound this once the ranks are cheap: 2^22 samples take 186 us with 20 million
// counters and 280 with 12376 (294 and 370 with the ranks as they were). Few counters are
// worse, as the samples meet on them: 330 counters take 1450 us. In LDS (LDS_BINS) those are
// 66 and 32 us, with one atomic per counter and workgroup at the end.
template <bool LDS_BINS, int TH>
__global__ __launch_bounds__(TH) void outcome_histogram_kernel(
    const int *__restrict__ samples, int S, HistShape h, int bins, unsigned *__restrict__ counts,
    int words, unsigned *__restrict__ outside) {
  extern __shared__ unsigned hist_lds[];
  unsigned *T = hist_lds;
  int *tile = (int *)(T + (h.m + 1) * (h.n + 1));
  unsigned *local = (unsigned *)(tile + TH * (h.m | 1));
  if (LDS_BINS)
    for (int e = threadIdx.x; e < bins; e += TH) local[e] = 0;
  hist_table<TH>(T, h);
  for (int64_t base = (int64_t)blockIdx.x * TH; base < S; base += (int64_t)gridDim.x * TH) {
    const int rows = (int)min((int64_t)TH, (int64_t)S - base);
    hist_stage<TH>(tile, samples + base * h.ld, rows, h);
    __syncthreads();
    bool out = false;
    if ((int)threadIdx.x < rows) {
      const unsigned rank = hist_rank(tile + threadIdx.x * (h.m | 1), T, h);
      out = rank == kHistOutside;
      if (!out) atomicAdd(LDS_BINS ? local + rank : counts + (int64_t)rank * words, 1u);
    }
    hist_add_outside(out, outside);
    __syncthreads();  // the tile is overwritten next
  }
  if (LDS_BINS)
    for (int e = threadIdx.x; e < bins; e += TH)
      if (const unsigned v = local[e]) atomicAdd(counts + (int64_t)e * words, v);
}

// Many counters and many samples: no atomic on memory at all. The counters are cut into
// buckets of 2^shift; a first kernel takes the samples in chunks and writes each chunk's
// ranks, their low bits as 16-bit offsets, in the order of the buckets, with a table of where
// each bucket's run begins in each chunk; a second kernel counts one bucket per workgroup in
// LDS, over its run of every chunk, and writes the counters once, so they need no clearing.
//
// The sample loads bound the first kernel and the counters' stores the second. 2^22 samples,
// per call: 160 us of 20 modes with 20 million counters, 96 of 18 modes with 100947; 178 and 134
// when a tile was loaded only after the one before it had been ranked and the offsets went from
// registers to their places in memory, two bytes each, instead of through LDS. (The direct kernel
// took 35% longer, and the 32-bit counters with a clearing and a widening pass 446.) The direct
// kernel gains nothing from loads a tile ahead: 286 counters in LDS 62 us against 49, as the
// registers cost it a workgroup per CU.
//
// Rows per thread, so samples per chunk: about 512 chunks are two workgroups per CU; fewer
// leave CUs without loads in flight (2^20 samples of 20 modes into 20 million counters in 128,
// 256 and 512 chunks, before the loads ahead: 92, 69 and 63 us), more cut the runs short (2^22 in
// 512, 1024 and 2048: 154, 170 and 180).
constexpr int kHistPartThreads = 512;
constexpr int kHistMaxShift = 14, kHistMaxBuckets = 4096;

template <int ROWS>
__global__ __launch_bounds__(kHistPartThreads) void hist_partition_kernel(
    const int *__restrict__ samples, int S, HistShape h, int shift, int buckets,
    uint16_t *__restrict__ offsets, uint16_t *__restrict__ starts, unsigned *__restrict__ outside) {
  constexpr int TH = kHistPartThreads, WAVES = TH / 64;
  extern __shared__ unsigned hist_lds[];
  unsigned *T = hist_lds;
  int *tile = (int *)(T + (h.m + 1) * (h.n + 1));
  uint16_t *sorted = (uint16_t *)tile;                                 // [ROWS * TH], at the end
  unsigned *fill = (unsigned *)(tile + TH * max(h.m | 1, ROWS / 2));  // [buckets]
  unsigned *wave_sum = fill + buckets;                                 // [WAVES]
  for (int e = threadIdx.x; e < buckets; e += TH) fill[e] = 0;
  const int64_t first = (int64_t)blockIdx.x * (ROWS * TH);
  const auto rows_at = [&](int it) {
    return (int)max((int64_t)0, min((int64_t)TH, (int64_t)S - first - it * TH));
  };
  HistTile<TH> in;
  in.init(samples, h);
  in.load(samples + first * h.ld, rows_at(0), h);
  hist_table<TH>(T, h);
  unsigned rank[ROWS], slot[ROWS];
#pragma unroll
  for (int it = 0; it < ROWS; ++it) {
    const int64_t base = first + it * TH;
    const int rows = rows_at(it);
    in.stage(tile, samples + base * h.ld, rows, h);
    if (it + 1 < ROWS) in.load(samples + (base + TH) * h.ld, rows_at(it + 1), h);
    __syncthreads();
    rank[it] = kHistOutside;
    slot[it] = 0;
    if ((int)threadIdx.x < rows) {
      rank[it] = hist_rank(tile + threadIdx.x * (h.m | 1), T, h);
      if (rank[it] != kHistOutside) slot[it] = atomicAdd(fill + (rank[it] >> shift), 1u);
    }
    hist_add_outside((int)threadIdx.x < rows && rank[it] == kHistOutside, outside);
    __syncthreads();
  }
  // exclusive sums over the buckets, a contiguous piece per thread
  const int per = (buckets + TH - 1) / TH, b0 = min((int)threadIdx.x * per, buckets),
            b1 = min(b0 + per, buckets);
  unsigned mine = 0;
  for (int b = b0; b < b1; ++b) mine += fill[b];
  unsigned upto = mine;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned v = __shfl_up(upto, o);
    if (lane >= o) upto += v;
  }
  if (lane == 63) wave_sum[wave] = upto;
  __syncthreads();
  unsigned at = upto - mine;
  for (int w = 0; w < wave; ++w) at += wave_sum[w];
  uint16_t *col = starts + blockIdx.x;
  for (int b = b0; b < b1; ++b) {
    const unsigned c = fill[b];
    fill[b] = at;
    col[(int64_t)b * gridDim.x] = (uint16_t)at;
    at += c;
  }
  unsigned total = 0;
  for (int w = 0; w < WAVES; ++w) total += wave_sum[w];
  if (threadIdx.x == TH - 1) col[(int64_t)buckets * gridDim.x] = (uint16_t)total;
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ROWS; ++it)
    if (rank[it] != kHistOutside)
      sorted[fill[rank[it] >> shift] + slot[it]] = (uint16_t)(rank[it] & ((1u << shift) - 1));
  __syncthreads();
  // two at a time; past an odd total one more of the chunk's own, which nothing reads
  unsigned *out = (unsigned *)(offsets + first);
  for (unsigned e = threadIdx.x; 2 * e < total; e += TH) out[e] = ((const unsigned *)sorted)[e];
}

constexpr int kHistCountThreads = 1024, kHistRunLanes = 8;

__global__ __launch_bounds__(kHistCountThreads) void hist_count_kernel(
    const uint16_t *__restrict__ offsets, const uint16_t *__restrict__ starts, int chunk,
    int chunks, int shift, int64_t bins, int64_t *__restrict__ counts, int add) {
  extern __shared__ unsigned hist_lds[];
  constexpr int TH = kHistCountThreads, RL = kHistRunLanes;
  const int width = 1 << shift;
  for (int e = threadIdx.x; e < width; e += TH) hist_lds[e] = 0;
  __syncthreads();
  const uint16_t *lo = starts + (int64_t)blockIdx.x * chunks, *hi = lo + chunks;
  for (int c = threadIdx.x / RL; c < chunks; c += TH / RL) {
    const int end = hi[c];
    const uint16_t *run = offsets + (int64_t)c * chunk;
    for (int i = lo[c] + (threadIdx.x & (RL - 1)); i < end; i += 4 * RL) {
      int o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = i + u * RL < end ? run[i + u * RL] : -1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (o[u] >= 0) atomicAdd(hist_lds + o[u], 1u);
    }
  }
  __syncthreads();
  const int64_t b0 = (int64_t)blockIdx.x << shift;
  const int own = (int)min((int64_t)width, bins - b0);
  for (int e = threadIdx.x; e < own; e += TH)
    counts[b0 + e] = (add ? counts[b0 + e] : 0) + (int64_t)hist_lds[e];
}

// Clears 64-bit counters and the word pair of `outside`.
__global__ __launch_bounds__(256) void hist_clear_kernel(int64_t *__restrict__ counts, int64_t bins,
                                                         int64_t *__restrict__ outside) {
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < bins; e += step) counts[e] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0 && outside) *outside = 0;
}

}  // namespace tb

namespace {

// Number of outcomes, or -1 past 2^31 - 1.
int64_t outcome_count(int n, int m, int losses) {
  // C(n + m - 1, m - 1) without losses, C(n + m, m) with (all l <= n), exact in
  // unsigned 128-bit while it stays below the limit.
  const int top = losses ? n + m : n + m - 1;
  const int k = losses ? m : m - 1;
  unsigned __int128 c = 1;
  for (int i = 1; i <= k; ++i) {
    c = c * (unsigned __int128)(top - k + i) / (unsigned __int128)i;
    if (c > (unsigned __int128)0x7fffffff) return -1;
  }
  return (int64_t)c;
}

}  // namespace

extern "C" int64_t tb_outcome_count(int32_t n, int32_t m, int32_t losses) {
  if (n < 0 || m < 1) return tbh::fail(TB_EINVAL, "outcomes: n=%d m=%d", n, m);
  if (m > TB_HIST_MAX_M || n > TB_HIST_MAX_N)
    return tbh::fail(TB_ERANGE, "outcomes: m=%d n=%d beyond %d, %d", m, n, TB_HIST_MAX_M,
                     TB_HIST_MAX_N);
  const int64_t c = outcome_count(n, m, losses ? 1 : 0);
  if (c < 0) return tbh::fail(TB_ERANGE, "outcomes: more than 2^31 - 1 states (n=%d, m=%d)", n, m);
  return c;
}

namespace {
constexpr size_t kHistLds = 160 * 1024;

size_t hist_lds_bytes(const tb::HistShape &h, int threads, int64_t words) {
  return ((size_t)(h.m + 1) * (h.n + 1) + (size_t)threads * (h.m | 1) + (size_t)words) *
         sizeof(unsigned);
}

// The partition's tile also holds a chunk's sorted offsets.
size_t hist_part_lds(const tb::HistShape &h, int rows, int64_t buckets) {
  const int tile = std::max(h.m | 1, rows / 2);
  return ((size_t)(h.m + 1) * (h.n + 1) + (size_t)tb::kHistPartThreads * tile +
          (size_t)buckets + tb::kHistPartThreads / 64) * sizeof(unsigned);
}

template <typename K>
int32_t hist_allow_lds(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return TB_OK;
  return tbh::check_hip(hipFuncSetAttribute((const void *)kernel,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                        "histogram LDS");
}

// Threads of the kernel that counts in LDS, 0 where it is not taken: the counters have to fit
// beside a tile, and a counter has to take more than a few samples.
int hist_lds_threads(const tb::HistShape &h, int64_t bins, int S) {
  if (S < 4 * bins) return 0;
  for (const int th : {1024, 512})
    if (hist_lds_bytes(h, th, bins) <= kHistLds) return th;
  return 0;
}

template <bool LDS_BINS, int TH>
int32_t hist_direct(const int32_t *samples, int S, const tb::HistShape &h, int64_t bins,
                    unsigned *counts, int words, unsigned *outside, hipStream_t s) {
  const size_t lds = hist_lds_bytes(h, TH, LDS_BINS ? bins : 0);
  auto kernel = &tb::outcome_histogram_kernel<LDS_BINS, TH>;
  if (const int32_t rc = hist_allow_lds(kernel, lds)) return rc;
  // persistent, so the table is built, and LDS counters are added, once per workgroup; as
  // many as the CUs hold at once
  const int per_cu = (int)std::min<size_t>(kHistLds / lds, LDS_BINS ? 2048 / TH : 6);
  const int64_t tiles = ((int64_t)S + TH - 1) / TH;
  hipLaunchKernelGGL(kernel, dim3((int)std::min<int64_t>(tiles, 256 * std::max(per_cu, 1))),
                     dim3(TH), lds, s, samples, S, h, (int)bins, counts, words, outside);
  return tbh::check_hip(hipGetLastError(), "outcome_histogram_kernel");
}

int32_t hist_count(const int32_t *samples, int S, const tb::HistShape &h, int64_t bins,
                   unsigned *counts, int words, unsigned *outside, hipStream_t s) {
  switch (hist_lds_threads(h, bins, S)) {
    case 1024: return hist_direct<true, 1024>(samples, S, h, bins, counts, words, outside, s);
    case 512: return hist_direct<true, 512>(samples, S, h, bins, counts, words, outside, s);
  }
  return hist_direct<false, 256>(samples, S, h, bins, counts, words, outside, s);
}

// The partition of the large case: about 1024 buckets, more where a bucket would not fit LDS.
struct HistParts {
  bool use;
  int shift, buckets, rows, chunk, slab_chunks;
  size_t starts_at, bytes;  // of the table in the workspace; whole workspace
};

// From here on the partition is the faster one: 2^18 samples take 49 us with 20 million
// counters and 26 with 177100 (direct 47 and 23), 2^20 take 63 and 39 (direct 76 and 58).
constexpr int kHistPartMinSamples = 1 << 19;

// Samples whose ranks are held at a time (32 MiB).
constexpr int64_t kHistSlab = 1 << 24;

HistParts hist_parts(const tb::HistShape &h, int64_t bins, int S) {
  HistParts p{};
  if (S < kHistPartMinSamples || hist_lds_threads(h, bins, S)) return p;
  while (p.shift < tb::kHistMaxShift && (bins >> p.shift) >= 1024) ++p.shift;
  const int64_t buckets = ((bins - 1) >> p.shift) + 1;
  p.rows = S <= 1 << 20 ? 4 : S <= 1 << 21 ? 8 : 16;
  if (buckets > tb::kHistMaxBuckets || hist_part_lds(h, p.rows, buckets) > kHistLds) return p;
  p.use = true;
  p.buckets = (int)buckets;
  p.chunk = p.rows * tb::kHistPartThreads;
  const int64_t most = std::min<int64_t>(S, kHistSlab);
  p.slab_chunks = (int)((most + p.chunk - 1) / p.chunk);
  p.starts_at = (size_t)p.slab_chunks * p.chunk * sizeof(uint16_t);
  p.bytes = p.starts_at + (size_t)p.slab_chunks * (buckets + 1) * sizeof(uint16_t);
  return p;
}

int32_t hist_check(const int32_t *samples, int32_t ld, int32_t S, int32_t m, int32_t n,
                   int32_t losses, const void *counts, int64_t *bins) {
  if (S < 0) return tbh::fail(TB_EINVAL, "histogram: samples=%d < 0", S);
  *bins = tb_outcome_count(n, m, losses);
  if (*bins < 0) return (int32_t)*bins;
  if (S == 0) return TB_OK;
  if (!samples || !counts) return tbh::fail(TB_EINVAL, "histogram: NULL pointer");
  if (ld < m) return tbh::fail(TB_EINVAL, "histogram: ld=%d < m=%d", ld, m);
  return TB_OK;
}

}  // namespace
extern "C" int32_t tb_outcome_histogram(const int32_t *samples, int32_t ld, int32_t samples_n,
                                        int32_t m, int32_t n, int32_t losses, uint32_t *counts,
                                        uint32_t *outside, void *stream) {
  int64_t bins = 0;
  const int32_t rc = hist_check(samples, ld, samples_n, m, n, losses, counts, &bins);
  if (rc != TB_OK || samples_n == 0) return rc;
  const tb::HistShape h{m, n, ld, losses ? 1 : 0};
  return hist_count(samples, samples_n, h, bins, counts, 1, outside, (hipStream_t)stream);
}

extern "C" size_t tb_outcome_histogram64_workspace_size(int32_t samples_n, int32_t m, int32_t n,
                                                        int32_t losses) {
  const int64_t bins = samples_n > 0 ? tb_outcome_count(n, m, losses) : 0;
  return bins > 0 ? hist_parts({m, n, m, losses ? 1 : 0}, bins, samples_n).bytes : 0;
}

extern "C" int32_t tb_outcome_histogram64(const int32_t *samples, int32_t ld, int32_t samples_n,
                                          int32_t m, int32_t n, int32_t losses, int64_t *counts,
                                          int64_t *outside, void *workspace,
                                          size_t workspace_bytes, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  int64_t bins = 0;
  if (const int32_t rc = hist_check(samples, ld, samples_n, m, n, losses, counts, &bins)) return rc;
  if (!counts) return tbh::fail(TB_EINVAL, "histogram: NULL pointer");
  const tb::HistShape h{m, n, ld, losses ? 1 : 0};
  const HistParts p = hist_parts(h, bins, samples_n);
  const bool parts =
      p.use && workspace && ((uintptr_t)workspace & 3) == 0 && workspace_bytes >= p.bytes;
  const int64_t clear = parts ? 0 : bins;
  hipLaunchKernelGGL(tb::hist_clear_kernel,
                     dim3((int)std::min<int64_t>(std::max<int64_t>((clear + 255) / 256, 1), 4096)),
                     dim3(256), 0, s, counts, clear, outside);
  if (const int32_t rc = tbh::check_hip(hipGetLastError(), "hist_clear_kernel")) return rc;
  if (samples_n == 0) return TB_OK;
  if (!parts)
    return hist_count(samples, samples_n, h, bins, (unsigned *)counts, 2, (unsigned *)outside, s);
  uint16_t *offsets = (uint16_t *)workspace;
  uint16_t *starts = (uint16_t *)((char *)workspace + p.starts_at);
  const size_t lds = hist_part_lds(h, p.rows, p.buckets);
  const size_t lds_count = sizeof(unsigned) << p.shift;
  auto partition = p.rows == 4   ? &tb::hist_partition_kernel<4>
                   : p.rows == 8 ? &tb::hist_partition_kernel<8>
                                 : &tb::hist_partition_kernel<16>;
  if (const int32_t rc = hist_allow_lds(partition, lds)) return rc;
  for (int64_t at = 0; at < samples_n; at += kHistSlab) {
    const int S = (int)std::min<int64_t>(kHistSlab, samples_n - at);
    const int chunks = (S + p.chunk - 1) / p.chunk;
    hipLaunchKernelGGL(partition, dim3(chunks), dim3(tb::kHistPartThreads), lds, s,
                       samples + at * ld, S, h, p.shift, p.buckets, offsets, starts,
                       (unsigned *)outside);
    if (const int32_t rc = tbh::check_hip(hipGetLastError(), "hist_partition_kernel")) return rc;
    hipLaunchKernelGGL(tb::hist_count_kernel, dim3(p.buckets), dim3(tb::kHistCountThreads),
                       lds_count, s, offsets, starts, p.chunk, chunks, p.shift, bins, counts, at > 0);
    if (const int32_t rc = tbh::check_hip(hipGetLastError(), "hist_count_kernel")) return rc;
  }
  return TB_OK;
}
