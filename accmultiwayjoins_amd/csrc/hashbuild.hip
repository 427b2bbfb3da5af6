// Bucketed hash-table build (the AMHJ build phase).
//
// Reference: QueryProcessor::build_hash_multiway (MHJ-GPU/QueryProcessor.cuh:76-110) builds,
// for each build relation, B = floorPowerOf2(N) buckets on the first column with bucket of key
// k = k & (B-1), by a multi-pass MSB-first radix partition with atomics
// (MHJ-GPU/Indexing/radix_partitioning.cuh:17-48, :423-497). The row order inside a bucket is
// arbitrary there, and payload columns are reached through idx_in_origin gathers.
//
// Here the same bucket function is kept, but the table is built by a stable LSD radix sort of
// one 64-bit composite key per row:
//     hi32 = rotr32(key, log_b)   -> bucket bits on top, the remaining key bits below
//     lo32 = val ^ 0x80000000     -> signed value order (only sorted on when requested)
// so rows end bucket-major and key-minor (each key's rows form one contiguous run) and the
// second column is stored inline next to its key (no idx_in_origin gather on the probe).
//
// Two builds of the same table: up to kHashSmallRows rows one workgroup sorts the rows in LDS and
// writes everything (hash_small_kernel); above, the columns go through the tiled radix sort
// (colsort.hip) and one more launch derives the bucket index (bucket_index_kernel).
#include "colsort.h"

namespace amj {

// First row of [0, n) whose bucket is >= b, found by a whole wave: 64 positions per step, so four
// dependent loads for 16 M rows.
__device__ __forceinline__ uint64_t wave_lower_bucket(const int32_t* __restrict__ keys, uint64_t n,
                                                      uint32_t mask, uint64_t b) {
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t pos = lo + (uint64_t)lane_id() * step;
    const bool less = pos < hi && (uint64_t)((uint32_t)keys[pos < hi ? pos : lo] & mask) < b;
    const uint64_t k = (uint64_t)__popcll(__ballot(less));
    if (k == 0) break;
    const uint64_t next = lo + k * step;
    lo += (k - 1) * step + 1;
    hi = next < hi ? next : hi;
  }
  return lo;
}

// Bucket pointers of the sorted keys: ptrs[b] = first row whose bucket is >= b, ptrs[B] = n. A workgroup takes kIdxBuckets consecutive buckets: it finds their rows, reads those keys
// once, in order, notes the first row of every bucket present in LDS, and a suffix minimum over
// the buckets fills the empty ones. A workgroup whose buckets hold more than kIdxScanRows
// rows (a heavy key) searches each bucket's bound instead, so no workgroup reads a long run. One
// search per bucket in all of [0, n) (the only way before) took 53 us for 4 M rows and buckets,
// this 20 us.
constexpr uint32_t kIdxBuckets = 2048;
constexpr uint32_t kIdxItems = kIdxBuckets / kBlock;
constexpr uint64_t kIdxScanRows = 16 * kIdxBuckets;
__global__ __launch_bounds__(kBlock) void bucket_index_kernel(const int32_t* __restrict__ keys,
                                                              uint64_t n, uint64_t buckets,
                                                              uint32_t* __restrict__ ptrs) {
  __shared__ uint32_t first[kIdxBuckets];
  __shared__ uint64_t range[2];
  __shared__ uint32_t wave_min[kWavesPerBlock];
  const uint32_t mask = (uint32_t)(buckets - 1);
  const uint64_t b0 = (uint64_t)blockIdx.x * kIdxBuckets;
  const uint32_t nb = (uint32_t)(buckets - b0 < kIdxBuckets ? buckets - b0 : kIdxBuckets);
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  if (w < 2) {
    const uint64_t r = wave_lower_bucket(keys, n, mask, w == 0 ? b0 : b0 + nb);
    if (lane == 0) range[w] = r;
  }
  for (uint32_t i = tid; i < kIdxBuckets; i += kBlock) first[i] = 0xffffffffu;
  __syncthreads();
  const uint64_t r0 = range[0], r1 = range[1];
  if (r1 - r0 <= kIdxScanRows) {
    for (uint64_t r = r0 + tid; r < r1; r += kBlock) {
      const uint32_t b = (uint32_t)keys[r] & mask;
      if (r == r0 || ((uint32_t)keys[r - 1] & mask) != b) first[b - (uint32_t)b0] = (uint32_t)r;
    }
  } else {
    for (uint32_t i = tid; i < nb; i += kBlock) {
      uint64_t lo = r0, hi = r1;
      while (lo < hi) {
        const uint64_t mid = lo + ((hi - lo) >> 1);
        if (((uint32_t)keys[mid] & mask) < (uint32_t)b0 + i) lo = mid + 1;
        else hi = mid;
      }
      first[i] = (uint32_t)lo;
    }
  }
  __syncthreads();
  uint32_t v[kIdxItems];
  uint32_t m = 0xffffffffu;
#pragma unroll
  for (int i = (int)kIdxItems - 1; i >= 0; --i) {
    v[i] = first[tid * kIdxItems + i];
    m = min(m, v[i]);
  }
  uint32_t suf = m;  // minimum over the lanes from this one on
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_down(suf, d, kWave);
    if (lane + d < kWave) suf = min(suf, y);
  }
  if (lane == 0) wave_min[w] = suf;
  uint32_t after = __shfl_down(suf, 1, kWave);
  if (lane == kWave - 1) after = 0xffffffffu;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWavesPerBlock; ++i)
    if (i > w) after = min(after, wave_min[i]);
  after = min(after, (uint32_t)r1);
#pragma unroll
  for (int i = (int)kIdxItems - 1; i >= 0; --i) {
    after = min(after, v[i]);
    first[tid * kIdxItems + i] = after;
  }
  __syncthreads();
  for (uint32_t i = tid; i < nb; i += kBlock) ptrs[b0 + i] = first[i];
  if (b0 + nb == buckets && tid == 0) ptrs[buckets] = (uint32_t)n;
}

hipError_t launch_bucket_index(const int32_t* keys, uint64_t n, uint64_t buckets, uint32_t* ptrs,
                               hipStream_t s) {
  const uint64_t blocks = (buckets + kIdxBuckets - 1) / kIdxBuckets;
  hipLaunchKernelGGL(bucket_index_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, keys, n,
                     buckets, ptrs);
  return hipGetLastError();
}

// The whole build of a table of up to 1024 * ITEMS rows in one workgroup: rows in registers, every
// sorting pass through one LDS copy, then the columns and the bucket pointers. Bound
// by the latency of its few passes: 16 us for 4,096 rows, where the tiled build (three kernels per
// digit and three around them) takes about 90. 8,192 rows are what registers and LDS hold at
// eight rows per lane.
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
template <int ITEMS>
__global__ __launch_bounds__(kSmallThreads) void hash_small_kernel(
    const ColSort c, uint32_t log_b, uint32_t* __restrict__ ptrs,
    uint32_t* __restrict__ flag_out) {
  __shared__ uint64_t tile[kSmallThreads * ITEMS];
  __shared__ uint32_t wrun[kSmallWaves][256];
  __shared__ uint64_t wave_or[kSmallWaves];
  __shared__ uint32_t scan_lds[4];
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const uint32_t n = (uint32_t)c.n;
  const uint32_t base = (uint32_t)w * (kWave * ITEMS) + (uint32_t)lane;
  uint64_t key[ITEMS];
  uint64_t diff = 0;
  bool out = false;
  with_rows(c, c.in64, [&](auto load) {
    const uint64_t k0 = load(0);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = base + (uint32_t)r * kWave;
      key[r] = load(i < n ? i : n - 1);
      diff |= key[r] ^ k0;
      out |= rotl32((uint32_t)(key[r] >> 32), c.rot) >= c.key_limit;
      if (i >= n) key[r] = ~0ull;  // rows past the end sort last: largest, and last in the input
    }
  });
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) diff |= __shfl_xor(diff, d, kWave);
  if (lane == 0) wave_or[w] = diff;
  const bool any_out = __syncthreads_or(out);
  diff = 0;
#pragma unroll
  for (int i = 0; i < kSmallWaves; ++i) diff |= wave_or[i];
  // the passes keep the rows past the end last: their digits are the largest, and they come last
  // in the input of the first pass
  bool placed = false;
  for (int d = 0; d < 8; ++d) {
    if (!((c.mask >> d) & 1u) || ((diff >> (8 * d)) & 0xffull) == 0) continue;
    const uint32_t shift = 8u * (uint32_t)d;
#pragma unroll
    for (int i = 0; i < kSmallWaves * 256 / kSmallThreads; ++i)
      (&wrun[0][0])[i * kSmallThreads + tid] = 0;
    __syncthreads();
    uint32_t rk[ITEMS];
    rank_rounds(key, rk, shift, wrun[w], [](int) { return true; });
    __syncthreads();
    uint32_t tot = 0;
    if (tid < 256)
#pragma unroll
      for (int i = 0; i < kSmallWaves; ++i) tot += wrun[i][tid];
    uint32_t all;
    uint32_t q = scan256(tot, scan_lds, &all);
    if (tid < 256)
#pragma unroll
      for (int i = 0; i < kSmallWaves; ++i) {
        const uint32_t t = wrun[i][tid];
        wrun[i][tid] = q;
        q += t;
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      tile[wrun[w][(uint32_t)(key[r] >> shift) & 0xffu] + rk[r]] = key[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) key[r] = tile[base + (uint32_t)r * kWave];
    placed = true;
    __syncthreads();
  }
  if (!placed) {  // all rows equal in the sorted digits: as they came
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) tile[base + (uint32_t)r * kWave] = key[r];
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = base + (uint32_t)r * kWave;
    if (i < n) col_store(c, i, key[r]);
  }
  if (!ptrs) return;
  const uint32_t buckets = 1u << log_b;
  const auto bucket = [&](uint32_t i) {
    return log_b == 0 ? 0u : (uint32_t)(tile[i] >> 32) >> (32u - log_b);
  };
  const auto lower = [&](uint32_t b) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (bucket(mid) < b) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  for (uint32_t b = (uint32_t)tid; b < buckets; b += kSmallThreads) ptrs[b] = lower(b);
  if (tid == 0) {
    ptrs[buckets] = n;
    *flag_out = any_out ? 1u : 0u;
  }
}

hipError_t launch_hash_small(const ColSort& c, uint32_t log_b, uint32_t* ptrs,
                             uint32_t* flag_out, hipStream_t s) {
  if (c.n == 0 || c.n > kHashSmallRows) return hipErrorInvalidValue;
#define LAUNCH(I)                                                                               \
  hipLaunchKernelGGL(hash_small_kernel<I>, dim3(1), dim3(kSmallThreads), 0, s, c, log_b, ptrs, \
                     flag_out)
  if (c.n <= kSmallThreads) LAUNCH(1);
  else if (c.n <= 4 * kSmallThreads) LAUNCH(4);
  else LAUNCH(8);
#undef LAUNCH
  return hipGetLastError();
}

hipError_t launch_small_sort(const ColSort& c, hipStream_t s) {
  return launch_hash_small(c, 0, nullptr, nullptr, s);
}

// Bucket bounds of sorted composites (the pairwise engine's partitions).
__device__ __forceinline__ uint64_t bucket_of(uint64_t comp, uint32_t log_b) {
  return log_b == 0 ? 0ull : (uint64_t)((uint32_t)(comp >> 32) >> (32u - log_b));
}

// ptrs[b] = first row whose bucket is >= b (ptrs[B] = n): one lower-bound search per bucket,
// so the work per thread stays logarithmic however skewed the buckets are.
__global__ __launch_bounds__(kBlock) void bucket_ptrs_kernel(const uint64_t* __restrict__ comp,
                                                             uint64_t n, uint32_t log_b,
                                                             uint64_t buckets,
                                                             uint32_t* __restrict__ ptrs) {
  for (uint64_t b = (uint64_t)blockIdx.x * kBlock + threadIdx.x; b <= buckets;
       b += (uint64_t)gridDim.x * kBlock) {
    uint64_t lo = 0, hi = n;  // first row with bucket >= b lies in [lo, hi]
    while (lo < hi) {
      const uint64_t mid = lo + ((hi - lo) >> 1);
      if (bucket_of(comp[mid], log_b) < b) lo = mid + 1;
      else hi = mid;
    }
    ptrs[b] = (uint32_t)lo;
  }
}

static unsigned grid_for(uint64_t n) {
  uint64_t g = (n + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  if (g == 0) g = 1;
  return (unsigned)g;
}

hipError_t launch_bucket_ptrs(const uint64_t* comp, uint64_t n, uint32_t log_b,
                              uint64_t buckets, uint32_t* ptrs, hipStream_t s) {
  if (n == 0) return hipMemsetAsync(ptrs, 0, (buckets + 1) * sizeof(uint32_t), s);
  hipLaunchKernelGGL(bucket_ptrs_kernel, dim3(grid_for(buckets + 1)), dim3(kBlock), 0, s, comp,
                     n, log_b, buckets, ptrs);
  return hipGetLastError();
}

}  // namespace amj
