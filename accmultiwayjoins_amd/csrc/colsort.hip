// Radix sort of rows straight from their columns (hash tables, grouped probe rows, tries, launch
// orders), with the digits chosen on the device.
//
// A row's composite is (rotr32(key ^ flip, rot) << 32) | (val ^ 2^31). A sort is one statistics
// pass over the columns (the bits in which rows differ, whether they are already in order,
// whether a key lies past the bucket range) and three launches per pass: the digit counts of
// every tile, their scan (one workgroup per digit value) and the scatter. The first pass packs
// the composites as it reads the columns and the last one writes the finished columns. The first
// pass takes its digit from the statistics in device memory; the host reads them (its wait is
// over before that pass is) and launches exactly the passes left.
//
// What it replaces packed the composites in a pass of their own, found the differing bits in a
// second one behind a host wait, scanned the counts in three launches and unpacked in a last
// pass: 16 B per row and sorting pass + 48 B per row besides; here 24 B per sorting pass + 8 B.
// Three tables of 4 M rows and a probe relation of 16 M (20-bit keys, three digits each) with
// their bucket indexes: 1.34 ms of kernels before, 0.80 ms now.
#include <algorithm>

#include "colsort.h"

namespace amj {

constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / kWave;
constexpr int kTileItems = 16;
constexpr int kTile = kTileThreads * kTileItems;  // rows per tile
constexpr int kDigits = 256;

struct SortStats {
  uint64_t diff;  // bits in which some row differs from the first
  uint32_t flags;  // kDown, kPast
  uint32_t pad;
};
constexpr uint32_t kDown = 1;  // some row orders below its predecessor (in the sorted digits)
constexpr uint32_t kPast = 2;  // some key lies at or past key_limit

static uint64_t tiles_of(uint64_t n) { return (n + kTile - 1) / kTile; }

// statistics, then the 256 digit totals of the running pass, then the tile counts
constexpr size_t kTotalsAt = 256;
constexpr size_t kFixedBytes = kTotalsAt + kDigits * sizeof(uint32_t);

size_t col_sort_temp_bytes(uint64_t n) {
  return kFixedBytes + (size_t)kDigits * tiles_of(n) * sizeof(uint32_t);
}

__device__ __forceinline__ uint64_t digit_bits(uint32_t mask) {
  uint64_t m = 0;
#pragma unroll
  for (int d = 0; d < 8; ++d)
    if ((mask >> d) & 1u) m |= 0xffull << (8 * d);
  return m;
}

// One read of the columns, bound by it.
constexpr int kStatRounds = 8;
__global__ __launch_bounds__(kBlock) void sort_stats_kernel(const ColSort c, SortStats* st) {
  const uint64_t sorted = digit_bits(c.mask);
  const uint64_t limit = c.key_limit ? c.key_limit : 1ull << 32;
  const int lane = lane_id();
  uint64_t diff = 0;
  bool down = false, out = false;
  // a wave reads kStatRounds x 64 consecutive rows at a time, all its loads in flight together;
  // only the first row's predecessor is a load of its own
  constexpr int kRows = kStatRounds * kWave;
  const uint64_t waves = (uint64_t)gridDim.x * kWavesPerBlock;
  with_rows(c, c.in64, [&](auto load) {
    const uint64_t k0 = load(0);
    for (uint64_t r0 = ((uint64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave) * kRows;
         r0 < c.n; r0 += waves * kRows) {
      uint64_t k[kStatRounds];
      uint64_t edge = load(r0 ? r0 - 1 : 0);
#pragma unroll
      for (int j = 0; j < kStatRounds; ++j) {
        const uint64_t i = r0 + (uint64_t)j * kWave + lane;
        k[j] = load(i < c.n ? i : c.n - 1);  // the last row again: changes nothing
      }
      if (r0 == 0) edge = 0;
#pragma unroll
      for (int j = 0; j < kStatRounds; ++j) {
        uint64_t prev = __shfl_up(k[j], 1, kWave);
        if (lane == 0) prev = edge;
        edge = __shfl(k[j], kWave - 1, kWave);
        down |= (prev & sorted) > (k[j] & sorted);
        diff |= k[j] ^ k0;
        out |= rotl32((uint32_t)(k[j] >> 32), c.rot) >= limit;
      }
    }
  });
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) diff |= __shfl_xor(diff, d, kWave);
  __shared__ uint64_t wave_diff[kWavesPerBlock];
  if (lane == 0) wave_diff[threadIdx.x / kWave] = diff;
  const bool any_down = __syncthreads_or(down), any_out = __syncthreads_or(out);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 1; i < kWavesPerBlock; ++i) diff |= wave_diff[i];
    // one line updated by every workgroup serialises them (65 us for 1,024 of them): only what
    // is not there yet is written
    const volatile SortStats* now = st;
    const uint32_t flags = (any_down ? kDown : 0u) | (any_out ? kPast : 0u);
    if (diff & ~now->diff) atomicOr((unsigned long long*)&st->diff, (unsigned long long)diff);
    if (flags & ~now->flags) atomicOr(&st->flags, flags);
  }
}

// Digits to sort by, as a mask: the sorted ones in which rows differ (none when the rows are
// already in order).
__host__ __device__ __forceinline__ uint32_t active_digits(uint32_t mask, uint64_t diff,
                                                           uint32_t flags) {
  uint32_t m = 0;
  for (int d = 0; d < 8; ++d)
    if ((flags & kDown) && ((mask >> d) & 1u) && ((diff >> (8 * d)) & 0xffull)) m |= 1u << d;
  return m;
}

// Pass p of n sorts by bits [shift, shift + 8). The first pass is launched before the host knows
// n and shift (n = 0 here) and reads them from the statistics.
struct Pass {
  uint32_t p, n, shift;
};
__device__ __forceinline__ Pass settle(const ColSort& c, const SortStats* st, Pass a) {
  if (a.n == 0) {
    const uint32_t m = active_digits(c.mask, st->diff, st->flags);
    a.n = (uint32_t)__popc(m);
    a.shift = m ? 8u * (uint32_t)(__ffs((int)m) - 1) : 0u;
  }
  return a;
}

// Where pass p of n reads (the input composites, or nullptr: the columns) and writes: the last
// pass writes the output, the ones before it alternate so that no pass writes what it reads.
__device__ __forceinline__ const uint64_t* pass_src(const ColSort& c, uint32_t p, uint32_t n) {
  if (p == 0) return c.in64;
  return ((n - p) & 1u) ? c.buf_x : c.buf_y;
}

__global__ __launch_bounds__(kTileThreads) void sort_count_kernel(
    const ColSort c, const SortStats* __restrict__ st, Pass pass, uint32_t* __restrict__ hist,
    uint64_t tiles, uint64_t* __restrict__ mail) {
  if (mail && blockIdx.x == 0 && threadIdx.x == 0) {
    mail[0] = st->diff;
    mail[1] = st->flags;
  }
  pass = settle(c, st, pass);
  if (pass.n == 0) return;
  __shared__ uint32_t cnt[kDigits];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t shift = pass.shift;
  const uint64_t* src = pass_src(c, pass.p, pass.n);
  const uint64_t t0 = (uint64_t)blockIdx.x * kTile;
  const auto count = [&](uint64_t k) { atomicAdd(&cnt[(uint32_t)(k >> shift) & 0xffu], 1u); };
  with_rows(c, src, [&](auto load) {
    if (t0 + kTile <= c.n) {  // a whole tile: no predicates, every load in flight at once
      uint64_t k[kTileItems];
#pragma unroll
      for (int i = 0; i < kTileItems; ++i)
        k[i] = load(t0 + (uint64_t)i * kTileThreads + threadIdx.x);
#pragma unroll
      for (int i = 0; i < kTileItems; ++i) count(k[i]);
    } else {
      for (uint64_t idx = t0 + threadIdx.x; idx < c.n; idx += kTileThreads) count(load(idx));
    }
  });
  __syncthreads();
  hist[(uint64_t)threadIdx.x * tiles + blockIdx.x] = cnt[threadIdx.x];
}

// Workgroup d: rows with digit value d before every tile, and their total.
__global__ __launch_bounds__(kBlock) void sort_scan_kernel(const ColSort c,
                                                           const SortStats* __restrict__ st,
                                                           Pass pass,
                                                           uint32_t* __restrict__ hist,
                                                           uint64_t tiles,
                                                           uint32_t* __restrict__ totals) {
  if (settle(c, st, pass).n == 0) return;
  __shared__ uint32_t lds[4];
  constexpr int kItems = 8;
  uint32_t carry = 0;
  uint32_t* row = hist + (uint64_t)blockIdx.x * tiles;
  for (uint64_t t0 = 0; t0 < tiles; t0 += kBlock * kItems) {
    uint32_t v[kItems], sum = 0;
    const uint64_t i0 = t0 + (uint64_t)threadIdx.x * kItems;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      v[i] = i0 + i < tiles ? row[i0 + i] : 0u;
      sum += v[i];
    }
    uint32_t total;
    uint32_t off = carry + scan256(sum, lds, &total);
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      if (i0 + i < tiles) row[i0 + i] = off;
      off += v[i];
    }
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Stable scatter of one tile: wave w owns the tile's rows [w, w + 1) * kTile / waves, 64 per round,
// so (wave, round, lane) is the input order. The keys are placed in digit order in LDS and leave
// in that order: consecutive lanes write consecutive rows of a digit's run.
__global__ __launch_bounds__(kTileThreads) void sort_scatter_kernel(
    const ColSort c, const SortStats* __restrict__ st, Pass pass,
    const uint32_t* __restrict__ hist, uint64_t tiles, const uint32_t* __restrict__ totals) {
  constexpr int kPerWave = kTile / kTileWaves;
  __shared__ uint64_t tile[kTile];
  __shared__ uint32_t wrun[kTileWaves][kDigits];  // per-wave digit counts, then offsets
  __shared__ uint32_t goff[kDigits];              // output row of the digit's first slot, - slot
  __shared__ uint32_t scan_lds[4];
  pass = settle(c, st, pass);
  const int tid = threadIdx.x, w = tid / kWave, lane = lane_id();
  const uint64_t t0 = (uint64_t)blockIdx.x * kTile;
  const uint32_t tile_n = (uint32_t)(c.n - t0 < (uint64_t)kTile ? c.n - t0 : (uint64_t)kTile);
  if (pass.n == 0) {  // already in order: the rows go out as they are
    with_rows(c, c.in64, [&](auto load) {
      for (uint32_t j = tid; j < tile_n; j += kTileThreads) col_store(c, t0 + j, load(t0 + j));
    });
    return;
  }
  const uint32_t shift = pass.shift;
  const uint64_t* src = pass_src(c, pass.p, pass.n);
#pragma unroll
  for (int i = 0; i < kTileWaves; ++i) wrun[i][tid] = 0;
  __syncthreads();
  const uint64_t base = t0 + (uint64_t)w * kPerWave;
  uint64_t key[kTileItems];
  uint32_t rk[kTileItems];
  with_rows(c, src, [&](auto load) {
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
      const uint64_t idx = base + (uint64_t)r * kWave + lane;
      key[r] = load(idx < c.n ? idx : c.n - 1);
    }
  });
  const auto valid = [&](int r) { return base + (uint64_t)r * kWave + lane < c.n; };
  rank_rounds(key, rk, shift, wrun[w], valid);
  __syncthreads();
  {  // digit tid: tile offset, then each wave's first slot for it
    uint32_t cn[kTileWaves], tot = 0;
#pragma unroll
    for (int i = 0; i < kTileWaves; ++i) {
      cn[i] = wrun[i][tid];
      tot += cn[i];
    }
    uint32_t all;
    uint32_t q = scan256(tot, scan_lds, &all);
    // rows with a smaller digit + rows with this one in earlier tiles
    goff[tid] = scan256(totals[tid], scan_lds, &all) + hist[(uint64_t)tid * tiles + blockIdx.x] - q;
#pragma unroll
    for (int i = 0; i < kTileWaves; ++i) {
      wrun[i][tid] = q;
      q += cn[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kTileItems; ++r)
    if (valid(r)) {
      const uint32_t d = (uint32_t)(key[r] >> shift) & 0xffu;
      tile[wrun[w][d] + rk[r]] = key[r];
    }
  __syncthreads();
  const bool last = pass.p + 1 == pass.n;
  uint64_t* dst = ((pass.n - pass.p - 1) & 1u) ? c.buf_x : c.buf_y;
#pragma unroll
  for (int i = 0; i < kTileItems; ++i) {
    const uint32_t j = (uint32_t)i * kTileThreads + tid;
    if (j < tile_n) {
      const uint64_t k = tile[j];
      const uint32_t at = goff[(uint32_t)(k >> shift) & 0xffu] + j;
      if (last) col_store(c, at, k);
      else dst[at] = k;
    }
  }
}

hipError_t run_col_sort(const ColSort& c, void* temp, uint64_t* mail, hipEvent_t known,
                        hipStream_t s, ColSortFacts* facts) {
  *facts = ColSortFacts{};
  if (c.n == 0) return hipSuccess;
  if (c.n >= (1ull << 32)) return hipErrorInvalidValue;
  SortStats* st = (SortStats*)temp;
  uint32_t* totals = (uint32_t*)((char*)temp + kTotalsAt);
  uint32_t* hist = (uint32_t*)((char*)temp + kFixedBytes);
  const uint64_t tiles = tiles_of(c.n);
  hipError_t e = hipMemsetAsync(st, 0, sizeof(SortStats), s);
  if (e != hipSuccess) return e;
  const unsigned sgrid = (unsigned)std::min<uint64_t>(
      (c.n + kBlock * kStatRounds * 4 - 1) / (kBlock * kStatRounds * 4), 512);
  hipLaunchKernelGGL(sort_stats_kernel, dim3(sgrid), dim3(kBlock), 0, s, c, st);
  const auto count = [&](Pass a) {
    hipLaunchKernelGGL(sort_count_kernel, dim3((unsigned)tiles), dim3(kTileThreads), 0, s, c, st, a,
                       hist, tiles, a.p == 0 ? mail : nullptr);
  };
  const auto place = [&](Pass a) {
    hipLaunchKernelGGL(sort_scan_kernel, dim3(kDigits), dim3(kBlock), 0, s, c, st, a, hist, tiles,
                       totals);
    hipLaunchKernelGGL(sort_scatter_kernel, dim3((unsigned)tiles), dim3(kTileThreads), 0, s, c, st,
                       a, hist, tiles, totals);
  };
  count(Pass{0, 0, 0});
  e = hipEventRecord(known, s);
  if (e != hipSuccess) return e;
  place(Pass{0, 0, 0});
  e = hipEventSynchronize(known);
  if (e != hipSuccess) return e;
  const uint64_t diff = ((volatile uint64_t*)mail)[0], flags = ((volatile uint64_t*)mail)[1];
  facts->past_limit = (flags & kPast) != 0;
  const uint32_t active = active_digits(c.mask, diff, (uint32_t)flags);
  const uint32_t n = (uint32_t)__builtin_popcount(active);
  uint32_t p = 0;
  for (uint32_t d = 0; d < 8; ++d) {
    if (!((active >> d) & 1u)) continue;
    if (p > 0) {
      count(Pass{p, n, 8 * d});
      place(Pass{p, n, 8 * d});
    }
    ++p;
  }
  return hipGetLastError();
}

}  // namespace amj
