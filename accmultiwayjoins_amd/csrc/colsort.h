// Radix sort of rows from their columns (colsort.hip).
#pragma once

#include "amj_internal.h"

namespace amj {

// Stable sort of n rows (fewer than 2^32) by the digits of `mask` (bit d: bits [8d, 8d + 8)) of
// their composites (rotr32(key ^ flip, rot) << 32) | (val ^ 2^31), or of in64 when given. The
// result goes to out64, or (out64 == nullptr) back to columns out_key / out_val. buf_x and buf_y
// hold n composites each; with out64, buf_y must be out64. Inputs, buffers and outputs do not
// overlap otherwise.
struct ColSort {
  const int32_t* key = nullptr;
  const int32_t* val = nullptr;  // nullptr: one column
  const uint64_t* in64 = nullptr;
  uint64_t n = 0;
  uint32_t rot = 0;
  uint32_t flip = 0;
  uint32_t mask = 0xff;
  uint32_t key_limit = 0;  // != 0: report whether a key (unsigned) is at or past it
  uint64_t* buf_x = nullptr;
  uint64_t* buf_y = nullptr;
  uint64_t* out64 = nullptr;
  int32_t* out_key = nullptr;
  int32_t* out_val = nullptr;
};

// f(load), load(i) being row i's composite, with the kind of source (composites, two columns, one
// column) fixed inside: a test of it per row would keep the compiler from issuing the loads of
// several rows together.
template <typename F>
__device__ __forceinline__ void with_rows(const ColSort& c, const uint64_t* composites, F&& f) {
  const int32_t *key = c.key, *val = c.val;
  const uint32_t flip = c.flip, rot = c.rot;
  if (composites) {
    f([=](uint64_t i) { return composites[i]; });
  } else if (val) {
    f([=](uint64_t i) {
      return ((uint64_t)rotr32((uint32_t)key[i] ^ flip, rot) << 32) |
             ((uint32_t)val[i] ^ 0x80000000u);
    });
  } else {
    f([=](uint64_t i) { return (uint64_t)rotr32((uint32_t)key[i] ^ flip, rot) << 32; });
  }
}

__device__ __forceinline__ void col_store(const ColSort& c, uint64_t at, uint64_t k) {
  if (c.out64) {
    c.out64[at] = k;
    return;
  }
  c.out_key[at] = (int32_t)(rotl32((uint32_t)(k >> 32), c.rot) ^ c.flip);
  if (c.out_val) c.out_val[at] = (int32_t)((uint32_t)k ^ 0x80000000u);
}

// exclusive scan of one value per thread over the first 256 threads of a block (all
// threads of the block call it)
__device__ __forceinline__ uint32_t scan256(uint32_t v, uint32_t* lds, uint32_t* total) {
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const uint32_t incl = wave_incl_scan_u32(v);
  if (lane == kWave - 1 && w < 4) lds[w] = incl;
  __syncthreads();
  uint32_t off = 0, all = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t s = lds[i];
    if (i < w) off += s;
    all += s;
  }
  __syncthreads();
  *total = all;
  return off + incl - v;
}

// Rank of every key of a wave's rounds among the wave's keys of the same digit, in input order:
// a ballot multisplit per round and a running count per digit in `run` (the wave's own LDS
// row). Keys of rounds past the end are marked invalid by the caller's `valid`.
template <int ITEMS, typename Valid>
__device__ __forceinline__ void rank_rounds(const uint64_t (&key)[ITEMS], uint32_t (&rk)[ITEMS],
                                            uint32_t shift, uint32_t* run, const Valid& valid) {
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool ok = valid(r);
    const uint32_t d = (uint32_t)(key[r] >> shift) & 0xffu;
    uint64_t m = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t rank = mbcnt(m);
    __asm__ __volatile__("" ::: "memory");  // LDS ops of one wave complete in order
    const uint32_t before = run[d];
    rk[r] = before + rank;
    __asm__ __volatile__("" ::: "memory");
    if (ok && rank == 0) run[d] = before + (uint32_t)__popcll(m);
    __asm__ __volatile__("" ::: "memory");
  }
}

size_t col_sort_temp_bytes(uint64_t n);
struct ColSortFacts {
  bool past_limit = false;  // some key lies at or past key_limit
};
// Enqueues the sort on s. mail: two words of pinned host memory. The call waits for the statistics
// (event `known`, recorded inside) but not for the sort.
hipError_t run_col_sort(const ColSort& c, void* temp, uint64_t* mail, hipEvent_t known,
                        hipStream_t s, ColSortFacts* facts);

// The same for at most kHashSmallRows rows (hashbuild.hip): one launch, no buffers, no wait.
hipError_t launch_small_sort(const ColSort& c, hipStream_t s);

}  // namespace amj
