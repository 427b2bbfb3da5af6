// Sorted CSR trie build for the leapfrog triejoin (ALFTJ).
//
// Reference: constructSortedTrie<D,C,2> (LFTJ-GPU/multi_partitioning.cuh:129-293) sorts the
// (col0, col1) pairs with two cub radix sorts, marks run boundaries (extractMasks, :104-121) and
// compacts the distinct level-0 values and their child offsets with segmented selects; the last
// level is the sorted col1. It keeps duplicate pairs (a duplicate edge is a duplicate child).
//
// Here: one stable radix sort of the columns (colsort.hip) orders the pairs, as the 64-bit
// composites ((col0 ^ 2^31) << 32 | (col1 ^ 2^31)), by (col0, col1) in signed order; duplicates are
// dropped (the triejoin intersects sets) and the level-0 values and offsets compacted in the same
// pass. When the level-0 values are small non-negative integers (vertex ids) a table
// value -> child range is added so that "is v a level-0 value, and what are its children" is one
// 8-byte load.
#include "amj_internal.h"
#include "colsort.h"
#include "lftj.h"
#include "runtime.h"

namespace amj {

// Sorted pairs are compacted a tile of kTrieTile at a time, in two launches around one scan of the
// tiles' counts: keep = first occurrence of a pair, head = first pair of its col0. (Flags, their
// scans and the compaction as separate passes over n took 1.5 ms for 64 M pairs and 17 launches;
// this reads the pairs twice: 0.4 ms and five.)
constexpr int kTrieItems = 8;
constexpr uint64_t kTrieTile = (uint64_t)kBlock * kTrieItems;

// Thread's kTrieItems consecutive pairs of its tile (k) and their flags, as bit masks.
__device__ __forceinline__ void trie_flags(const uint64_t* __restrict__ k, uint64_t n, uint64_t i0,
                                           uint64_t (&v)[kTrieItems], uint32_t& keep,
                                           uint32_t& head) {
  uint64_t prev = i0 && i0 < n ? k[i0 - 1] : 0ull;
  keep = head = 0;
#pragma unroll
  for (int j = 0; j < kTrieItems; ++j) v[j] = i0 + j < n ? k[i0 + j] : 0ull;
#pragma unroll
  for (int j = 0; j < kTrieItems; ++j) {
    if (i0 + j < n) {
      const bool first = i0 + j == 0;
      if (first || v[j] != prev) keep |= 1u << j;
      if (first || (v[j] >> 32) != (prev >> 32)) head |= 1u << j;
    }
    prev = v[j];
  }
}

// counts[tile] = pairs kept | heads << 32; counts[tiles] = 0; the first and last col0 to mail.
__global__ __launch_bounds__(kBlock) void trie_count_kernel(const uint64_t* __restrict__ k,
                                                            uint64_t n, uint64_t tiles,
                                                            uint64_t* __restrict__ counts,
                                                            uint32_t* __restrict__ max_run,
                                                            uint64_t* __restrict__ mail) {
  uint64_t v[kTrieItems];
  uint32_t keep, head;
  trie_flags(k, n, (uint64_t)blockIdx.x * kTrieTile + (uint64_t)threadIdx.x * kTrieItems, v, keep,
             head);
  const uint64_t sum = wave_sum_u64((uint64_t)__popc(keep) | ((uint64_t)__popc(head) << 32));
  __shared__ uint64_t part[kWavesPerBlock];
  if (lane_id() == 0) part[threadIdx.x / kWave] = sum;
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint64_t s = 0;
#pragma unroll
  for (int i = 0; i < kWavesPerBlock; ++i) s += part[i];
  counts[blockIdx.x] = s;
  if (blockIdx.x == 0) {
    counts[tiles] = 0;
    *max_run = 0;
    mail[0] = (k[0] >> 32) | (k[n - 1] & 0xffffffff00000000ull);
  }
}

// d1, d0 and off from the scanned counts (base[tiles] = the totals).
__global__ __launch_bounds__(kBlock) void trie_write_kernel(const uint64_t* __restrict__ k,
                                                            uint64_t n, uint64_t tiles,
                                                            const uint64_t* __restrict__ base,
                                                            int32_t* __restrict__ d0,
                                                            uint32_t* __restrict__ off,
                                                            int32_t* __restrict__ d1) {
  uint64_t v[kTrieItems];
  uint32_t keep, head;
  trie_flags(k, n, (uint64_t)blockIdx.x * kTrieTile + (uint64_t)threadIdx.x * kTrieItems, v, keep,
             head);
  const uint64_t mine = (uint64_t)__popc(keep) | ((uint64_t)__popc(head) << 32);
  const uint64_t incl = wave_incl_scan_u64(mine);
  __shared__ uint64_t part[kWavesPerBlock];
  const int w = threadIdx.x / kWave;
  if (lane_id() == kWave - 1) part[w] = incl;
  __syncthreads();
  uint64_t at = base[blockIdx.x] + incl - mine;
#pragma unroll
  for (int i = 0; i < kWavesPerBlock; ++i)
    if (i < w) at += part[i];
  uint32_t p = (uint32_t)at, q = (uint32_t)(at >> 32);
#pragma unroll
  for (int j = 0; j < kTrieItems; ++j) {
    if ((head >> j) & 1u) {
      d0[q] = (int32_t)((uint32_t)(v[j] >> 32) ^ 0x80000000u);
      off[q++] = p;
    }
    if ((keep >> j) & 1u) d1[p++] = (int32_t)((uint32_t)v[j] ^ 0x80000000u);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0)
    off[(uint32_t)(base[tiles] >> 32)] = (uint32_t)base[tiles];
}

// The longest child run, and (vrange != nullptr) vrange[v] = child range of level-0 value v (the
// table is zeroed first: absent values keep the empty range [0, 0)); every level-0 value has at
// least one child.
__global__ __launch_bounds__(kBlock) void trie_ranges_kernel(const int32_t* __restrict__ d0,
                                                             const uint32_t* __restrict__ off,
                                                             uint32_t n0,
                                                             uint2* __restrict__ vrange,
                                                             uint32_t* __restrict__ max_run) {
  __shared__ uint32_t red[kWavesPerBlock];
  uint32_t m = 0;
  for (uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x; j < n0;
       j += (uint64_t)gridDim.x * kBlock) {
    const uint32_t lo = off[j], hi = off[j + 1];
    m = max(m, hi - lo);
    if (vrange) vrange[(uint32_t)d0[j]] = make_uint2(lo, hi);
  }
#pragma unroll
  for (int d = kWave / 2; d >= 1; d >>= 1) m = max(m, (uint32_t)__shfl_xor(m, d, kWave));
  if (lane_id() == 0) red[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 1; i < kWavesPerBlock; ++i) m = max(m, red[i]);
    if (m > *(volatile uint32_t*)max_run) atomicMax(max_run, m);
  }
}

static unsigned grid_for(uint64_t n) {
  uint64_t g = (n + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  return g ? (unsigned)g : 1u;
}

// Longest child run, optional value -> child range table, timing and the device view. Expects d0,
// off, d1, n0 and n1 set, lo_v and hi_v the first and last level-0 value, *mr (device) zeroed and
// ev[0] recorded at the start of the build.
static int finish_trie(amj_ctx_t* ctx, TrieDev* out, int32_t lo_v, int32_t hi_v, uint32_t* mr) {
  hipStream_t s = ctx->stream;
  const uint32_t n0 = out->n0;
  ctx->mail[MAIL_TRIE] = 0;
  if (n0) {
    // value -> child range table when level-0 values are small non-negative integers
    const uint64_t span = (uint64_t)(uint32_t)hi_v + 1;
    if (lo_v >= 0 && span <= std::max<uint64_t>(4ull * n0, 1ull << 20)) {
      AMJ_TRY(dmalloc(ctx, (void**)&out->vrange, span * 8));
      out->vrange_n = (uint32_t)span;
      AMJ_HIP_TRY(ctx, hipMemsetAsync(out->vrange, 0, span * 8, s));
    }
    hipLaunchKernelGGL(trie_ranges_kernel, dim3(std::min(grid_for(n0), 1024u)), dim3(kBlock), 0, s,
                       (const int32_t*)out->d0, (const uint32_t*)out->off, n0, out->vrange, mr);
    AMJ_HIP_TRY(ctx, hipMemcpyAsync(ctx->mail + MAIL_TRIE, mr, 4, hipMemcpyDeviceToHost, s));
  }
  AMJ_HIP_TRY(ctx, hipEventRecord(ctx->ev[1], s));
  AMJ_HIP_TRY(ctx, hipEventSynchronize(ctx->ev[1]));
  out->build_ms = elapsed_ms(ctx->ev[0], ctx->ev[1]);
  out->max_run = (uint32_t)mail_word(ctx, MAIL_TRIE);
  out->view = LRel{out->d0, out->off, out->d1, out->vrange, n0, out->vrange_n};
  return AMJ_OK;
}

int build_trie(amj_ctx_t* ctx, const int32_t* c0, const int32_t* c1, uint64_t n,
               TrieDev* out) {
  *out = TrieDev{};
  if (n >= (1ull << 32)) {
    set_error(ctx, AMJ_ERR_ARG, "trie build: relations must have fewer than 2^32 rows");
    return AMJ_ERR_ARG;
  }
  hipStream_t s = ctx->stream;
  out->distinct = true;  // duplicate pairs are dropped
  AMJ_HIP_TRY(ctx, hipEventRecord(ctx->ev[0], s));
  void* mr = nullptr;
  AMJ_TRY(scratch(ctx, SLOT_FLAG, 256, &mr));
  if (n == 0) {
    AMJ_TRY(dmalloc(ctx, (void**)&out->off, 4));
    AMJ_HIP_TRY(ctx, hipMemsetAsync(out->off, 0, 4, s));
    return finish_trie(ctx, out, 0, 0, (uint32_t*)mr);
  }
  const uint64_t tiles = (n + kTrieTile - 1) / kTrieTile;
  void *alt = nullptr, *keys = nullptr, *tmp = nullptr, *base = nullptr, *stmp = nullptr;
  AMJ_TRY(scratch(ctx, SLOT_SORT_KEYS, n * 8, &keys));
  AMJ_TRY(scratch(ctx, SLOT_TRIE0, (tiles + 1) * 8, &base));
  AMJ_TRY(scratch(ctx, SLOT_SCAN_TEMP, scan_temp_elems(tiles + 1) * 8, &stmp));
  ColSort c;
  c.key = c0;
  c.val = c1;
  c.n = n;
  c.flip = 0x80000000u;  // signed order
  c.mask = 0xffu;
  c.buf_y = c.out64 = (uint64_t*)keys;
  if (n <= kHashSmallRows) {
    AMJ_HIP_TRY(ctx, launch_small_sort(c, s));
  } else {
    AMJ_TRY(scratch(ctx, SLOT_SORT_ALT, n * 8, &alt));
    AMJ_TRY(scratch(ctx, SLOT_SORT_TEMP, col_sort_temp_bytes(n), &tmp));
    c.buf_x = (uint64_t*)alt;
    ColSortFacts facts;
    AMJ_HIP_TRY(ctx, run_col_sort(c, tmp, ctx->mail + MAIL_SORT, ctx->ev[6], s, &facts));
  }
  hipLaunchKernelGGL(trie_count_kernel, dim3((unsigned)tiles), dim3(kBlock), 0, s,
                     (const uint64_t*)keys, n, tiles, (uint64_t*)base, (uint32_t*)mr,
                     ctx->mail + MAIL_TRIE + 1);
  AMJ_HIP_TRY(ctx, exclusive_scan_u64((const uint64_t*)base, (uint64_t*)base, tiles + 1,
                                      (uint64_t*)stmp, s, ctx->mail + MAIL_TRIE));
  AMJ_HIP_TRY(ctx, hipStreamSynchronize(s));
  const uint64_t totals = mail_word(ctx, MAIL_TRIE), ends = mail_word(ctx, MAIL_TRIE + 1);
  const uint32_t m = (uint32_t)totals, n0 = (uint32_t)(totals >> 32);
  AMJ_TRY(dmalloc(ctx, (void**)&out->d1, ((uint64_t)m + kTriePad) * 4));
  out->n1 = m;
  AMJ_TRY(dmalloc(ctx, (void**)&out->d0, (uint64_t)n0 * 4));
  out->n0 = n0;
  AMJ_TRY(dmalloc(ctx, (void**)&out->off, ((uint64_t)n0 + 1) * 4));
  hipLaunchKernelGGL(trie_write_kernel, dim3((unsigned)tiles), dim3(kBlock), 0, s,
                     (const uint64_t*)keys, n, tiles, (const uint64_t*)base, out->d0, out->off,
                     out->d1);
  return finish_trie(ctx, out, (int32_t)((uint32_t)ends ^ 0x80000000u),
                     (int32_t)((uint32_t)(ends >> 32) ^ 0x80000000u), (uint32_t*)mr);
}

// Host CSR (e.g. a deserialised .tr file) -> device trie. Level 0 must be strictly increasing
// and every child run sorted (duplicate children are kept, as in the reference's tries).
int trie_from_host(amj_ctx_t* ctx, uint64_t n0, const int32_t* d0, const uint64_t* off,
                   uint64_t n1, const int32_t* d1, TrieDev* out) {
  *out = TrieDev{};
  if (n0 >= (1ull << 32) || n1 >= (1ull << 32)) {
    set_error(ctx, AMJ_ERR_ARG, "trie levels must hold fewer than 2^32 values");
    return AMJ_ERR_ARG;
  }
  if (off[0] != 0 || off[n0] != n1) {
    set_error(ctx, AMJ_ERR_ARG, "trie offsets must start at 0 and end at the child count");
    return AMJ_ERR_ARG;
  }
  std::vector<uint32_t> off32(n0 + 1);
  out->distinct = true;
  for (uint64_t j = 0; j < n0; ++j) {
    if (off[j + 1] < off[j] || (j > 0 && d0[j] <= d0[j - 1])) {
      set_error(ctx, AMJ_ERR_ARG, "trie level 0 must be strictly increasing with monotone offsets");
      return AMJ_ERR_ARG;
    }
    for (uint64_t k = off[j] + 1; k < off[j + 1]; ++k)
      if (d1[k] < d1[k - 1]) {
        set_error(ctx, AMJ_ERR_ARG, "trie child lists must be sorted");
        return AMJ_ERR_ARG;
      } else if (d1[k] == d1[k - 1]) {
        out->distinct = false;
      }
    off32[j] = (uint32_t)off[j];
  }
  off32[n0] = (uint32_t)n1;
  hipStream_t s = ctx->stream;
  AMJ_HIP_TRY(ctx, hipEventRecord(ctx->ev[0], s));
  AMJ_TRY(dmalloc(ctx, (void**)&out->d0, n0 * 4));
  out->n0 = (uint32_t)n0;
  AMJ_TRY(dmalloc(ctx, (void**)&out->off, (n0 + 1) * 4));
  AMJ_TRY(dmalloc(ctx, (void**)&out->d1, (n1 + kTriePad) * 4));
  out->n1 = (uint32_t)n1;
  if (n0) AMJ_HIP_TRY(ctx, hipMemcpyAsync(out->d0, d0, n0 * 4, hipMemcpyHostToDevice, s));
  if (n1) AMJ_HIP_TRY(ctx, hipMemcpyAsync(out->d1, d1, n1 * 4, hipMemcpyHostToDevice, s));
  AMJ_HIP_TRY(ctx, hipMemcpyAsync(out->off, off32.data(), (n0 + 1) * 4, hipMemcpyHostToDevice, s));
  void* mr = nullptr;
  AMJ_TRY(scratch(ctx, SLOT_FLAG, 256, &mr));
  AMJ_HIP_TRY(ctx, hipMemsetAsync(mr, 0, 4, s));
  AMJ_HIP_TRY(ctx, hipStreamSynchronize(s));
  return finish_trie(ctx, out, n0 ? d0[0] : 0, n0 ? d0[n0 - 1] : 0, (uint32_t*)mr);
}

void free_trie(amj_ctx_t* ctx, TrieDev* t) {
  if (!t) return;
  if (ctx) (void)hipStreamSynchronize(ctx->stream);
  dfree(ctx, t->d0);
  dfree(ctx, t->off);
  dfree(ctx, t->d1);
  dfree(ctx, t->vrange);
  *t = TrieDev{};
}

}  // namespace amj
