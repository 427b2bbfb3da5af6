// Depth-first building blocks of the leapfrog triejoin shared by the unit engine (lftj.hip)
// and the persistent work-sharing engine (lftj_ws.hip): level 0 of a unit, the next 64
// candidates of a level checked against the other lists, and the sinks that receive the
// candidates that pass the last attribute (count, write at scanned positions, direct output).
#pragma once

#include "lftj_common.h"

namespace amj {

// Level 0 from root r of driver0 on every lane where `valid`.
template <int A, uint64_t SH = 0>
__device__ __forceinline__ void level0_at(const LPlan& P, uint64_t r, bool valid, LLv<A>& l) {
  sfor<0, A>([&](auto a) { l.b[a] = 0; });
  sfor<0, kR>([&](auto q) { l.lo[q] = 0u; l.hi[q] = 0u; });
  int32_t v = 0;
  const LRel& d = P.rel[P.driver0];
  if (valid) v = d.d0[r];
  bool ok = valid;
  if (valid) {
    if constexpr (SH != 0) ok = check_and_open_fixed<A, SH, 0>(P, v, -1, l);
    else ok = check_and_open(P, 0, v, -1, true, l);
  }
  l.b[0] = v;
  choose_driver<A, SH>(P, 1, ok, l);
  finish(l);
}

// The entries of `l` cut to candidates [c0, c1) of the flattened level.
template <int A>
__device__ __forceinline__ void restrict_range(LLv<A>& l, uint32_t c0, uint32_t c1) {
  const uint32_t b = l.excl > c0 ? l.excl : c0;
  const uint32_t e = l.excl + l.dlen < c1 ? l.excl + l.dlen : c1;
  const uint32_t n = e > b ? e - b : 0u;
  l.dptr = n ? l.dptr + (b - l.excl) : l.dptr;
  l.dlen = n;
  finish(l);
}

// Level 0 of a unit: P.rpu (0: 64) consecutive level-0 values of driver0, one per lane.
template <int A, uint64_t SH = 0>
__device__ __forceinline__ void level0(const LPlan& P, uint64_t unit, LLv<A>& l) {
  const uint32_t rpu = P.rpu ? P.rpu : (uint32_t)kWave;
  const uint32_t lane = (uint32_t)lane_id();
  const uint64_t r = unit * rpu + lane;
  level0_at<A, SH>(P, r, lane < rpu && r < P.roots, l);
}

// Result hash in two parts (hash_tuple: one round per pair of attributes): the first pair's round,
// which all results of one entry share, and the rest.
template <int A>
__device__ __forceinline__ uint64_t hash_first_pair(int32_t b0, int32_t b1) {
  return mix64((uint64_t)A ^ ((uint64_t)(uint32_t)b0 | ((uint64_t)(uint32_t)b1 << 32)));
}
template <int A>
__device__ __forceinline__ uint64_t hash_rest(uint64_t h, const int32_t (&b)[A]) {
  static_assert(A == 3 || A == 4, "one round after the first pair");
  uint64_t w = (uint32_t)b[2];
  if constexpr (A == 4) w |= (uint64_t)(uint32_t)b[3] << 32;
  return mix64(h ^ w);
}

// What happens to the candidates that pass the last attribute (`ok` per lane, bindings in b):
// counted, written at their scanned positions, or gathered for direct output. put() is the same
// with the hash of the first pair given (kHashes sinks only look at it).
struct CountSink {
  static constexpr bool kCounts = true;  // add() is enough: the bindings are not looked at
  static constexpr bool kHashes = false, kStores = false;
  uint64_t count = 0;
  __device__ __forceinline__ void add(uint32_t n) { count += n; }
  template <int A>
  __device__ __forceinline__ void operator()(bool ok, const int32_t (&)[A]) {
    count += (uint64_t)__popcll(__ballot(ok));
  }
  template <int A>
  __device__ __forceinline__ void put(bool ok, const int32_t (&b)[A], uint64_t) {
    (*this)(ok, b);
  }
};

// Count and checksum only (the work-sharing engine's passes without output).
template <bool HASH>
struct CountHashSink {
  static constexpr bool kCounts = !HASH, kHashes = HASH, kStores = false;
  uint64_t count = 0;
  __device__ __forceinline__ void add(uint32_t n) { count += n; }
  uint64_t csum = 0;  // per-lane checksum partial
  template <int A>
  __device__ __forceinline__ void operator()(bool ok, const int32_t (&b)[A]) {
    count += (uint64_t)__popcll(__ballot(ok));
    if (HASH && ok) {
      int32_t w[kMaxAttrs];
      sfor<0, kMaxAttrs>([&](auto a) { w[a] = (a < A) ? b[(a < A) ? (int)a : 0] : 0; });
      csum += hash_tuple(w, A);
    }
  }
  template <int A>
  __device__ __forceinline__ void put(bool ok, const int32_t (&b)[A], uint64_t h) {
    count += (uint64_t)__popcll(__ballot(ok));
    if (HASH && ok) csum += hash_rest<A>(h, b);
  }
};

template <int MODE>
struct WriteSink {
  static constexpr bool kCounts = false, kHashes = mode_hash<MODE>(), kStores = mode_mat<MODE>();
  LOut cols;
  uint64_t out_base;  // absolute row of the next result (uniform)
  uint64_t csum;      // per-lane checksum partial
  template <int A>
  __device__ __forceinline__ void operator()(bool ok, const int32_t (&b)[A]) {
    const uint64_t m = __ballot(ok);
    if (ok) {
      if (mode_hash<MODE>()) {
        int32_t w[kMaxAttrs];
        sfor<0, kMaxAttrs>([&](auto a) { w[a] = (a < A) ? b[(a < A) ? (int)a : 0] : 0; });
        csum += hash_tuple(w, A);
      }
      if (mode_mat<MODE>()) {
        const uint64_t pos = out_base + mbcnt(m);
        sfor<0, A>([&](auto a) { cols.c[a][pos] = b[a]; });
      }
    }
    out_base += (uint64_t)__popcll(m);
  }
  template <int A>
  __device__ __forceinline__ void put(bool ok, const int32_t (&b)[A], uint64_t h) {
    const uint64_t m = __ballot(ok);
    if (ok) {
      if (mode_hash<MODE>()) csum += hash_rest<A>(h, b);
      if (mode_mat<MODE>()) {
        const uint64_t pos = out_base + mbcnt(m);
        sfor<0, A>([&](auto a) { cols.c[a][pos] = b[a]; });
      }
    }
    out_base += (uint64_t)__popcll(m);
  }
};

// Direct output: results gather in a per-wave LDS buffer of kLftjDirectRows rows; rows at or
// past `capacity` are not written (the reserved total then tells the host to run again with a
// larger allocation).
//   * chunk = 0: one atomic reservation on the launch's row counter per full buffer.
//   * chunk > 0: rows are reserved `chunk` at a time (a multiple of kLftjDirectRows) and a wave
//     fills its chunk buffer by buffer, so the shared counter sees one update per `chunk` rows
//     instead of one per buffer (one counter updated by every wave serialises them: about 14 ns
//     per update on this device, which bounded a whole triangle pass). Only a wave's last chunk
//     is left partly unused; the wave records that tail (`tail_of`) and a fill-up pass moves the
//     rows found past the result count into the tails below it (launch_chunk_fill).
constexpr uint32_t kLftjDirectRows = 256;
typedef __attribute__((address_space(3))) int32_t lds_i32;

// The checksum is taken from the buffer when it is flushed, with every lane busy, rather than
// per result on the lanes whose candidate passed.
template <int A, bool HASH>
struct DirectSink {
  static constexpr bool kCounts = false, kHashes = false, kStores = true;  // hashes when it flushes
  LOut cols;
  uint64_t capacity;
  unsigned long long* rows;  // rows reserved by the whole launch
  lds_i32* buf;              // attribute a of row i at buf[a * kLftjDirectRows + i]
  uint32_t fill;             // rows held (uniform)
  uint64_t csum;
  uint32_t chunk = 0;        // rows per reservation (0: one reservation per buffer)
  uint64_t cur = ~0ull;      // first row of the wave's current chunk (~0: none yet)
  uint32_t used = 0;         // rows of the current chunk taken
  uint64_t count = 0;        // rows passed to the sink (uniform)

  __device__ __forceinline__ void flush() {
    if (fill == 0) return;
    // rows [0, na) of the buffer go to base_a + i, rows [na, fill) to base_b + i - na
    uint64_t base_a = 0, base_b = 0;
    uint32_t na = fill;
    if (chunk) {
      const uint32_t rem = cur == ~0ull ? 0u : chunk - used;
      na = fill < rem ? fill : rem;
      base_a = cur + used;
      if (fill > rem) {
        unsigned long long r0 = 0;
        if (lane_id() == 0)
          r0 = __hip_atomic_fetch_add(rows, (unsigned long long)chunk, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        base_b = uniform((uint64_t)r0);
        cur = base_b;
        used = fill - na;
      } else {
        used += fill;
      }
    } else {
      unsigned long long r0 = 0;
      if (lane_id() == 0)
        r0 = __hip_atomic_fetch_add(rows, (unsigned long long)fill, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
      base_a = uniform((uint64_t)r0);
    }
    count += fill;
    __asm__ __volatile__("" ::: "memory");  // LDS ops of one wave complete in order
    for (uint32_t i = (uint32_t)lane_id(); i < fill; i += kWave) {
      const uint64_t pos = i < na ? base_a + i : base_b + (i - na);
      int32_t w[kMaxAttrs];
      sfor<0, kMaxAttrs>([&](auto a) {
        if constexpr ((int)a < A) w[a] = buf[(int)a * kLftjDirectRows + i];
        else w[a] = 0;
      });
      if (HASH) csum += hash_tuple(w, A);
      if (pos < capacity) sfor<0, A>([&](auto a) { cols.c[a][pos] = w[a]; });
    }
    __asm__ __volatile__("" ::: "memory");
    fill = 0;
  }

  // Chunked, after the last flush: the unused tail of the wave's last chunk, recorded by lane 0
  // as tail[chunk index] when the chunk lies inside the allocation.
  __device__ __forceinline__ void tail_of(uint64_t* tail) const {
    if (chunk && cur != ~0ull && lane_id() == 0 && cur + chunk <= capacity)
      tail[cur / chunk] = chunk - used;
  }

  __device__ __forceinline__ void operator()(bool ok, const int32_t (&b)[A]) {
    const uint64_t m = __ballot(ok);
    const uint32_t n = (uint32_t)__popcll(m);
    if (n == 0) return;
    if (fill + n > kLftjDirectRows) flush();
    __asm__ __volatile__("" ::: "memory");
    if (ok) {
      const uint32_t slot = fill + mbcnt(m);
      sfor<0, A>([&](auto a) { buf[a * kLftjDirectRows + slot] = b[a]; });
    }
    __asm__ __volatile__("" ::: "memory");
    fill += n;
  }
  __device__ __forceinline__ void put(bool ok, const int32_t (&b)[A], uint64_t) { (*this)(ok, b); }
};

// Candidates [c, c + 64) of the flattened level `par` (those below `end` are valid) checked
// for attribute i: ch gets the parent's bindings and child ranges, b[i] = the candidate, and
// the ranges of the relations rooted at i opened. Returns whether the candidate passed.
template <int A, int i, uint64_t SH = 0>
__device__ __forceinline__ bool lchild(const LPlan& P, const LLv<A>& par, uint32_t c,
                                       uint32_t end, LLv<A>& ch) {
  const uint32_t g = c + (uint32_t)lane_id();
  const bool valid = g < end;
  const int p = (int)parent_of_slots(par.excl, par.dlen, c);
  const uint32_t k = g - (uint32_t)__shfl(par.excl, p, kWave);
  const int32_t* src = (const int32_t*)__shfl((uint64_t)par.dptr, p, kWave);
  const int drel = __shfl(par.drel, p, kWave);
  sfor<0, A>([&](auto a) { ch.b[a] = __shfl(par.b[a], p, kWave); });
  sfor<0, kR>([&](auto q) {
    ch.lo[q] = __shfl(par.lo[q], p, kWave);
    ch.hi[q] = __shfl(par.hi[q], p, kWave);
  });
  const int32_t v = valid ? ld_at<false>(src, k) : 0;
  bool ok = valid;
  if constexpr (SH != 0) {
    ok = ok && check_and_open_fixed<A, SH, i>(P, v, drel, ch);
  } else {
    const bool drel_root = P.child_mask[i] == 0u;
    ok = ok && check_and_open(P, i, v, drel, drel_root, ch);
  }
  ch.b[i] = v;
  return ok;
}

// Cooperative levels of the compiled shapes: entries whose lists are long enough are run by the
// whole wave, which keeps the values of one list in LDS and checks the other list's values
// against them; the rest go through the flattened enumeration.
constexpr uint32_t kCoopMinCands = 32;
// What a level reports as it goes: steps of 64 candidates or list values. The unit engine has no use
// for it; the work-sharing engine's idle waves take it as progress (ws_queue.h).
struct NoSteps {
  __device__ __forceinline__ void operator()(uint32_t) const {}
};
constexpr uint32_t kStageInts = 1024;  // values of the checked list, at most
// 4-clique pairs (descend_clique_pairs): the checked list of an entry, and the entry's
// intersection.
constexpr uint32_t kCliqueOther = 768;
// LDS words per wave: the kept list's table (or, in a list no table could be made of, its values),
// and the queue of results. 4-cliques have besides the entry's intersection and its table. Sized
// so that four workgroups (4-cliques: three) fit a CU.
constexpr uint32_t kTriTable = 2048, kFourTable = 1024, kPairTable = 1024;
constexpr uint32_t kQueue = 128;                               // results: a word and a byte each
constexpr uint32_t kQueueWords = kQueue + kQueue / 4;
template <uint64_t SH>
constexpr uint32_t stage_ints() {
  return SH == kShapeFour ? kFourTable + kCliqueOther + kPairTable + kQueueWords
                          : kTriTable + kQueueWords;
}
static_assert(kStageInts <= kTriTable && kCliqueOther <= kFourTable && kCliqueOther <= kPairTable,
              "a list fits its table's room");
static_assert(kStageInts <= kFourTable, "descend_last_fixed stages into the 4-clique's table");

__device__ __forceinline__ uint32_t readlane_u32(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int lane) {
  return (uint64_t)readlane_u32((uint32_t)v, lane) |
         ((uint64_t)readlane_u32((uint32_t)(v >> 32), lane) << 32);
}

// Are v[j] in the ascending run st[0, n) of LDS (n the same on every lane)? The K searches
// advance together, so K reads are in flight at every step; ok[j] is cleared for a miss. The
// position is kept as an LDS pointer, so a step is one add, one read, one compare and one
// select per search.
template <int K>
__device__ __forceinline__ void lds_has(const lds_i32* st, uint32_t n, const int32_t (&v)[K],
                                        bool (&ok)[K]) {
  if (n == 0) {
    sfor<0, K>([&](auto j) { ok[j] = false; });
    return;
  }
  const lds_i32* b[K];
  sfor<0, K>([&](auto j) { b[j] = st; });
  while (n > 1) {
    const uint32_t half = n >> 1;
    const lds_i32* c[K];
    int32_t x[K];
    sfor<0, K>([&](auto j) {
      c[j] = b[j] + half;
      x[j] = *c[j];
    });
    sfor<0, K>([&](auto j) { b[j] = x[j] <= v[j] ? c[j] : b[j]; });
    n -= half;
  }
  sfor<0, K>([&](auto j) { ok[j] = ok[j] && *b[j] == v[j]; });
}

// Chunks of 64 candidates a wave checks at once in the cooperative last level.
constexpr int kCoopChunks = 4;

// The values of an ascending list, kept in LDS for membership tests: a cuckoo table (every value in
// one of its two slots, so a test is two independent reads), at most 7/16 full; or, when the list
// is too long for the room or the insertion does not settle (values that share their slots), the
// list itself, searched.
//
// An empty slot s holds s ^ 1, which no test of that slot can match: the first hash of s ^ 1 is
// s ^ 1 (values below 2^11 hash to themselves), and kHashMul was chosen so that its second hash is
// not s either, for every slot of every table size from 64 to 2,048.
constexpr uint32_t kHashMul = 0x9ad2d5u;
struct LdsSet {
  lds_i32* t;          // table or list
  uint32_t n = 0;      // values
  uint32_t m4 = 0;     // byte mask of a slot's offset (0: t is the list)

  static __device__ __forceinline__ uint32_t mix(int32_t v) {
    return (uint32_t)v ^ ((uint32_t)v >> 11);
  }
  __device__ __forceinline__ uint32_t slot1(uint32_t x) const { return (x << 2) & m4; }
  __device__ __forceinline__ uint32_t slot2(uint32_t x) const {
    return (__umul24(x, kHashMul) >> 10) & m4;
  }
  __device__ __forceinline__ lds_i32* at(uint32_t off) const {
    return (lds_i32*)((__attribute__((address_space(3))) char*)t + off);
  }
  // load(i): value i of the list, i < n_values (n_values > 0); `room` words at t
  template <typename Load>
  __device__ __forceinline__ void fill(uint32_t n_values, uint32_t room, Load&& load) {
    const uint32_t lane = (uint32_t)lane_id();
    __asm__ __volatile__("" ::: "memory");  // LDS ops of one wave complete in order
    n = n_values;
    uint32_t words = (uint32_t)kWave;
    while (words < room && words < 4 * n_values) words <<= 1;
    bool settled = 16 * n_values <= 7 * words;
    if (settled) {
      m4 = (words - 1) << 2;
      for (uint32_t i = lane; i < words; i += kWave) t[i] = (int32_t)(i ^ 1u);
      __asm__ __volatile__("" ::: "memory");
      for (uint32_t j0 = 0; j0 < n_values && settled; j0 += kWave) {
        bool todo = j0 + lane < n_values;
        int32_t v = load(todo ? j0 + lane : n_values - 1);
        uint32_t off = slot1(mix(v));
        int left = 48;  // rounds of evictions
        for (; left && __ballot(todo); --left) {
          if (todo) {
            const int32_t old = __hip_atomic_exchange(at(off), v, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_WAVEFRONT);
            todo = (uint32_t)old != ((off >> 2) ^ 1u);
            v = old;
            const uint32_t x = mix(old), o1 = slot1(x);
            off = o1 == off ? slot2(x) : o1;
          }
        }
        settled = __ballot(todo) == 0ull;
      }
    }
    if (!settled) {
      m4 = 0;
      __asm__ __volatile__("" ::: "memory");
      for (uint32_t j = lane; j < n_values; j += kWave) t[j] = load(j);
    }
    __asm__ __volatile__("" ::: "memory");
  }
  // live[j] loses the lanes whose v[j] is not in the list
  template <int K>
  __device__ __forceinline__ void keep(const int32_t (&v)[K], uint64_t (&live)[K]) const {
    if (m4) {
      int32_t a[K], b[K];  // all reads in flight together
      sfor<0, K>([&](auto j) {
        const uint32_t x = mix(v[j]);
        a[j] = *at(slot1(x));
        b[j] = *at(slot2(x));
      });
      sfor<0, K>([&](auto j) { live[j] &= __ballot(a[j] == v[j]) | __ballot(b[j] == v[j]); });
    } else {
      bool ok[K];
      sfor<0, K>([&](auto j) { ok[j] = true; });
      lds_has<K>(t, n, v, ok);
      sfor<0, K>([&](auto j) { live[j] &= __ballot(ok[j]); });
    }
  }
};

// Results gathered to full waves, in the order they came: a ring of (value, tag < 64) pairs.
struct Hits {
  lds_i32* ring;
  uint32_t head = 0, n = 0;  // uniform

  __device__ __forceinline__ __attribute__((address_space(3))) uint8_t* tags() const {
    return (__attribute__((address_space(3))) uint8_t*)(ring + kQueue);
  }
  __device__ __forceinline__ void push(uint64_t m, int32_t v, int tag) {
    if (__builtin_amdgcn_inverse_ballot_w64(m)) {
      const uint32_t at = (head + n + mbcnt(m)) & (kQueue - 1);
      ring[at] = v;
      tags()[at] = (uint8_t)tag;
    }
    n += (uint32_t)__popcll(m);
  }
  // Takes the first min(n, 64): f(valid, value, tag).
  template <typename F>
  __device__ __forceinline__ void take(F&& f) {
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t k = n < (uint32_t)kWave ? n : (uint32_t)kWave;
    __asm__ __volatile__("" ::: "memory");  // LDS ops of one wave complete in order
    const uint32_t at = (head + lane) & (kQueue - 1);
    const int32_t v = ring[at];
    const int tag = (int)tags()[at] & (kWave - 1);
    head += k;
    n -= k;
    __asm__ __volatile__("" ::: "memory");
    f(lane < k, v, tag);
  }
};

// The lists of the entries in `m` (lane p's list: ptr, len > 0, in a child array with kTriePad
// readable values after its end), one after the other, kStream x 64 values at a time: enter(p)
// before an entry's values, then step(v, live, p), v[j] being the values of chunk j, live[j] its
// lanes that hold one (0: chunk not there). The next values, of the same list or the next entry's,
// are loaded before the current ones are taken; the loads have neither conditions nor address
// arithmetic per lane.
constexpr int kStream = 4;
static_assert(kStream * kWave <= (int)kTriePad, "a batch may be read past the end of a list");
template <typename Enter, typename Step>
__device__ __forceinline__ void stream_lists(uint64_t m, const int32_t* ptr, uint32_t len,
                                             Enter&& enter, Step&& step) {
  if (m == 0) return;
  constexpr uint32_t kTake = (uint32_t)(kStream * kWave);
  const uint32_t lane = (uint32_t)lane_id();
  const auto fetch = [&](const int32_t* q, int32_t (&v)[kStream]) {
    typedef __attribute__((address_space(1))) const char gchar;
    uint32_t off = lane * 4u;
    __asm__("" : "+v"(off));  // kept a 32-bit offset from the uniform q, not a 64-bit address
    const gchar* at = (const gchar*)q + off;
    sfor<0, kStream>([&](auto j) {
      v[j] = *(__attribute__((address_space(1))) const int32_t*)(at + (int)j * 4 * kWave);
    });
  };
  int p = __ffsll((unsigned long long)m) - 1;
  const int32_t* q = (const int32_t*)readlane_u64((uint64_t)ptr, p);
  uint32_t l = readlane_u32(len, p);
  int32_t v[kStream];
  fetch(q, v);
  for (;;) {
    m &= m - 1;
    const int pn = m ? __ffsll((unsigned long long)m) - 1 : p;
    const int32_t* qn = (const int32_t*)readlane_u64((uint64_t)ptr, pn);
    const uint32_t ln = readlane_u32(len, pn);
    enter(p);
    for (;;) {
      int32_t w[kStream];
      const bool more = l > kTake;
      q = more ? q + kTake : qn;
      fetch(q, w);
      uint64_t live[kStream];
      sfor<0, kStream>([&](auto j) { live[j] = __ballot(lane + (uint32_t)j * kWave < l); });
      step(v, live, p);
      sfor<0, kStream>([&](auto j) { v[j] = w[j]; });
      if (!more) break;
      l -= kTake;
    }
    if (!m) break;
    p = pn;
    l = ln;
  }
}

// Lists of this many values on average are streamed one by one, shorter ones flattened over the
// wave: a list pays for whole chunks of 64, a flattened chunk for finding every value's list.
constexpr uint32_t kStreamMean = 96;

// Which of an entry's two child lists is checked against and which is streamed. With lists free of
// duplicates that are whole (not cut to a window of candidates) the first relation's list is
// kept in LDS and the second one's streamed: consecutive entries share their first value, so
// the kept list and its table stay. Otherwise the candidates' own list is streamed, which is what
// decides how often a duplicate is produced.
template <int A>
struct PairLists {
  const int32_t *set, *str;
  uint32_t set_n, str_n;
  __device__ __forceinline__ PairLists(const LPlan& P, const LLv<A>& l, int ra, int rb) {
    const int32_t* pa = P.rel[ra].d1 + l.lo[ra];
    const int32_t* pb = P.rel[rb].d1 + l.lo[rb];
    const uint32_t na = l.hi[ra] - l.lo[ra], nb = l.hi[rb] - l.lo[rb];
    const bool drives_b = l.drel == rb;
    const bool whole = l.dlen == (drives_b ? nb : na);
    const bool stream_b = drives_b || (P.distinct && whole);
    set = stream_b ? pa : pb;
    set_n = stream_b ? na : nb;
    str = drives_b || !stream_b ? l.dptr : pb;
    str_n = drives_b || !stream_b ? l.dlen : nb;
  }
};

// Last attribute of a triangle (compiled shape kShapeTri): a2 in the children of a0 (relation 1)
// and of a1 (relation 2). Entries with at least kCoopMinCands candidates whose lists both fit the
// stage are run by the whole wave: the children of a0 stay in LDS (a table) while the children of
// every a1 are streamed past them, two independent LDS reads per value; the results (one value in
// eleven on R-MAT 22) are gathered to full waves. They come in entry order, ascending.
//
// Bound by the streamed loads (23.8 G values for R-MAT 22) and about 15 VALU instructions per 64 of
// them. The version before staged the longer list of every entry and searched the shorter one in
// it (26 G values staged, 11.6 G searched in 9 to 10 steps), and its sinks saw the one in six
// lanes that passed. R-MAT 22, count / write with checksum: 31.8 / 43.9 ms before, 27.6 / 35 ms now
// (880 M lines of 128 B fetched past the L2 per pass, 4.2 TB/s); R-MAT 20, count with checksum 5.6
// -> 4.6 ms.
template <int A, uint64_t SH, typename Sink, typename Steps>
__device__ __forceinline__ void descend_tri_last(const LPlan& P, const LLv<A>& par, Sink& sink,
                                                 lds_i32* stage, const Steps& steps) {
  static_assert(A == 3 && SH == kShapeTri, "triangle shape only");
  const uint32_t na = par.hi[1] - par.lo[1], nb = par.hi[2] - par.lo[2];
  const bool coop = par.dlen >= kCoopMinCands && (par.drel == 1 ? nb : na) <= kStageInts;
  {  // entries with few candidates (or a long list to check): flattened
    LLv<A> sm = par;
    sm.dlen = coop ? 0u : par.dlen;
    finish(sm);
    for (uint32_t c = 0; c < sm.T; c += (uint32_t)kWave) {
      LLv<A> ch;
      steps(1u);
      const bool ok = lchild<A, 2, SH>(P, sm, c, sm.T, ch);
      sink(ok, ch.b);
    }
  }
  const PairLists<A> pl(P, par, 1, 2);
  LdsSet set;
  set.t = stage;
  Hits hits;
  hits.ring = stage + kTriTable;
  const uint64_t h01 = Sink::kHashes ? hash_first_pair<A>(par.b[0], par.b[1]) : 0ull;
  const auto emit = [&]() {
    hits.take([&](bool ok, int32_t v, int p) {
      int32_t b[A] = {0, 0, v};
      if constexpr (Sink::kStores) {
        b[0] = __shfl(par.b[0], p, kWave);
        b[1] = __shfl(par.b[1], p, kWave);
      }
      sink.put(ok, b, Sink::kHashes ? __shfl(h01, p, kWave) : 0ull);
    });
  };
  uint64_t kept = 0;
  stream_lists(
      __ballot(coop), pl.str, pl.str_n,
      [&](int p) {
        const uint64_t src = readlane_u64((uint64_t)pl.set, p);
        const uint32_t n = readlane_u32(pl.set_n, p);
        steps(1u + readlane_u32(pl.str_n, p) / kWave);
        if (src == kept && n == set.n) return;
        kept = src;
        set.fill(n, kTriTable, [&](uint32_t i) { return ld_at<true>((const int32_t*)src, i); });
      },
      [&](const int32_t (&v)[kStream], uint64_t (&live)[kStream], int p) {
        set.keep(v, live);
        sfor<0, kStream>([&](auto j) {
          if constexpr (Sink::kCounts) {
            sink.add((uint32_t)__popcll(live[j]));
          } else if (live[j]) {
            hits.push(live[j], v[j], p);
            if (hits.n >= (uint32_t)kWave) emit();
          }
        });
      });
  while (hits.n) emit();
}

// The last attribute of a 4-clique outside the clique pairs. An entry whose driver list holds at
// least kCoopMinCands candidates and whose other child lists (every child list of the attribute
// but the driver's) hold at most kStageInts values together is run by the whole wave: the other
// lists are copied to the wave's LDS stage once, and each chunk of 64 candidates is checked
// there by binary searches of uniform length (one global load per candidate instead of a
// chain of dependent ones). The other entries go through the flattened enumeration.
template <int A, int I, uint64_t SH, typename Sink, typename Steps>
__device__ __forceinline__ void descend_last_fixed(const LPlan& P, const LLv<A>& par, Sink& sink,
                                                   lds_i32* stage, const Steps& steps) {
  constexpr uint32_t cm = (uint32_t)(SH >> (12 * I + 6)) & 63u;
  constexpr int nc = bit_count(cm);
  static_assert(nc >= 2, "the last attribute has a driver and at least one list to check");
  constexpr int no = nc - 1;
  constexpr int K = kCoopChunks;
  // this lane's other lists, as in check_and_open_fixed
  int di = 0;
  sfor<1, nc>([&](auto j) {
    if (par.drel == nth_bit(cm, (int)j)) di = (int)j;
  });
  const int32_t* optr[no];
  uint32_t olen[no];
  uint32_t total = 0;
  sfor<0, no>([&](auto k) {
    constexpr int ra = nth_bit(cm, (int)k), rb = nth_bit(cm, (int)k + 1);
    const bool next = (int)k >= di;
    const uint32_t lo = next ? par.lo[rb] : par.lo[ra];
    const uint32_t hi = next ? par.hi[rb] : par.hi[ra];
    optr[k] = (next ? P.rel[rb].d1 : P.rel[ra].d1) + lo;
    olen[k] = hi - lo;
    total += hi - lo;
  });
  const bool coop = par.dlen >= kCoopMinCands && total <= kStageInts;

  // entries with few candidates (or long other lists): flattened
  {
    LLv<A> sm = par;
    sm.dlen = coop ? 0u : par.dlen;
    finish(sm);
    for (uint32_t c = 0; c < sm.T; c += (uint32_t)kWave) {
      LLv<A> ch;
      steps(1u);
      const bool ok = lchild<A, I, SH>(P, sm, c, sm.T, ch);
      sink(ok, ch.b);
    }
  }

  // the others, one entry at a time; consecutive entries often check the same list (children
  // of one parent value), which then stays staged
  uint64_t m = __ballot(coop);
  const uint32_t lane = (uint32_t)lane_id();
  uint64_t staged[no];
  uint32_t soff[no], slen[no];
  sfor<0, no>([&](auto k) {
    staged[k] = 0ull;
    soff[k] = 0u;
    slen[k] = 0u;
  });
  while (m) {
    const int p = __ffsll((unsigned long long)m) - 1;
    m &= m - 1;
    const int32_t* dp = (const int32_t*)readlane_u64((uint64_t)par.dptr, p);
    const uint32_t dl = readlane_u32(par.dlen, p);
    steps(1u + dl / kWave);
    const int32_t* src[no];
    uint32_t n[no];
    bool same = true;
    sfor<0, no>([&](auto k) {
      src[k] = (const int32_t*)readlane_u64((uint64_t)optr[k], p);
      n[k] = readlane_u32(olen[k], p);
      same = same && (uint64_t)src[k] == staged[k] && n[k] == slen[k];
    });
    if (!same) {
      __asm__ __volatile__("" ::: "memory");  // earlier reads of the stage are done (in order)
      uint32_t at = 0;
      sfor<0, no>([&](auto k) {
        for (uint32_t j0 = 0; j0 < n[k]; j0 += 4u * kWave) {
          int32_t t[4];
          sfor<0, 4>([&](auto u) {
            const uint32_t j = j0 + (uint32_t)u * kWave + lane;
            t[u] = j < n[k] ? ld_at<false>(src[k], j) : 0;
          });
          sfor<0, 4>([&](auto u) {
            const uint32_t j = j0 + (uint32_t)u * kWave + lane;
            if (j < n[k]) stage[at + j] = t[u];
          });
        }
        staged[k] = (uint64_t)src[k];
        soff[k] = at;
        slen[k] = n[k];
        at += n[k];
      });
      __asm__ __volatile__("" ::: "memory");  // LDS ops of one wave complete in order
    }
    int32_t b[A];
    sfor<0, A>([&](auto a) {
      if constexpr ((int)a < I) b[a] = (int32_t)readlane_u32((uint32_t)par.b[a], p);
      else b[a] = 0;
    });
    for (uint32_t c = 0; c < dl; c += (uint32_t)(K * kWave)) {
      int32_t v[K];
      bool ok[K];
      sfor<0, K>([&](auto j) {
        const uint32_t g = c + (uint32_t)j * kWave + lane;
        ok[j] = g < dl;
        v[j] = ok[j] ? ld_at<false>(dp, g) : 0;
      });
      sfor<0, no>([&](auto k) { lds_has<K>(stage + soff[k], slen[k], v, ok); });
      sfor<0, K>([&](auto j) {
        if (c + (uint32_t)j * kWave < dl) {
          b[I] = v[j];
          sink(ok[j], b);
        }
      });
    }
  }
}

// Attributes 2 and 3 of a 4-clique (compiled shape kShapeFour) whose relations (0,2) and (0,3)
// are one trie, and (1,2) and (1,3) another. For an entry (a0, a1) the third attribute takes
// L = children(a0) ∩ children'(a1), and the fourth takes the same L intersected with the children
// of a2 in relation (2,3). An entry whose lists hold at most kCliqueOther values is run by the
// whole wave: L is formed once (the children of a1 streamed past those of a0, kept in LDS; the
// values found appended in order), L gets a table of its own, and every child of every a2 of L is
// one test in it (two LDS reads). The other entries take the generic path.
//
// Bound by issue and LDS latency: the table of L (up to 448 values) decides how many workgroups
// fit a CU; one of a quarter of the size, with a fourth workgroup per CU, was slower (R-MAT 18 dense
// cores have longer L: 72 ms against 44). Searching L instead, chunks flattened over the wave:
// R-MAT 18 / 20 62 / 298 ms (unit engine, count + checksum), now 44 / 174 ms.
template <int A, uint64_t SH, typename Sink, typename Steps>
__device__ __forceinline__ void descend_clique_pairs(const LPlan& P, const LLv<A>& par, Sink& sink,
                                                     lds_i32* stage, const Steps& steps) {
  static_assert(A == 4 && SH == kShapeFour, "4-clique shape only");
  constexpr int K = kCoopChunks;
  const uint32_t na = par.hi[1] - par.lo[1], nb = par.hi[3] - par.lo[3];
  const bool clique = par.dlen > 0 && na <= kCliqueOther && (par.drel == 1 ? nb : na) <= kCliqueOther;

  // entries with a long list to check: the generic levels
  {
    LLv<A> sm = par;
    sm.dlen = clique ? 0u : par.dlen;
    finish(sm);
    for (uint32_t c = 0; c < sm.T; c += (uint32_t)kWave) {
      LLv<A> ch;
      steps(1u);
      const bool ok = lchild<A, 2, SH>(P, sm, c, sm.T, ch);
      choose_driver<A, SH>(P, 3, ok, ch);
      finish(ch);
      if (ch.T) descend_last_fixed<A, 3, SH>(P, ch, sink, stage, steps);
    }
  }

  const PairLists<A> pl(P, par, 1, 3);
  LdsSet set, pair;  // the kept list; L
  set.t = stage;
  lds_i32* lst = stage + kFourTable;  // L, ascending
  pair.t = lst + kCliqueOther;
  Hits hits;
  hits.ring = pair.t + kPairTable;
  uint64_t kept = 0;
  uint64_t m = __ballot(clique);
  const uint32_t lane = (uint32_t)lane_id();
  const LRel& r5 = P.rel[5];
  while (m) {
    const int p = __ffsll((unsigned long long)m) - 1;
    m &= m - 1;
    const uint64_t src = readlane_u64((uint64_t)pl.set, p);
    const uint32_t n = readlane_u32(pl.set_n, p);
    steps(1u + readlane_u32(pl.str_n, p) / kWave);
    if (src != kept || n != set.n) {
      kept = src;
      set.fill(n, kFourTable, [&](uint32_t i) { return ld_at<true>((const int32_t*)src, i); });
    }
    // L = the streamed values found in the kept list, in order
    uint32_t nl = 0;
    stream_lists(
        1ull << p, pl.str, pl.str_n, [](int) {},
        [&](const int32_t (&v)[kStream], uint64_t (&live)[kStream], int) {
          set.keep(v, live);
          sfor<0, kStream>([&](auto j) {
            if (__builtin_amdgcn_inverse_ballot_w64(live[j])) lst[nl + mbcnt(live[j])] = v[j];
            nl += (uint32_t)__popcll(live[j]);
          });
        });
    __asm__ __volatile__("" ::: "memory");
    if (nl == 0) continue;
    int32_t b[A];
    b[0] = (int32_t)readlane_u32((uint32_t)par.b[0], p);
    b[1] = (int32_t)readlane_u32((uint32_t)par.b[1], p);
    const uint64_t h01 = Sink::kHashes ? hash_first_pair<A>(b[0], b[1]) : 0ull;
    pair.fill(nl, kPairTable, [&](uint32_t i) { return lst[i]; });
    // every a2 of L (64 at a time), its children in (2,3) checked against L: streamed list by
    // list, or, when the lists are short, flattened over the wave
    for (uint32_t g0 = 0; g0 < nl; g0 += (uint32_t)kWave) {
      const bool has = g0 + lane < nl;
      const int32_t a2 = has ? lst[g0 + lane] : 0;
      uint32_t clo = 0, chi = 0;
      const bool f = has && root_range<true>(r5, a2, clo, chi);
      const uint32_t clen = f ? chi - clo : 0u;
      const uint32_t incl = wave_scan_add_dpp(clen);
      const uint32_t T = lane63(incl);
      steps(1u + T / kWave);
      const uint64_t fm = __ballot(f);
      const auto emit = [&]() {
        hits.take([&](bool ok, int32_t v, int q) {
          b[2] = __shfl(a2, q, kWave);
          b[3] = v;
          sink.put(ok, b, h01);
        });
      };
      const auto found = [&](uint64_t hit, int32_t v, int q) {
        if constexpr (Sink::kCounts) {
          sink.add((uint32_t)__popcll(hit));
        } else if (hit) {
          hits.push(hit, v, q);
          if (hits.n >= (uint32_t)kWave) emit();
        }
      };
      if (T >= kStreamMean * (uint32_t)__popcll(fm)) {
        stream_lists(
            fm, r5.d1 + clo, clen, [](int) {},
            [&](const int32_t (&v)[kStream], uint64_t (&live)[kStream], int q) {
              pair.keep(v, live);
              sfor<0, kStream>([&](auto j) { found(live[j], v[j], q); });
            });
      } else {
        const uint32_t excl = incl - clen;
        for (uint32_t c = 0; c < T; c += (uint32_t)(K * kWave)) {
          int q[K];
          int32_t a3[K];
          uint64_t live[K];
          sfor<0, K>([&](auto j) {
            const uint32_t cj = c + (uint32_t)j * kWave;
            const uint32_t g = cj + lane;
            q[j] = (int)parent_of_slots(excl, clen, cj < T ? cj : 0u);
            const uint32_t k = g - (uint32_t)__shfl(excl, q[j], kWave);
            const uint32_t qlo = (uint32_t)__shfl(clo, q[j], kWave);
            live[j] = __ballot(g < T);
            a3[j] = ld_at<true>(r5.d1, g < T ? qlo + k : clo);
          });
          pair.keep(a3, live);
          sfor<0, K>([&](auto j) { found(live[j], a3[j], q[j]); });
        }
      }
      while (hits.n) emit();
    }
  }
}

template <int A, int i, uint64_t SH = 0, typename Sink, typename Steps = NoSteps>
__device__ __forceinline__ void descend(const LPlan& P, const LLv<A>& par, Sink& sink,
                                        lds_i32* stage = nullptr, const Steps& steps = {}) {
  if constexpr (SH == kShapeTri && i == A - 1) {
    descend_tri_last<A, SH>(P, par, sink, stage, steps);
  } else if constexpr (SH != 0 && i == A - 1) {
    descend_last_fixed<A, i, SH>(P, par, sink, stage, steps);
  } else if constexpr (SH == kShapeFour && i == 2) {
    // (0,2) and (0,3) one trie, (1,2) and (1,3) another: the clique pairs apply
    const bool same = P.rel[1].d1 == P.rel[2].d1 && P.rel[1].off == P.rel[2].off &&
                      P.rel[1].d0 == P.rel[2].d0 && P.rel[3].d1 == P.rel[4].d1 &&
                      P.rel[3].off == P.rel[4].off && P.rel[3].d0 == P.rel[4].d0;
    if (same) {
      descend_clique_pairs<A, SH>(P, par, sink, stage, steps);
      return;
    }
    for (uint32_t c = 0; c < par.T; c += (uint32_t)kWave) {
      LLv<A> ch;
      steps(1u);
      const bool ok = lchild<A, i, SH>(P, par, c, par.T, ch);
      choose_driver<A, SH>(P, i + 1, ok, ch);
      finish(ch);
      if (ch.T) descend<A, i + 1, SH>(P, ch, sink, stage, steps);
    }
  } else {
    for (uint32_t c = 0; c < par.T; c += (uint32_t)kWave) {
      LLv<A> ch;
      steps(1u);
      const bool ok = lchild<A, i, SH>(P, par, c, par.T, ch);
      if constexpr (i == A - 1) {
        sink(ok, ch.b);
      } else {
        choose_driver<A, SH>(P, i + 1, ok, ch);
        finish(ch);
        if (ch.T) descend<A, i + 1, SH>(P, ch, sink, stage, steps);
      }
    }
  }
}

}  // namespace amj
