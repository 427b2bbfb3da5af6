// Work-sharing substrate of the persistent engines: the AMHJ probe (dynamic.hip) and the
// leapfrog triejoin (lftj_ws.hip) run the same protocol over their own task records.
//
// Reference: TaskBook (MHJ-GPU/TaskBook.cuh:13-109) appends tasks with atomicAdd, GCQueue
// (common-utils/cuda/GCQueue.cuh:30-107) hands them out through CAS on tagged slots, and
// CBarrier (MHJ-GPU/CBarrier.cuh:9-46) ends the kernel when every warp is idle; none of them
// checks capacity. Here:
//   * persistent waves claim units (64 probe rows / some roots) from counters in guided chunks;
//   * task slots are reserved with one fetch-add on the queue tail, clamped to the capacity
//     (requests past the end get nothing, and the wave then keeps its work);
//   * a task record is published by its own ready flag (release store after the record), and
//     the taker acquires it; every control-block counter is otherwise relaxed;
//   * a wave leaves when no unit is left, no published task is unclaimed and no wave holds
//     claimed work; every wait is bounded by a wall-clock limit without progress (error flag,
//     never a hang), and working waves report progress as they go.
#pragma once

#include "amj_internal.h"
#include "ws_split.h"

namespace amj {

// Control block of one launch (zeroed by the host). Updates of one cache line serialise across
// the device (tens of ns each), so what is updated often has a line of its own, and units are
// claimed from kUnitShards counters (ws_split.h; a wave starts with the shard of its workgroup's
// XCD and goes on to the others). Count of a 1 M-row chain (15,625
// units): 1.25 ms with one counter, 0.85 with eight.
static_assert(kUnitShards == kXcds, "one claim counter per XCD");
struct alignas(128) WsShard {
  unsigned long long next;  // units of the shard claimed
};
struct alignas(128) WsCtl {
  WsShard shard[kUnitShards];
  unsigned long long q_tail;     // task slots reserved (may pass cap: clamp on read)
  unsigned long long q_head;     // task slots claimed
  alignas(128) unsigned long long out_rows;  // output rows reserved (the results, plus unused
                                             // chunk tails)
  alignas(128) unsigned long long progress;  // tasks completed, plus heartbeats
  unsigned int busy;             // waves holding units or a task
  unsigned int flags;            // 1: a wait hit the time limit
  alignas(128) unsigned long long count;  // results
  unsigned long long csum;       // checksum, sum of the waves' partials mod 2^64
  unsigned long long pushed;     // tasks published
};

constexpr uint32_t kFlagSpin = 1u;

struct WsArgs {
  WsCtl* ctl;
  uint32_t* tasks;       // cap records of the engine's record size
  uint32_t* ready;       // cap flags
  uint64_t cap;          // task slots
  uint64_t split;        // children per task (multiple of 64); 0 disables sharing
  uint64_t units;        // units to claim
  uint64_t out_cap;      // output rows available
  uint64_t stall_ticks;  // wall-clock ticks without progress before a wave gives up
  uint64_t max_claim;    // most units claimed at once (0: kMaxClaim)
};

// Per-wave sharing state.
struct WsWave {
  bool qfull;      // the queue has no room left in this launch: stop asking
  uint32_t iters;  // frontier steps taken (uniform), for the heartbeat
};

// Every access to the control block is relaxed: an acquire at agent scope invalidates the
// CU's vector caches, and idle waves polling with acquires (or workers finishing chunks with
// acquire-release updates) evicted the data the working waves on the same CU were reading.
// No data is published through these counters: a task record is published by its own flag,
// and a wave that leaves early on a stale view only gives up parallelism.
__device__ __forceinline__ unsigned long long ld_rlx(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned int ld_rlx(const unsigned int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T add_relaxed(T* p, T v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wave-uniform result of an atomic done by lane 0.
__device__ __forceinline__ uint64_t lane0_u64(uint64_t v) {
  return uniform(__shfl(v, 0, kWave));
}

// n (uniform) steps of a working wave; every kBeatSteps steps it reports progress. A launch without
// a control block (the size samples) only counts.
__device__ __forceinline__ void ws_step(const WsArgs& A, WsWave& W, uint32_t n = 1u) {
  const bool beat = ws_beat(W.iters, n);
  W.iters += n;
  if (beat && A.ctl && lane_id() == 0) add_relaxed(&A.ctl->progress, 1ull);
}

// Reserve up to k task slots with one fetch-add; returns the first slot, the number granted in
// *got, and sets *full once the queue has no room left.
__device__ __forceinline__ uint64_t reserve_tasks(const WsArgs& A, uint64_t k, uint64_t* got,
                                                  bool* full) {
  uint64_t first = 0, n = 0, f = 0;
  if (lane_id() == 0) {
    const unsigned long long tl = add_relaxed(&A.ctl->q_tail, (unsigned long long)k);
    n = ws_granted(tl, k, A.cap);
    first = n ? tl : 0;
    f = tl + k >= A.cap ? 1 : 0;
  }
  *got = lane0_u64(n);
  *full = lane0_u64(f) != 0;
  return lane0_u64(first);
}

// Task slots published or being published: q_tail clamped to the queue's capacity.
__device__ __forceinline__ unsigned long long queue_end(const WsArgs& A) {
  const unsigned long long tl = ld_rlx(&A.ctl->q_tail);
  return tl < A.cap ? tl : A.cap;
}

// Flag of a written record: the record is visible device-wide before its flag.
__device__ __forceinline__ void publish_task(const WsArgs& A, uint64_t slot) {
  __threadfence();
  if (lane_id() == 0)
    __hip_atomic_store(&A.ready[slot], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// Claim a published task; -1: none available, -2: its record never became ready.
__device__ __forceinline__ int64_t try_pop(const WsArgs& A) {
  int64_t r = -1;
  if (lane_id() == 0) {
    unsigned long long h = ld_rlx(&A.ctl->q_head);
    const unsigned long long tl = queue_end(A);
    if (h < tl && __hip_atomic_compare_exchange_strong(&A.ctl->q_head, &h, h + 1,
                                                       __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT)) {
      r = (int64_t)h;
      const uint64_t t0 = wall_clock64();
      while (__hip_atomic_load(&A.ready[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
        if (wall_clock64() - t0 > A.stall_ticks) {
          __hip_atomic_fetch_or(&A.ctl->flags, kFlagSpin, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
          r = -2;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
  }
  r = (int64_t)lane0_u64((uint64_t)r);
  if (r >= 0)  // every lane acquires the record (its flag is set by now)
    (void)__hip_atomic_load(&A.ready[r], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
  return r;
}

// The persistent loop of a wave: claim units in guided chunks and run them
// (run_units(first, end, step)), then take tasks (run_task(slot)) until the launch has drained.
//
// A claim is one update of one counter. A wave counts as busy from its first claim until it finds
// no work, not per claim, and reports progress from its heartbeat (ws_step) and per task, not per
// claim; running out of work is seen in busy (one more update per wave cost 0.25 ms of the 2.5 that
// counting 20 M probe rows takes). With a busy, a progress and a claim update per claim,
// quarter-size claims down to one unit, and all three counters in one line, that count (312,500
// units, fan-out 1) took 9.9 ms, of which the lookups are 1.2.
template <typename RunUnits, typename RunTask>
__device__ __forceinline__ void ws_serve(const WsArgs& A, RunUnits&& run_units,
                                         RunTask&& run_task) {
  uint64_t seen = ~0ull, since = 0;  // progress counter last seen, and when it last moved
  bool units_left = true, working = false;
  uint32_t shard = blockIdx.x % kUnitShards;  // workgroup b runs on XCD b % 8
  int naps = 1;
  const auto work = [&](bool on) {  // only kept for the waits for tasks
    if (A.split && on != working && lane_id() == 0) add_relaxed(&A.ctl->busy, on ? 1u : ~0u);
    working = on;
  };
  for (;;) {
    if (units_left) {
      uint64_t u = 0, n = 0;
      uint32_t tried = 0;
      for (; tried < kUnitShards; ++tried) {
        const uint64_t size = ws_shard_units(A.units, shard);
        if (lane_id() == 0) {
          unsigned long long* next = &A.ctl->shard[shard].next;
          const unsigned long long at = ld_rlx(next);
          if (at < size) {
            const uint64_t k = ws_claim(A.units, size, at, (uint64_t)gridDim.x * kWavesPerBlock,
                                        A.max_claim);
            u = add_relaxed(next, (unsigned long long)k);
            n = ws_granted(u, k, size);
          }
        }
        n = lane0_u64(n);
        if (n) break;
        shard = (shard + 1) % kUnitShards;  // this one is used up, and stays so
      }
      if (n) {
        work(true);
        const uint64_t first = ws_unit_of_shard(lane0_u64(u), shard);
        run_units(first, first + n * kUnitShards, kUnitShards);
        continue;
      }
      units_left = false;
    }
    if (A.split == 0) break;  // without sharing there are no tasks to wait for
    const int64_t slot = try_pop(A);
    if (slot >= 0) {
      work(true);
      run_task((uint64_t)slot);
      if (lane_id() == 0) add_relaxed(&A.ctl->progress, 1ull);
      naps = 1;
      continue;
    }
    work(false);
    if (slot == -2) break;
    uint32_t done = 0;
    if (lane_id() == 0)
      done = (ld_rlx(&A.ctl->busy) == 0u && ld_rlx(&A.ctl->q_head) >= queue_end(A)) ? 1u : 0u;
    if (uniform(__shfl(done, 0, kWave))) break;
    // no work here while other waves hold some: give up only if nothing moves for long
    // (a wave that runs out of work moves busy)
    const uint64_t prog = lane0_u64(
        lane_id() == 0 ? ws_moved(ld_rlx(&A.ctl->progress), ld_rlx(&A.ctl->busy)) : 0ull);
    const uint64_t now = wall_clock64();
    if (prog != seen) {
      seen = prog;
      since = now;
    } else if (now - since > A.stall_ticks) {
      if (lane_id() == 0)
        __hip_atomic_fetch_or(&A.ctl->flags, kFlagSpin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
    // idle waves look again after one, two, four and then eight naps of 64 x 64 cycles (about 2 us
    // each), so that thousands of them leave the counters to the waves that work
    for (int i = 0; i < naps; ++i) __builtin_amdgcn_s_sleep(64);
    naps = naps < 8 ? 2 * naps : 8;
  }
}

// Count and checksum of a wave added to the control block when it leaves.
__device__ __forceinline__ void ws_accumulate(const WsArgs& A, uint64_t count, uint64_t csum) {
  const uint64_t cs = wave_sum_u64(csum);
  if (lane_id() == 0) {
    add_relaxed(&A.ctl->count, (unsigned long long)count);
    add_relaxed(&A.ctl->csum, (unsigned long long)cs);
  }
}

}  // namespace amj
