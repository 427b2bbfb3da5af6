// CPU model of the work-sharing protocol of the persistent engines (ws_queue.h), restated with
// C++ atomics on many host threads, plus a check of the range and claim arithmetic both GPU
// engines share (ws_split.h, compiled here unchanged).
//
// The reference's substrate (TaskBook.cuh:13-109 task append, GCQueue.cuh:30-107 tagged CAS
// queue, CBarrier.cuh:9-46 idle barrier) has no capacity check; the protocol modelled here
// claims units from several counters (every worker starts at its own and goes on to the others),
// reserves task slots with a clamped fetch-add, publishes each record with a release store of its
// own flag, claims it with a CAS on the head, and ends when no unit is left, no published task is
// unclaimed and nobody holds work, with every wait bounded. A worker counts as busy from its first
// claim until it finds no work; progress is reported from its steps and per task, and a waiting
// worker also sees others start and run out of work.
//
// A "unit" u owns W(u) children (heavily skewed); a worker walks a range 64 children at a
// time and, when more than split + 64 are left, shares the tail as tasks, exactly as
// ws_ldescend / dyn_descend do. Every child must be visited exactly once, every record read
// only after its flag, every worker must leave, and a record whose flag never comes must end
// in the error flag, not a hang. The program stops at its first failure (exit code 1).
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "ws_split.h"

using namespace amj;

#define CHECK(c, ...)                                          \
  do {                                                         \
    if (!(c)) {                                                \
      std::fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); \
      std::fprintf(stderr, __VA_ARGS__);                       \
      std::fprintf(stderr, "\n");                              \
      std::exit(1);                                            \
    }                                                          \
  } while (0)

static uint64_t mix(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// ---- 1. range arithmetic ----------------------------------------------------------------
static void check_split_math() {
  uint64_t cases = 0;
  for (uint64_t split = 64; split <= 512; split += 64)
    for (uint64_t c = 0; c <= 640; c += 64)
      for (uint64_t c1 = c; c1 <= c + 4 * 1024 + 70; ++c1) {
        if (!ws_should_split(c, c1, split)) {
          CHECK(c1 - c <= split + 64, "no split with %llu left", (unsigned long long)(c1 - c));
          continue;
        }
        const uint64_t k = ws_pieces(c, c1, split);
        CHECK(k >= 1, "no pieces");
        for (uint64_t got = 0; got <= k; ++got) {
          // kept [c, keep_end) and the published pieces must tile [c, c1) in order
          const uint64_t keep_end = ws_keep_end(c, c1, split, k, got);
          CHECK(keep_end >= c + split && keep_end <= c1, "keep_end out of range");
          CHECK(got == 0 || keep_end < c1, "a published piece is empty");
          uint64_t at = keep_end;
          for (uint64_t j = 0; j < got; ++j) {
            uint64_t p0 = 0, p1 = 0;
            ws_piece(c, c1, split, k, got, j, &p0, &p1);
            CHECK(p0 == at, "piece %llu starts at %llu, expected %llu", (unsigned long long)j,
                  (unsigned long long)p0, (unsigned long long)at);
            CHECK(p1 > p0 && p1 - p0 <= split && p1 <= c1, "bad piece [%llu,%llu)",
                  (unsigned long long)p0, (unsigned long long)p1);
            CHECK(p0 % 64 == c % 64, "piece not aligned with the walk");
            at = p1;
          }
          CHECK(at == (got ? c1 : keep_end), "pieces do not end at c1");
          if (got == 0) CHECK(keep_end == c1, "nothing published but the range shrank");
          ++cases;
        }
      }
  for (uint64_t cap = 1; cap <= 64; ++cap)
    for (uint64_t tail = 0; tail <= 80; ++tail)
      for (uint64_t want = 1; want <= 20; ++want) {
        const uint64_t n = ws_granted(tail, want, cap);
        CHECK(n <= want, "granted more than asked");
        CHECK(tail + n <= cap || n == 0, "granted past the capacity");
        CHECK(tail >= cap || n == std::min(want, cap - tail), "granted less than room");
      }
  std::printf("split arithmetic: %llu cases ok\n", (unsigned long long)cases);
}

// ---- 2. claim arithmetic ----------------------------------------------------------------
// Shards and claims give every unit once, whatever the number of units, waves and the cap.
static void check_claim_math() {
  uint64_t cases = 0;
  for (uint64_t units = 0; units <= 5 * kUnitShards + 1; ++units) {
    uint64_t sum = 0;
    std::vector<int> seen(units, 0);
    for (uint32_t s = 0; s < kUnitShards; ++s) {
      const uint64_t size = ws_shard_units(units, s);
      sum += size;
      for (uint64_t k = 0; k < size; ++k) {
        const uint64_t u = ws_unit_of_shard(k, s);
        CHECK(u < units && u % kUnitShards == s, "unit %llu of shard %u", (unsigned long long)u, s);
        ++seen[u];
      }
    }
    CHECK(sum == units, "shards hold %llu of %llu units", (unsigned long long)sum,
          (unsigned long long)units);
    for (int n : seen) CHECK(n == 1, "a unit in %d shards", n);
  }
  for (uint64_t units : {1ull, 7ull, 9ull, 63ull, 64ull, 100ull, 255ull, 256ull, 5000ull, 312500ull})
    for (uint64_t waves : {1ull, 4ull, 16ull, 4096ull})
      for (uint64_t cap : {0ull, 1ull, 2ull, 3ull, 64ull})
        for (uint32_t s = 0; s < kUnitShards; ++s) {
          const uint64_t size = ws_shard_units(units, s);
          uint64_t at = 0, got = 0;  // one worker after the other, as the counter orders them
          while (at < size) {
            const uint64_t k = ws_claim(units, size, at, waves, cap);
            CHECK(k >= 1 && k <= (cap ? cap : kMaxClaim), "claim of %llu", (unsigned long long)k);
            CHECK(units < kManyUnits * waves || (cap && cap < kMinClaim) || k >= kMinClaim,
                  "claim of %llu with many units per wave", (unsigned long long)k);
            got += ws_granted(at, k, size);
            at += k;
            ++cases;
          }
          CHECK(got == size, "claims gave %llu of %llu units", (unsigned long long)got,
                (unsigned long long)size);
          CHECK(ws_granted(at, 5, size) == 0, "granted past the shard");
        }
  // reports: one per kBeatSteps steps, however the steps come
  uint32_t steps = 0, beats = 0;
  for (uint32_t i = 0; steps < 100 * kBeatSteps; ++i) {
    const uint32_t n = i % 97 + 1;
    beats += ws_beat(steps, n) ? 1 : 0;
    steps += n;
  }
  CHECK(beats == steps / kBeatSteps, "%u reports in %u steps", beats, steps);
  CHECK(ws_beat(kBeatSteps - 1, 1) && !ws_beat(kBeatSteps, kBeatSteps - 1), "report early or late");
  std::printf("claim arithmetic: %llu claims ok\n", (unsigned long long)cases);
}

// ---- 3. the protocol ------------------------------------------------------------------------
struct Ctl {
  std::atomic<uint64_t> shard[kUnitShards] = {};
  std::atomic<uint64_t> q_tail{0}, q_head{0}, pushed{0}, progress{0};
  std::atomic<uint32_t> busy{0}, flags{0};
};

struct Task {
  uint64_t unit, c0, c1;  // the record: which unit's children [c0, c1)
};

struct Model {
  uint64_t units, split, cap, stall_ns;
  uint64_t max_claim = 0;  // WsArgs::max_claim
  int workers;
  bool withhold_one;  // a worker reserves a slot and never publishes it (the stuck case)
  uint32_t step_weight = 1;  // steps counted for 64 children
  uint64_t step_us = 0;      // time they take
  std::vector<uint64_t> width;          // children per unit
  std::vector<uint64_t> first;          // offset of a unit's children in `visits`
  std::vector<std::atomic<uint32_t>> visits;
  std::vector<std::atomic<uint32_t>> unit_runs;
  std::vector<Task> tasks;
  std::vector<std::atomic<uint32_t>> ready;
  Ctl ctl;
  std::atomic<uint64_t> withheld{0};

  Model(uint64_t u, uint64_t sp, uint64_t cp, int w, uint64_t seed, bool withhold)
      : units(u), split(sp), cap(cp), stall_ns(2'000'000'000ull), workers(w),
        withhold_one(withhold), width(u), first(u + 1), tasks(cp), ready(cp) {
    uint64_t total = 0;
    for (uint64_t i = 0; i < u; ++i) {
      const uint64_t r = mix(seed ^ i);
      // skew: most units small, a few hubs with tens of thousands of children
      width[i] = (r % 100 < 3) ? 20000 + r % 40000 : r % 200;
      first[i] = total;
      total += width[i];
    }
    first[u] = total;
    visits = std::vector<std::atomic<uint32_t>>(total);
    unit_runs = std::vector<std::atomic<uint32_t>>(u);
  }

  static uint64_t now_ns() {
    return (uint64_t)std::chrono::duration_cast<std::chrono::nanoseconds>(
               std::chrono::steady_clock::now().time_since_epoch())
        .count();
  }

  // reserve_tasks: one fetch-add, clamped
  uint64_t reserve(uint64_t k, uint64_t* got, bool* full) {
    const uint64_t tl = ctl.q_tail.fetch_add(k, std::memory_order_relaxed);
    *got = ws_granted(tl, k, cap);
    *full = tl + k >= cap;
    return *got ? tl : 0;
  }
  uint64_t queue_end() const {
    const uint64_t tl = ctl.q_tail.load(std::memory_order_relaxed);
    return tl < cap ? tl : cap;
  }

  // ws_ldescend over one unit's children [c0, c1)
  struct Worker {
    bool qfull = false;
    uint32_t iters = 0;
  };
  void walk(uint64_t unit, uint64_t c0, uint64_t c1, Worker& w) {
    uint64_t end = c1;
    bool& qfull = w.qfull;
    for (uint64_t c = c0; c < end; c += 64) {
      // ws_step
      const bool beat = step_weight && ws_beat(w.iters, step_weight);
      w.iters += step_weight;
      if (beat) ctl.progress.fetch_add(1, std::memory_order_relaxed);
      if (step_us) std::this_thread::sleep_for(std::chrono::microseconds(step_us));
      if (!qfull && ws_should_split(c, end, split)) {
        const uint64_t k = ws_pieces(c, end, split);
        uint64_t got = 0;
        bool full = false;
        const uint64_t slot = reserve(k, &got, &full);
        if (full) qfull = true;
        if (got) {
          for (uint64_t j = 0; j < got; ++j) {
            uint64_t p0 = 0, p1 = 0;
            ws_piece(c, end, split, k, got, j, &p0, &p1);
            CHECK(slot + j < cap, "slot %llu past capacity", (unsigned long long)(slot + j));
            tasks[slot + j] = Task{unit, p0, p1};
            if (withhold_one && withheld.exchange(1) == 0) continue;  // never published
            ready[slot + j].store(1, std::memory_order_release);
          }
          ctl.pushed.fetch_add(got, std::memory_order_relaxed);
          end = ws_keep_end(c, end, split, k, got);
        }
      }
      const uint64_t stop = std::min(c + 64, end);
      for (uint64_t g = c; g < stop; ++g) visits[first[unit] + g].fetch_add(1);
    }
  }

  // try_pop: -1 none, -2 the record never became ready
  int64_t try_pop() {
    uint64_t h = ctl.q_head.load(std::memory_order_relaxed);
    const uint64_t tl = queue_end();
    if (h < tl && ctl.q_head.compare_exchange_strong(h, h + 1, std::memory_order_relaxed)) {
      const uint64_t t0 = now_ns();
      while (ready[h].load(std::memory_order_relaxed) == 0) {
        if (now_ns() - t0 > stall_ns) {
          ctl.flags.fetch_or(1, std::memory_order_relaxed);
          return -2;
        }
        std::this_thread::yield();
      }
      (void)ready[h].load(std::memory_order_acquire);
      return (int64_t)h;
    }
    return -1;
  }

  // ws_serve of worker number id
  void serve(int id) {
    Worker w;
    uint64_t seen = ~0ull, since = 0;
    bool units_left = true, working = false;
    uint32_t shard = (uint32_t)id % kUnitShards;
    const auto work = [&](bool on) {
      if (split && on != working) ctl.busy.fetch_add(on ? 1u : ~0u, std::memory_order_relaxed);
      working = on;
    };
    for (;;) {
      if (units_left) {
        uint64_t u = 0, n = 0;
        for (uint32_t tried = 0; tried < kUnitShards; ++tried) {
          const uint64_t size = ws_shard_units(units, shard);
          const uint64_t at = ctl.shard[shard].load(std::memory_order_relaxed);
          if (at < size) {
            const uint64_t k = ws_claim(units, size, at, (uint64_t)workers, max_claim);
            u = ctl.shard[shard].fetch_add(k, std::memory_order_relaxed);
            n = ws_granted(u, k, size);
          }
          if (n) break;
          shard = (shard + 1) % kUnitShards;
        }
        if (n) {
          work(true);
          for (uint64_t k = u; k < u + n; ++k) {
            const uint64_t v = ws_unit_of_shard(k, shard);
            CHECK(v < units, "unit %llu of %llu", (unsigned long long)v, (unsigned long long)units);
            unit_runs[v].fetch_add(1, std::memory_order_relaxed);
            walk(v, 0, width[v], w);
          }
          continue;
        }
        units_left = false;
      }
      if (split == 0) break;
      const int64_t slot = try_pop();
      if (slot >= 0) {
        work(true);
        const Task t = tasks[(uint64_t)slot];
        CHECK(t.unit < units && t.c0 < t.c1 && t.c1 <= width[t.unit], "bad task record");
        walk(t.unit, t.c0, t.c1, w);
        ctl.progress.fetch_add(1, std::memory_order_relaxed);
        continue;
      }
      work(false);
      if (slot == -2) break;
      if (ctl.busy.load(std::memory_order_relaxed) == 0 &&
          ctl.q_head.load(std::memory_order_relaxed) >= queue_end())
        break;
      const uint64_t prog = ws_moved(ctl.progress.load(std::memory_order_relaxed),
                                     ctl.busy.load(std::memory_order_relaxed));
      const uint64_t now = now_ns();
      if (prog != seen) {
        seen = prog;
        since = now;
      } else if (now - since > stall_ns) {
        ctl.flags.fetch_or(1, std::memory_order_relaxed);
        break;
      }
      std::this_thread::yield();
    }
    CHECK(!working || split == 0, "a worker left while it counted as busy");
  }

  // runs the workers; returns the error flag; every worker must have left
  uint32_t run() {
    std::vector<std::thread> th;
    for (int w = 0; w < workers; ++w) th.emplace_back([this, w] { serve(w); });
    for (auto& t : th) t.join();
    return ctl.flags.load();
  }
};

static void run_case(uint64_t units, uint64_t split, uint64_t cap, int workers, uint64_t seed,
                     uint64_t max_claim = 0) {
  Model m(units, split, cap, workers, seed, false);
  m.max_claim = max_claim;
  const uint32_t flags = m.run();
  CHECK(flags == 0, "error flag raised (units %llu split %llu cap %llu workers %d)",
        (unsigned long long)units, (unsigned long long)split, (unsigned long long)cap, workers);
  for (size_t i = 0; i < m.visits.size(); ++i)
    CHECK(m.visits[i].load() == 1, "child %zu visited %u times (split %llu cap %llu)", i,
          m.visits[i].load(), (unsigned long long)split, (unsigned long long)cap);
  for (uint64_t u = 0; u < units; ++u)
    CHECK(m.unit_runs[u].load() == 1, "unit %llu claimed %u times", (unsigned long long)u,
          m.unit_runs[u].load());
  CHECK(m.ctl.busy.load() == 0, "busy ended at %u", m.ctl.busy.load());
  CHECK(m.ctl.q_head.load() == std::min<uint64_t>(m.ctl.q_tail.load(), cap) || split == 0,
        "published tasks left unclaimed");
  std::printf("units %llu split %llu cap %llu workers %d: %zu children once each, %llu tasks\n",
              (unsigned long long)units, (unsigned long long)split, (unsigned long long)cap,
              workers, m.visits.size(), (unsigned long long)m.ctl.pushed.load());
}

// One unit that takes far longer than the stall limit while every other worker is idle: nothing is
// wrong as long as its worker's steps report, and the limit is what ends the waits if they do not.
static void run_slow_unit(bool reports) {
  Model m(3, 1 << 20, 16, 4, 13, false);
  for (uint64_t u = 0; u < 3; ++u) {
    m.width[u] = u == 1 ? 64 * 300 : 64;
    m.first[u + 1] = m.first[u] + m.width[u];
  }
  m.visits = std::vector<std::atomic<uint32_t>>(m.first[3]);
  m.step_us = 5000;             // 1.5 s in all
  m.stall_ns = 400'000'000ull;
  m.step_weight = reports ? kBeatSteps / 8 : 0;  // a report every 40 ms, or none
  const uint32_t flags = m.run();
  for (auto& v : m.visits) CHECK(v.load() == 1, "a child of a slow unit visited %u times", v.load());
  CHECK(flags == (reports ? 0u : 1u), "slow unit %s reports: flags %u", reports ? "with" : "without",
        flags);
  std::printf("slow unit %s reports: flag %u\n", reports ? "with" : "without", flags);
}

int main() {
  check_split_math();
  check_claim_math();
  const int hw = (int)std::max(2u, std::min(16u, std::thread::hardware_concurrency()));
  run_case(2000, 0, 16, hw, 1);        // no sharing
  run_case(2000, 1024, 8192, hw, 2);   // the ALFTJ default
  run_case(2000, 64, 8192, hw, 3);     // smallest tasks
  run_case(2000, 128, 7, hw, 4);       // queue fills: the rest is kept by its owner
  run_case(3000, 256, 1, 3, 5);        // one slot
  run_case(500, 64, 4096, 1, 6);       // one worker serves its own tasks
  run_case(4000, 192, 100000, 64, 7);  // many more workers than cores
  run_case(12000, 0, 16, hw, 9);        // many units per worker: claims of at least 4
  run_case(12000, 1024, 8192, hw, 10);  // ... with sharing
  run_case(12000, 0, 16, hw, 11, 2);    // claims capped below the minimum of 4
  run_case(12000, 256, 8192, hw, 12, 1);  // single-unit claims with sharing
  for (uint64_t u : {0, 1, 7, 8, 9, 25}) {  // few units: fewer than shards, than workers
    run_case(u, 0, 16, hw, 20 + u);
    run_case(u, 128, 64, hw, 60 + u);
  }
  run_slow_unit(true);
  run_slow_unit(false);
  // a reserved slot whose flag never comes: the taker gives up with the error flag
  Model m(200, 64, 4096, hw, 8, true);
  m.stall_ns = 200'000'000ull;
  const uint32_t flags = m.run();
  CHECK(m.withheld.load() == 1, "nothing was withheld");
  CHECK(flags == 1, "a missing record did not raise the error flag");
  std::printf("withheld record: every worker left, error flag raised\n");
  std::printf("OK\n");
  return 0;
}
