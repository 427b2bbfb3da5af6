// CPU test of a context's device blocks (blocks.h, compiled here unchanged) over a device of
// limited capacity: what the books say against what the device has given out, sizes, parking and
// its limits, allocations that need other contexts' parked blocks, and all of it from many
// threads. The program stops at its first failure (exit code 1).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <thread>

#include "blocks.h"

#define CHECK(c)                                                   \
  do {                                                             \
    if (!(c)) {                                                    \
      std::fprintf(stderr, "FAIL %s:%d: %s\n", __FILE__, __LINE__, #c); \
      std::exit(1);                                                \
    }                                                              \
  } while (0)

// Addresses only: nothing is allocated behind them.
struct Card {
  std::mutex mu;
  uint64_t capacity, used = 0, next = 1ull << 40;
  uint64_t gets = 0, drains = 0;
  std::map<uint64_t, uint64_t> live;  // address -> bytes
  explicit Card(uint64_t c) : capacity(c) {}
};
struct Device {
  Card* card;
  bool operator==(const Device& o) const { return card == o.card; }
  int get(size_t bytes, void** p) {
    std::lock_guard<std::mutex> g(card->mu);
    ++card->gets;
    if (card->used + bytes > card->capacity) return 2;
    card->used += bytes;
    card->live[card->next] = bytes;
    *p = (void*)card->next;
    card->next += (bytes + 4095) / 4096 * 4096 + 4096;
    return 0;
  }
  void put(void* p) {
    std::lock_guard<std::mutex> g(card->mu);
    const auto it = card->live.find((uint64_t)p);
    CHECK(it != card->live.end());  // given back once, by its address
    card->used -= it->second;
    card->live.erase(it);
  }
  void drain() {
    std::lock_guard<std::mutex> g(card->mu);
    ++card->drains;
  }
};
using amj::Blocks;
static const auto kNothing = [] {};

static uint64_t parked_sum(Blocks<Device>& b) { return b.parked_on_device(); }

static void sizes() {
  for (size_t n : {0ul, 1ul, 255ul, 4096ul, 4097ul, (1ul << 20) - 1, 1ul << 20, (1ul << 20) + 1,
                   62'804'220ul, 98'765'432ul, (512ul << 20) - 1, 512ul << 20}) {
    const size_t b = amj::block_bytes(n);
    CHECK(b >= n && b > 0);
    CHECK(b <= n + n / 16 + 4096);
    CHECK(amj::block_bytes(b) == b);
  }
  CHECK(amj::block_bytes((512ul << 20) + 1) == (512ul << 20) + 1);
}

static void books() {
  Card card(1ull << 40);
  {
    Blocks<Device> b(Device{&card});
    void* p[6];
    const size_t want[6] = {1, 62'804'220, 5000, 1ull << 33, 62'804'000, 0};
    for (int i = 0; i < 6; ++i) CHECK(b.take(want[i], &p[i], kNothing) == 0);
    CHECK(b.held() == card.used);  // what is held is what the device gave
    const uint64_t all = b.held();
    b.give(p[1], true);
    CHECK(parked_sum(b) == amj::block_bytes(want[1]) && card.used == all);
    CHECK(b.held() + parked_sum(b) == card.used);
    void* q = nullptr;
    const uint64_t gets = card.gets;
    CHECK(b.take(want[1] - 100, &q, kNothing) == 0);  // the same size class: the parked block
    CHECK(q == p[1] && card.gets == gets && parked_sum(b) == 0);
    b.give(p[3], true);  // too large to park
    CHECK(b.held() == card.used && parked_sum(b) == 0);
    b.give(p[0], false);
    CHECK(b.held() == card.used);
    CHECK(b.peak() == all);
    for (void* x : {p[2], q, p[4], p[5]}) b.give(x, true);
    CHECK(b.held() == 0 && parked_sum(b) == card.used);
  }
  CHECK(card.used == 0 && card.live.empty());  // the parked ones went back with the context
}

static void limits() {
  Card card(1ull << 40);
  Blocks<Device> b(Device{&card});
  std::vector<void*> p(400);
  for (auto& x : p) CHECK(b.take(100, &x, kNothing) == 0);
  for (auto& x : p) b.give(x, true);
  CHECK(parked_sum(b) == amj::kParkCount * 4096 && card.used == parked_sum(b));
  std::vector<void*> big(8);
  for (auto& x : big) CHECK(b.take(400ul << 20, &x, kNothing) == 0);
  for (auto& x : big) b.give(x, true);
  CHECK(parked_sum(b) <= amj::kParkTotal && card.used == parked_sum(b));
}

// An allocation that fails takes, in this order, what the context can do without, its own parked
// blocks and those of the other contexts on the device; blocks in use and other devices stay.
static void reclaim() {
  Card card(1000ul << 20), other(100ul << 20);
  Blocks<Device> a(Device{&card}), b(Device{&card}), far(Device{&other});
  void *pa = nullptr, *held = nullptr, *pf = nullptr, *p = nullptr;
  CHECK(a.take(300ul << 20, &pa, kNothing) == 0);
  CHECK(a.take(200ul << 20, &held, kNothing) == 0);
  CHECK(far.take(50ul << 20, &pf, kNothing) == 0);
  a.give(pa, true);
  far.give(pf, true);
  CHECK(b.parked_on_device() == 300ul << 20);
  int gave = 0;
  CHECK(b.take(400ul << 20, &p, [&] { ++gave; }) == 0);  // fits beside them
  CHECK(gave == 0 && b.parked_on_device() == 300ul << 20);
  b.give(p, false);
  CHECK(b.take(700ul << 20, &p, [&] { ++gave; }) == 0);  // needs a's parked block
  CHECK(gave == 1 && b.parked_on_device() == 0 && card.drains == 1);
  CHECK(a.held() == 200ul << 20 && card.used == a.held() + b.held());
  CHECK(far.parked_on_device() == 50ul << 20 && other.drains == 0);
  void* q = nullptr;
  CHECK(b.take(200ul << 20, &q, [&] { ++gave; }) == 2 && q == nullptr && gave == 2);
  CHECK(card.used == a.held() + b.held());
  // a block released through another context, or through none
  void* r = nullptr;
  CHECK(a.take(1000, &r, kNothing) == 0);
  b.give(r, true);
  CHECK(a.held() == 200ul << 20 && b.parked_on_device() == 0);
  CHECK(a.take(1000, &r, kNothing) == 0);
  Blocks<Device>::give_foreign(Device{&card}, r);
  CHECK(a.held() == 200ul << 20 && card.used == a.held() + b.held());
  a.give(held, false);
  b.give(p, false);
}

// Contexts on threads of their own, each also releasing and parking; the card is too small for all
// they would park, so they keep taking each other's parked blocks back.
static void threads() {
  Card card(64ul << 20);
  const int kThreads = 8;
  std::vector<std::unique_ptr<Blocks<Device>>> ctx;
  for (int t = 0; t < kThreads; ++t) ctx.emplace_back(new Blocks<Device>(Device{&card}));
  std::vector<std::thread> th;
  for (int t = 0; t < kThreads; ++t)
    th.emplace_back([&, t] {
      uint64_t s = 77 + t;
      std::vector<std::pair<void*, size_t>> mine;
      for (int i = 0; i < 3000; ++i) {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        if (mine.size() < 4 && (s >> 60) < 10) {
          const size_t n = (s >> 33) % (1u << 20) + 1;  // 8 threads x 4 x 1 MiB fit
          void* p = nullptr;
          CHECK(ctx[t]->take(n, &p, kNothing) == 0);
          {
            std::lock_guard<std::mutex> g(card.mu);
            CHECK(card.live.count((uint64_t)p) && card.live[(uint64_t)p] >= n);
          }
          mine.emplace_back(p, n);
        } else if (!mine.empty()) {
          const size_t k = (s >> 40) % mine.size();
          // now and then through a neighbour, as a program that mixes contexts up would
          ctx[(s >> 50) % 16 == 0 ? (t + 1) % kThreads : t]->give(mine[k].first, true);
          mine.erase(mine.begin() + (long)k);
        }
      }
      for (auto& m : mine) ctx[t]->give(m.first, true);
    });
  for (auto& t : th) t.join();
  for (auto& c : ctx) CHECK(c->held() == 0);
  CHECK(card.used == ctx[0]->parked_on_device());
  ctx.clear();
  CHECK(card.used == 0 && card.live.empty());
}

int main() {
  sizes();
  books();
  limits();
  reclaim();
  threads();
  std::printf("OK\n");
  return 0;
}
