// CPU test of a context's device blocks (blocks.h, compiled here unchanged) over a device of
// limited capacity: what the books say against what the device has given out, sizes, parking and
// its limits. The program stops at its first failure (exit code 1).
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

static uint64_t parked_sum(Blocks<Device>& b) { return b.parked(); }

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

int main() {
  sizes();
  books();
  limits();
  std::printf("OK\n");
  return 0;
}
