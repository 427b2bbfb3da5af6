// Device blocks of a context: what it holds, and what it keeps parked for its next allocations.
// Plain C++ over a Device (get / put / drain), so that the CPU test compiles the same lines with a
// device of its own.
//
// Allocating and freeing device memory costs 1.2 us a pair up to 1 MB, 24 us from 4 MB on and 260 us
// for 256 MB, more when the memory has to be cleared first. So a released block of up to kParkBlock
// bytes is parked, for a later request of its size (the context's work is in stream order, so it is
// reused without a wait); at most kParkTotal bytes and kParkCount blocks, oldest out first. Parked
// blocks are given back when an allocation fails, in this context or in another one of the device.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace amj {

constexpr size_t kParkBlock = 512u << 20;
constexpr uint64_t kParkTotal = 2ull << 30;
constexpr size_t kParkCount = 256;

// Bytes held for a request: whole pages of 4 KiB, above 1 MiB whole fragments of 64 KiB, so that
// sizes that differ a little share parked blocks and no block is more than a sixteenth larger than
// asked for (plus a page). Blocks too large to be parked are taken as they are.
constexpr size_t block_bytes(size_t bytes) {
  const size_t g = bytes > (1u << 20) ? 64u << 10 : 4u << 10;
  return bytes > kParkBlock ? bytes : bytes == 0 ? g : (bytes + g - 1) / g * g;
}

// Device: copyable; operator== (the same device); int get(size_t bytes, void** p), 0 on success;
// put(void* p); drain(), which waits for all work on the device.
template <typename Device>
class Blocks {
 public:
  explicit Blocks(const Device& dev) : dev_(dev) {
    std::lock_guard<std::mutex> g(registry().mu);
    registry().all.push_back(this);
  }
  Blocks(const Blocks&) = delete;
  Blocks& operator=(const Blocks&) = delete;
  ~Blocks() {
    {
      std::lock_guard<std::mutex> g(registry().mu);
      auto& all = registry().all;
      all.erase(std::find(all.begin(), all.end(), this));
    }
    clear();
  }

  // A block of at least `bytes`. When the device has none, give_way() (what else the context can do
  // without), this context's parked blocks and then those of the device's other contexts go back
  // to it. 0, or what Device::get returned last.
  template <typename GiveWay>
  int take(size_t bytes, void** p, GiveWay&& give_way) {
    const size_t size = block_bytes(bytes);
    *p = nullptr;
    {
      std::lock_guard<std::mutex> g(mu_);
      for (size_t i = parked_.size(); i-- > 0;)
        if (parked_[i].second == size) {
          *p = parked_[i].first;
          parked_.erase(parked_.begin() + (std::ptrdiff_t)i);
          parked_bytes_ -= size;
          break;
        }
    }
    if (!*p) {
      int rc = dev_.get(size, p);
      if (rc != 0) {
        give_way();
        clear();
        rc = dev_.get(size, p);
      }
      // other threads may take what was given back, and park again
      while (rc != 0 && others_give_way()) rc = dev_.get(size, p);
      if (rc != 0) {
        *p = nullptr;
        return rc;
      }
    }
    std::lock_guard<std::mutex> g(mu_);
    sizes_[*p] = size;
    held_ += size;
    peak_ = std::max(peak_, held_);
    return 0;
  }

  // Releases a block: parked if it may be, else given back. Its size is the one it was taken with;
  // a block of another context leaves that one's books and goes back to the device.
  void give(void* p, bool park) {
    if (!p) return;
    std::vector<Block> out;
    {
      std::unique_lock<std::mutex> g(mu_);
      const auto it = sizes_.find(p);
      if (it == sizes_.end()) {
        g.unlock();
        give_foreign(dev_, p);
        return;
      }
      const size_t size = it->second;
      sizes_.erase(it);
      held_ -= size;
      if (!park || size > kParkBlock) {
        out.emplace_back(p, size);
      } else {
        parked_.emplace_back(p, size);
        parked_bytes_ += size;
        while (parked_bytes_ > kParkTotal || parked_.size() > kParkCount) {
          out.push_back(parked_.front());
          parked_bytes_ -= parked_.front().second;
          parked_.erase(parked_.begin());
        }
      }
    }
    for (const Block& b : out) dev_.put(b.first);
  }

  // Releases a block of whichever context holds it, or of one that is gone.
  static void give_foreign(const Device& dev, void* p) {
    {
      std::lock_guard<std::mutex> r(registry().mu);
      for (Blocks* b : registry().all) {
        std::lock_guard<std::mutex> g(b->mu_);
        const auto it = b->sizes_.find(p);
        if (it == b->sizes_.end()) continue;
        b->held_ -= it->second;
        b->sizes_.erase(it);
        break;
      }
    }
    Device d = dev;
    d.put(p);
  }

  // Gives all parked blocks back.
  void clear() {
    std::vector<Block> out;
    take_parked(&out);
    for (const Block& b : out) dev_.put(b.first);
  }

  uint64_t held() const {
    std::lock_guard<std::mutex> g(mu_);
    return held_;
  }
  uint64_t peak() const {
    std::lock_guard<std::mutex> g(mu_);
    return peak_;
  }
  // Bytes parked by all contexts of the device: there for an allocation that needs them.
  uint64_t parked_on_device() const {
    std::lock_guard<std::mutex> r(registry().mu);
    uint64_t n = 0;
    for (const Blocks* b : registry().all) {
      if (!(b->dev_ == dev_)) continue;
      std::lock_guard<std::mutex> g(b->mu_);
      n += b->parked_bytes_;
    }
    return n;
  }

 private:
  using Block = std::pair<void*, size_t>;
  struct Registry {
    std::mutex mu;  // before any context's own
    std::vector<Blocks*> all;
  };
  static Registry& registry() {
    static Registry* r = new Registry;  // contexts may end after static objects do
    return *r;
  }

  void take_parked(std::vector<Block>* out) {
    std::lock_guard<std::mutex> g(mu_);
    out->insert(out->end(), parked_.begin(), parked_.end());
    parked_.clear();
    parked_bytes_ = 0;
  }

  bool others_give_way() {
    std::lock_guard<std::mutex> r(registry().mu);
    std::vector<Block> out;
    for (Blocks* b : registry().all)
      if (b != this && b->dev_ == dev_) b->take_parked(&out);
    if (out.empty()) return false;
    dev_.drain();  // their contexts' streams may still be at work on them
    for (const Block& b : out) dev_.put(b.first);
    return true;
  }

  mutable std::mutex mu_;
  Device dev_;
  std::unordered_map<void*, size_t> sizes_;  // of the blocks held
  std::vector<Block> parked_;                // oldest first
  uint64_t held_ = 0, peak_ = 0, parked_bytes_ = 0;
};

}  // namespace amj
