// tmp_cache.hpp -- the blocks of memory that the library keeps for
// temporaries: which block a call gets, which are let go.  Host C++ only: the
// allocations and releases are the caller's functions.
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

namespace mph {

// Free blocks of at most kTmpKeepBytes, and kTmpKeepBlocks of them, are held
// a device, and as much again in pinned host memory.
constexpr size_t kTmpKeepBytes = (size_t)2 << 30;
constexpr size_t kTmpKeepBlocks = 48;

constexpr int kTmpHost = -1;  // "device" of pinned host memory
struct TmpBlock {
  void* p = nullptr;
  size_t bytes = 0;
  int device = kTmpHost;
};

class TmpCache {
 public:
  // sizes in steps of an eighth of their power of two, at least 4 KiB, so
  // that calls of like size share blocks
  static size_t rounded(size_t bytes) {
    size_t step = 4096;
    while (step * 16 <= bytes) step <<= 1;
    return (bytes + step - 1) / step * step;
  }

  // The smallest held block of the device from `bytes` up that is not much
  // larger, of equals the one given back last.
  bool take(int device, size_t bytes, TmpBlock* b) {
    std::lock_guard<std::mutex> lk(m_);
    size_t best = blocks_.size();
    for (size_t i = 0; i < blocks_.size(); i++) {
      const TmpBlock& f = blocks_[i];
      if (f.device == device && f.bytes >= bytes &&
          f.bytes <= std::max<size_t>(4 * bytes, 1 << 16) &&
          (best == blocks_.size() || f.bytes <= blocks_[best].bytes))
        best = i;
    }
    if (best == blocks_.size()) return false;
    *b = blocks_[best];
    blocks_.erase(blocks_.begin() + (std::ptrdiff_t)best);
    return true;
  }

  // Holds b.  Over a limit, the device's blocks that have lain longest are
  // released (a block that is over it alone, at once): were b turned away
  // instead, blocks of sizes no longer asked for would stay, and every later
  // call would allocate and free its own.
  template <typename Release>
  void give(const TmpBlock& b, Release release) {
    TmpBlock old;
    {
      std::lock_guard<std::mutex> lk(m_);
      if (b.bytes > kTmpKeepBytes || !add(b)) old = b;
    }
    while (old.p || over(b.device, &old)) {
      release(old);
      old = TmpBlock{};
    }
  }

  // Releases the device's blocks; false: there were none.
  template <typename Release>
  bool trim(int device, Release release) {
    bool any = false;
    TmpBlock b;
    while (oldest(device, &b)) {
      release(b);
      any = true;
    }
    return any;
  }

  template <typename Release>
  void trim_all(Release release) {
    std::vector<TmpBlock> out;
    {
      std::lock_guard<std::mutex> lk(m_);
      out.swap(blocks_);
    }
    for (const TmpBlock& b : out) release(b);
  }

  // An allocation (get() is false when memory has run out) that may ask for
  // the memory held here.
  template <typename Get, typename Release>
  bool get_or_trim(int device, Get get, Release release) {
    return get() || (trim(device, release) && get());
  }

  size_t held(int device) {
    std::lock_guard<std::mutex> lk(m_);
    return sum(device).first;
  }

 private:
  std::pair<size_t, size_t> sum(int device) const {
    std::pair<size_t, size_t> t{0, 0};
    for (const TmpBlock& f : blocks_)
      if (f.device == device) {
        t.first += f.bytes;
        t.second++;
      }
    return t;
  }
  bool add(const TmpBlock& b) {
    try {
      blocks_.push_back(b);
    } catch (...) {
      return false;  // (called from destructors)
    }
    return true;
  }
  bool pop(int device, TmpBlock* b) {
    for (size_t i = 0; i < blocks_.size(); i++)
      if (blocks_[i].device == device) {
        *b = blocks_[i];
        blocks_.erase(blocks_.begin() + (std::ptrdiff_t)i);
        return true;
      }
    return false;
  }
  bool oldest(int device, TmpBlock* b) {
    std::lock_guard<std::mutex> lk(m_);
    return pop(device, b);
  }
  // the block to let go of, if the device's are over a limit
  bool over(int device, TmpBlock* b) {
    std::lock_guard<std::mutex> lk(m_);
    const auto t = sum(device);
    return (t.first > kTmpKeepBytes || t.second > kTmpKeepBlocks) && pop(device, b);
  }

  std::mutex m_;
  std::vector<TmpBlock> blocks_;  // in the order they were given back
};

}  // namespace mph
