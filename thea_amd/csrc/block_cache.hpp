// Device memory blocks kept between allocations, over a Driver (the HIP calls in capi.hip, a model of
// them in tests/block_cache_check.cpp).
//
// A freed block is kept for the next allocation of about its size (at least its request, at most a
// quarter more), up to `limit` bytes per device, oldest given back first. All of a device's blocks are
// given back by release() and reclaim(), and before any allocation of this library is reported as failed, whichever
// allocator it came from. Like a driver's free, free() waits for the device first, so a kept block is
// idle and any stream or thread may take it.
#pragma once

#include <cstddef>
#include <mutex>
#include <new>
#include <vector>

namespace thg {

// Driver: types Error and Stream; ok(e), out_of_memory(e) (which clears the driver's last error);
// alloc(p, n), alloc_async(p, n, stream) on the current device; free(p); wait(device), true if it is
// idle; trim(device), which gives back what the stream-ordered pool does not use.
template <class Driver> class BlockCache {
 public:
  using Error = typename Driver::Error;
  BlockCache(Driver d, size_t limit) : drv(d), limit_(limit) {}

  Error alloc(void **p, size_t n, int device, size_t *block) {
    *block = n;
    if (take(p, n, device, block)) return drv.success();
    Error e = drv.alloc(p, n);
    if (drv.out_of_memory(e)) {
      reclaim(device);
      e = drv.alloc(p, n);
    }
    return e;
  }

  Error alloc_async(void **p, size_t n, int device, typename Driver::Stream s) {
    Error e = drv.alloc_async(p, n, s);
    if (drv.out_of_memory(e)) {
      reclaim(device);
      e = drv.alloc_async(p, n, s);
    }
    return e;
  }

  // Called from destructors: nothing leaves it.
  void free(void *p, size_t block, int device) noexcept {
    if (block > limit_ || !drv.wait(device) || !keep(p, block, device)) {
      drv.free(p);
      return;
    }
    give_back(device, limit_);
  }

  // Gives back the device's kept blocks.
  void release(int device) { give_back(device, 0); }
  // Gives back the device's kept blocks and what its stream-ordered pool does not use.
  void reclaim(int device) {
    release(device);
    drv.trim(device);
  }

 private:
  struct Block {
    void *p;
    size_t bytes;
    int device;
  };
  Driver drv;
  const size_t limit_;
  std::mutex mu;
  std::vector<Block> kept;  // oldest first

  // False if there is no host memory to note the block.
  bool keep(void *p, size_t block, int device) {
    std::lock_guard<std::mutex> g(mu);
    try {
      kept.push_back({p, block, device});
    } catch (const std::bad_alloc &) {
      return false;
    }
    return true;
  }

  bool take(void **p, size_t n, int device, size_t *block) {
    std::lock_guard<std::mutex> g(mu);
    size_t best = kept.size();
    for (size_t i = 0; i < kept.size(); ++i)
      if (kept[i].device == device && kept[i].bytes >= n && kept[i].bytes - n <= n / 4 &&
          (best == kept.size() || kept[i].bytes < kept[best].bytes))
        best = i;
    if (best == kept.size()) return false;
    *p = kept[best].p;
    *block = kept[best].bytes;
    kept.erase(kept.begin() + best);
    return true;
  }

  // Gives the device's oldest blocks back until at most `most` bytes of them are kept.
  void give_back(int device, size_t most) {
    while (true) {
      void *p = nullptr;
      {
        std::lock_guard<std::mutex> g(mu);
        size_t held = 0, oldest = kept.size();
        for (size_t i = kept.size(); i-- > 0;)
          if (kept[i].device == device) {
            held += kept[i].bytes;
            oldest = i;
          }
        if (held <= most) return;
        p = kept[oldest].p;
        kept.erase(kept.begin() + oldest);
      }
      drv.free(p);
    }
  }
};

}  // namespace thg
