// devpool.hpp -- device memory kept between the objects of one context.
//
// A batch lives for one call in the usual program (the command line scores
// each alignment once), and hipMalloc / hipFree cost microseconds to hundreds
// of milliseconds each (the driver clears what it hands out: a maximiser's
// 20 GB of transition sets took 0.49 s of a 0.56 s call).  Freed blocks are
// kept per context and handed out again to that context only: its work is
// ordered on one stream, so a block's next user runs after its last one.  At
// most kKeep bytes are kept; beyond it, at the context's end, and when the
// device runs out of memory (any context's), blocks go back to the driver.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>

namespace pcsf {

class DevPool {
 public:
  static constexpr size_t kKeep = (size_t)16 << 30;

  // a context's id (0 is no context: nothing is kept)
  uint64_t open() {
    std::lock_guard<std::mutex> lock(mu_);
    const uint64_t id = ++last_;
    kept_[id];
    return id;
  }
  // the context's stream has drained
  void close(uint64_t id) {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = kept_.find(id);
    if (it == kept_.end()) return;
    give_back(it->second, 0);
    kept_.erase(it);
  }
  hipError_t alloc(uint64_t id, size_t bytes, void** out) {
    const size_t size = rounded(bytes);
    std::lock_guard<std::mutex> lock(mu_);
    auto it = kept_.find(id);
    if (it != kept_.end()) {
      // the smallest kept block that fits without wasting half of itself
      auto b = it->second.blocks.lower_bound(size);
      if (b != it->second.blocks.end() && b->first <= 2 * size) {
        *out = b->second;
        live_[*out] = {b->first, id};
        it->second.bytes -= b->first;
        it->second.blocks.erase(b);
        return hipSuccess;
      }
    }
    hipError_t e = hipMalloc(out, size);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      for (auto& k : kept_) give_back(k.second, 0);
      e = hipMalloc(out, size);
    }
    if (e == hipSuccess) live_[*out] = {size, id};
    return e;
  }
  void free(void* p) {
    std::lock_guard<std::mutex> lock(mu_);
    auto l = live_.find(p);
    if (l == live_.end()) return;
    const Live was = l->second;
    live_.erase(l);
    auto it = kept_.find(was.id);
    if (it == kept_.end() || was.bytes > kKeep) {
      (void)hipFree(p);
      return;
    }
    give_back(it->second, kKeep - was.bytes);
    it->second.blocks.emplace(was.bytes, p);
    it->second.bytes += was.bytes;
  }
  // back to the driver, not kept: for memory whose address a caller may have
  // given to streams of their own (hipFree waits for the whole device)
  void release(void* p) {
    std::lock_guard<std::mutex> lock(mu_);
    if (live_.erase(p)) (void)hipFree(p);
  }

 private:
  struct Kept {
    std::multimap<size_t, void*> blocks;
    size_t bytes = 0;
  };
  struct Live {
    size_t bytes;
    uint64_t id;
  };
  // 256-byte steps, an eighth of the size's power of two above 2 KB: batches of
  // nearly the same size share blocks
  static size_t rounded(size_t n) {
    size_t step = 256;
    while (step * 16 <= n) step *= 2;
    return (n + step - 1) / step * step;
  }
  // hipFree waits for the device, so a block still in use there is safe to give
  static void give_back(Kept& k, size_t down_to) {
    while (k.bytes > down_to) {
      auto b = std::prev(k.blocks.end());
      (void)hipFree(b->second);
      k.bytes -= b->first;
      k.blocks.erase(b);
    }
  }

  std::mutex mu_;
  uint64_t last_ = 0;
  std::unordered_map<uint64_t, Kept> kept_;
  std::unordered_map<void*, Live> live_;
};

}  // namespace pcsf
