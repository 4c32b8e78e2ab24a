// devpool.hpp -- device memory kept between the objects of one context.
//
// A batch lives for one call in the usual program (the command line scores
// each alignment once), and hipMalloc / hipFree cost microseconds to hundreds
// of milliseconds each, with the size and the state of the driver (a maximiser's
// 20 GB of transition sets: under 10 ms on some machines, half a second on
// others, where the driver clears what it hands out).  Freed blocks are
// kept per context and handed out again to that context only: its work is
// ordered on one stream, so a block's next user runs after its last one.  At
// most kKeep bytes are kept, the latest freed; beyond it, at the context's end,
// and when the device runs out of memory (any context's), blocks go back to the
// driver.  No lock is held while the driver allocates or frees, which can wait
// for the device.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

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
    std::vector<void*> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = kept_.find(id);
      if (it == kept_.end()) return;
      it->second.take_oldest(0, &out);
      kept_.erase(it);
    }
    to_driver(out);
  }
  hipError_t alloc(uint64_t id, size_t bytes, void** out) {
    size_t size = rounded(bytes);
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = kept_.find(id);
      if (it != kept_.end() && (*out = it->second.take_fitting(&size))) {
        live_[*out] = {size, id};
        return hipSuccess;
      }
    }
    hipError_t e = hipMalloc(out, size);
    if (e == hipErrorOutOfMemory) {
      // one thread at a time, so that none gives up while another gives back
      std::lock_guard<std::mutex> lock_empty(empty_);
      (void)hipGetLastError();
      std::vector<void*> all;
      {
        std::lock_guard<std::mutex> lock(mu_);
        for (auto& k : kept_) k.second.take_oldest(0, &all);
      }
      to_driver(all);
      e = hipMalloc(out, size);
    }
    if (e == hipSuccess) {
      std::lock_guard<std::mutex> lock(mu_);
      live_[*out] = {size, id};
    }
    return e;
  }
  void free(void* p) {
    std::vector<void*> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto l = live_.find(p);
      if (l == live_.end()) return;
      const Live was = l->second;
      live_.erase(l);
      auto it = kept_.find(was.id);
      if (it == kept_.end() || was.bytes > kKeep) {
        out.push_back(p);
      } else {
        it->second.take_oldest(kKeep - was.bytes, &out);
        it->second.put(was.bytes, p);
      }
    }
    to_driver(out);
  }
  // back to the driver, not kept: for memory whose address a caller may have
  // given to streams of their own (hipFree waits for the whole device)
  void release(void* p) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (!live_.erase(p)) return;
    }
    (void)hipFree(p);
  }

 private:
  struct Kept {
    struct Block {
      size_t bytes;
      void* p;
    };
    std::list<Block> by_age;  // the oldest first
    std::multimap<size_t, std::list<Block>::iterator> by_size;
    size_t bytes = 0;

    void put(size_t n, void* p) {
      by_age.push_back({n, p});
      by_size.emplace(n, std::prev(by_age.end()));
      bytes += n;
    }
    // the smallest block that fits without wasting half of itself (its size in
    // *size), or nullptr
    void* take_fitting(size_t* size) {
      auto b = by_size.lower_bound(*size);
      if (b == by_size.end() || b->first > 2 * *size) return nullptr;
      void* p = b->second->p;
      *size = b->first;
      bytes -= b->first;
      by_age.erase(b->second);
      by_size.erase(b);
      return p;
    }
    void take_oldest(size_t down_to, std::vector<void*>* out) {
      while (bytes > down_to) {
        const Block b = by_age.front();
        auto r = by_size.equal_range(b.bytes);
        while (r.first->second != by_age.begin()) ++r.first;
        by_size.erase(r.first);
        by_age.pop_front();
        bytes -= b.bytes;
        out->push_back(b.p);
      }
    }
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
  static void to_driver(const std::vector<void*>& blocks) {
    for (void* p : blocks) (void)hipFree(p);
  }

  std::mutex mu_, empty_;
  uint64_t last_ = 0;
  std::unordered_map<uint64_t, Kept> kept_;
  std::unordered_map<void*, Live> live_;
};

}  // namespace pcsf
