// Scratch memory of the single-op entry points: device blocks and pinned host
// staging kept between calls, because hipMalloc, hipFree (which waits for the
// whole device) and a synchronous copy each cost more than most of the ops'
// kernels (attention forward, 8192 packed tokens: 164 µs per call with them,
// 130 without; its kernel took 105 of them then).
//
// A block belongs to one call at a time: a Scratch takes it from the pool of
// its device under the pool's lock and gives it back only once the call's
// stream is idle, so calls on different threads and streams never share one
// and no kernel of an earlier call can still use it. The pool is bounded
// (kPoolBytes per device for what it keeps; a larger block is freed at the end
// of its call, the longest unused ones make room), emptied when an allocation
// of this library on its device fails, and released on request
// (dsb_release_workspaces).
#pragma once

#include <hip/hip_runtime.h>

#include <deque>
#include <mutex>
#include <vector>

namespace dsb {

constexpr size_t kPoolBytes = 512u << 20;  // kept per device
constexpr size_t kPinnedBytes = 16u << 20;  // kept, pinned host memory
constexpr int kPoolDevices = 64;

class BlockPool {
 public:
  struct Block {
    void* p = nullptr;
    size_t bytes = 0;
  };
  BlockPool(bool pinned, size_t limit) : pinned_(pinned), limit_(limit) {}

  // A block of at least `bytes`: a kept one at most twice as large, else new.
  Block get(size_t bytes) {
    const size_t need = round_up(bytes);
    {
      std::lock_guard<std::mutex> lk(mu_);
      auto best = kept_.end();
      for (auto it = kept_.begin(); it != kept_.end(); ++it)
        if (it->bytes >= need && it->bytes <= 2 * need &&
            (best == kept_.end() || it->bytes < best->bytes))
          best = it;
      if (best != kept_.end()) {
        const Block b = *best;
        kept_.erase(best);
        held_ -= b.bytes;
        return b;
      }
    }
    Block b;
    b.bytes = need;
    if (alloc(&b.p, need) != hipSuccess) {
      (void)hipGetLastError();
      trim(0);
      if (alloc(&b.p, need) != hipSuccess) b = Block{};
    }
    return b;
  }
  // Gives a block back, idle.
  void put(Block b) {
    if (!b.p) return;
    if (b.bytes > limit_) {
      release(b);
      return;
    }
    std::vector<Block> out;
    {
      // kept and the oldest evicted under one lock, so that calls returning
      // blocks together stay within the limit
      std::lock_guard<std::mutex> lk(mu_);
      kept_.push_back(b);
      held_ += b.bytes;
      evict(limit_, out);
    }
    for (const Block& v : out) release(v);
  }
  // Frees kept blocks, the longest kept first, down to `bytes`.
  void trim(size_t bytes) {
    std::vector<Block> out;
    {
      std::lock_guard<std::mutex> lk(mu_);
      evict(bytes, out);
    }
    for (const Block& b : out) release(b);
  }
  // Bytes kept.
  size_t held() {
    std::lock_guard<std::mutex> lk(mu_);
    return held_;
  }
  void release(const Block& b) { (void)(pinned_ ? hipHostFree(b.p) : hipFree(b.p)); }

 private:
  // under mu_: takes the longest kept blocks out until at most `bytes` stay
  void evict(size_t bytes, std::vector<Block>& out) {
    while (held_ > bytes && !kept_.empty()) {
      out.push_back(kept_.front());
      held_ -= kept_.front().bytes;
      kept_.pop_front();
    }
  }
  static size_t round_up(size_t bytes) {
    size_t r = 4096;
    while (r < bytes && r < (1u << 20)) r *= 2;
    return r >= bytes ? r : (bytes + (1u << 20) - 1) >> 20 << 20;
  }
  hipError_t alloc(void** p, size_t bytes) {
    return pinned_ ? hipHostMalloc(p, bytes, hipHostMallocPortable) : hipMalloc(p, bytes);
  }
  const bool pinned_;
  const size_t limit_;
  std::mutex mu_;
  std::deque<Block> kept_;
  size_t held_ = 0;
};

// The pools live until the process ends (never destroyed: the HIP runtime may
// be gone by then).
inline BlockPool& device_pool(int dev) {
  static std::mutex mu;
  static BlockPool* pools[kPoolDevices] = {};
  std::lock_guard<std::mutex> lk(mu);
  BlockPool*& p = pools[dev];
  if (!p) p = new BlockPool(false, kPoolBytes);
  return *p;
}
inline BlockPool& pinned_pool() {
  static BlockPool* p = new BlockPool(true, kPinnedBytes);
  return *p;
}

// hipMalloc on the current device for memory that is not the pool's; what the
// pool keeps there makes room if it fails.
inline hipError_t device_malloc(void** p, size_t bytes) {
  const hipError_t e = hipMalloc(p, bytes);
  int dev = 0;
  if (e == hipSuccess || hipGetDevice(&dev) != hipSuccess || dev >= kPoolDevices) return e;
  (void)hipGetLastError();
  device_pool(dev).trim(0);
  return hipMalloc(p, bytes);
}

// One call's scratch memory on stream s.
class Scratch {
 public:
  explicit Scratch(hipStream_t s) : s_(s) {
    if (hipGetDevice(&dev_) != hipSuccess || dev_ >= kPoolDevices) dev_ = -1;
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  ~Scratch() {
    // after a failure the stream may hold work that uses the blocks: wait for
    // it, and free rather than keep them if that cannot be established
    const bool idle = idle_ || hipStreamSynchronize(s_) == hipSuccess;
    for (const auto& b : host_) idle ? pinned_pool().put(b) : pinned_pool().release(b);
    for (const auto& b : dev_blocks_) idle ? device_pool(dev_).put(b) : device_pool(dev_).release(b);
  }
  // `count` T on the device (null when out of memory)
  template <class T>
  T* dev(size_t count) {
    if (dev_ < 0) return nullptr;
    const BlockPool::Block b = device_pool(dev_).get(count * sizeof(T) + 256);
    if (b.p) dev_blocks_.push_back(b);
    return (T*)b.p;
  }
  // `count` T of pinned host memory
  template <class T>
  T* host(size_t count) {
    const BlockPool::Block b = pinned_pool().get(count * sizeof(T) + 256);
    if (b.p) host_.push_back(b);
    return (T*)b.p;
  }
  // Waits for the stream: the call's results are complete, its blocks idle.
  hipError_t finish() {
    const hipError_t e = hipStreamSynchronize(s_);
    idle_ = e == hipSuccess;
    return e;
  }

 private:
  hipStream_t s_;
  int dev_ = -1;
  bool idle_ = false;
  std::vector<BlockPool::Block> dev_blocks_, host_;
};

}  // namespace dsb
