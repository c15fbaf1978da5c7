// Device and pinned host memory kept between contexts.
//
// A solve of a small problem otherwise spends more time in hipMalloc and
// hipFree than in its kernels, and a large one frees its ~100 arrays for
// milliseconds (each hipFree waits for the device and unmaps).  Blocks go back
// to the cache only after the streams that used them have drained, so a block
// taken from it has no work outstanding, whichever stream uses it next.
//
// The cache is bounded (kCacheLimit bytes per device, kPinnedLimit per device and
// pinned kind, kCacheBlocks blocks) and gives a block back to the system when it
// has lain unused for kCacheAge releases of a context.  Before an allocation is
// reported as out of memory, the blocks that stand in its way are given back:
// the device's, or all pinned ones.  What no context uses otherwise stays until
// release_all() (mba_release_cached_memory).  One lock; every thread and stream
// may use it.
#ifndef MBA_POOL_H_
#define MBA_POOL_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace mba {

enum class MemKind { kDevice, kPinned, kPinnedCoherent };

class MemCache {
 public:
  static constexpr size_t kCacheLimit = size_t(4) << 30, kPinnedLimit = size_t(128) << 20;
  static constexpr size_t kCacheBlocks = 256;
  static constexpr uint64_t kCacheAge = 64;

  static MemCache& get() {
    static MemCache* c = new MemCache();  // never destroyed: contexts may outlive static destructors
    return *c;
  }
  // A block of at least `bytes` on the current device (*size: its real size).
  hipError_t take(MemKind kind, size_t bytes, void** out, size_t* size) {
    int dev = 0;
    const hipError_t de = hipGetDevice(&dev);
    if (de != hipSuccess) return de;
    const size_t grain = kind == MemKind::kDevice ? size_t(1) << 16 : 4096;
    const size_t want = (bytes + grain - 1) / grain * grain;
    {
      std::lock_guard<std::mutex> g(m_);
      // The smallest block that fits and is not more than a quarter (or 1 MB) too large.
      size_t best = blocks_.size();
      for (size_t i = 0; i < blocks_.size(); ++i) {
        const Block& b = blocks_[i];
        if (b.dev != dev || b.kind != kind || b.size < want || b.size > want + std::max(want / 4, size_t(1) << 20))
          continue;
        if (best == blocks_.size() || b.size < blocks_[best].size) best = i;
      }
      if (best != blocks_.size()) {
        *out = blocks_[best].p;
        *size = blocks_[best].size;
        held(kind, dev) -= blocks_[best].size;
        blocks_.erase(blocks_.begin() + (long)best);
        return hipSuccess;
      }
    }
    hipError_t e = raw_alloc(kind, want, out);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      if (kind == MemKind::kDevice) drop([dev](const Block& b) { return b.kind == MemKind::kDevice && b.dev == dev; });
      else drop([](const Block& b) { return b.kind != MemKind::kDevice; });
      e = raw_alloc(kind, want, out);
    }
    *size = want;
    return e;
  }
  // A block that no queued or running work uses any more.
  void give(MemKind kind, int dev, void* p, size_t size) {
    if (!p) return;
    {
      std::lock_guard<std::mutex> g(m_);
      size_t& h = held(kind, dev);
      if (h + size <= (kind == MemKind::kDevice ? kCacheLimit : kPinnedLimit) && blocks_.size() < kCacheBlocks) {
        blocks_.push_back(Block{p, size, kind, dev, clock_});
        h += size;
        return;
      }
    }
    raw_free(kind, p);
  }
  // A context has gone: blocks unused for kCacheAge of these are freed.
  void tick() {
    uint64_t now;
    {
      std::lock_guard<std::mutex> g(m_);
      now = ++clock_;
    }
    drop([now](const Block& b) { return b.since + kCacheAge < now; });
  }
  // Every unused block back to the system.
  void release_all() {
    drop([](const Block&) { return true; });
  }

 private:
  struct Block {
    void* p;
    size_t size;
    MemKind kind;
    int dev;
    uint64_t since;
  };
  static constexpr int kDevices = 64;
  size_t& held(MemKind kind, int dev) { return held_[(int)kind][dev % kDevices]; }
  static hipError_t raw_alloc(MemKind kind, size_t bytes, void** out) {
    if (kind == MemKind::kDevice) return hipMalloc(out, bytes);
    return hipHostMalloc(out, bytes, kind == MemKind::kPinned ? hipHostMallocDefault : hipHostMallocCoherent);
  }
  static void raw_free(MemKind kind, void* p) {
    if (kind == MemKind::kDevice) (void)hipFree(p);
    else (void)hipHostFree(p);
  }
  template <typename F>
  void drop(F&& which) {
    std::vector<Block> gone;
    {
      std::lock_guard<std::mutex> g(m_);
      for (size_t i = 0; i < blocks_.size();) {
        if (which(blocks_[i])) {
          held(blocks_[i].kind, blocks_[i].dev) -= blocks_[i].size;
          gone.push_back(blocks_[i]);
          blocks_.erase(blocks_.begin() + (long)i);
        } else {
          ++i;
        }
      }
    }
    for (const Block& b : gone) raw_free(b.kind, b.p);
  }
  std::mutex m_;
  std::vector<Block> blocks_;
  size_t held_[3][kDevices] = {};
  uint64_t clock_ = 0;
};

// The device memory of one owner (a context, one build's temporaries): small
// arrays share slabs.  release() after the owner's streams have drained.
class DevicePool {
 public:
  hipError_t raw(void** out, size_t bytes) {
    bytes = (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
    if (bytes >= kSlab / 2) return take(bytes, out);
    if (left_ < bytes) {
      void* p = nullptr;
      const hipError_t e = take(kSlab, &p);
      if (e != hipSuccess) return e;
      cur_ = (char*)p;
      left_ = kSlab;
    }
    *out = cur_;
    cur_ += bytes;
    left_ -= bytes;
    return hipSuccess;
  }
  void release() {
    for (const Block& b : blocks_) MemCache::get().give(MemKind::kDevice, b.dev, b.p, b.size);
    blocks_.clear();
    cur_ = nullptr;
    left_ = 0;
  }

 private:
  static constexpr size_t kSlab = size_t(1) << 20;
  struct Block {
    void* p;
    size_t size;
    int dev;
  };
  hipError_t take(size_t bytes, void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    size_t size = 0;
    e = MemCache::get().take(MemKind::kDevice, bytes, out, &size);
    if (e == hipSuccess) blocks_.push_back(Block{*out, size, dev});
    return e;
  }
  std::vector<Block> blocks_;
  char* cur_ = nullptr;
  size_t left_ = 0;
};

// One pinned host block (returned to the cache by drop()).
struct PinnedBlock {
  void* p = nullptr;
  size_t size = 0;
  int dev = 0;
  MemKind kind = MemKind::kPinned;
  hipError_t take(size_t bytes, MemKind k = MemKind::kPinned) {
    kind = k;
    const hipError_t e = hipGetDevice(&dev);
    return e != hipSuccess ? e : MemCache::get().take(kind, bytes, &p, &size);
  }
  void drop() {
    MemCache::get().give(kind, dev, p, size);
    p = nullptr;
  }
};

}  // namespace mba

#endif  // MBA_POOL_H_
