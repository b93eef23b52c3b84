// The library's pool of device memory.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

namespace ddf {

// Stream-ordered allocation from a pool that the library keeps for each device; freed with hipFreeAsync.
// Of what has been freed the pool keeps kPoolKeep bytes for the next call and returns the rest to the
// device when a stream is synchronised (the default pool keeps nothing, and hipMalloc / hipFree map and
// unmap every buffer and wait for the device: 18 of 31 ms of a plan build for 25 facets).  A failing
// allocation gives the kept bytes back and tries once more, and so does ddf_trim_memory for other users of the
// device.  Safe from several threads and streams, as the runtime's pools are.
constexpr size_t kPoolKeep = size_t(4) << 30;
hipError_t pool_alloc(void** p, size_t bytes, hipStream_t st);
// gives back what the current device's pool holds unused beyond `keep` bytes
hipError_t pool_trim(size_t keep);

// The buffers of one object or call: small ones are cut from slabs of 2 MiB, growing to 32 MiB, since an
// allocation and its release take some 16 us of host time whatever their size (a plan has about 60).
class PoolArena {
 public:
  void* get(size_t bytes, hipStream_t st) {
    if (empty() && hipGetDevice(&dev_) != hipSuccess) return nullptr;
    bytes = (std::max<size_t>(bytes, 1) + 255) & ~size_t(255);
    if (bytes > left_) {
      const size_t slab = size_t(2 << 20) << std::min<size_t>(slabs_.size(), 4);
      const bool own = bytes > slab / 2;
      void* p = nullptr;
      if (pool_alloc(&p, own ? bytes : slab, st) != hipSuccess) return nullptr;
      (own ? own_ : slabs_).push_back(p);
      bytes_ += own ? bytes : slab;
      if (own) return p;
      cur_ = static_cast<char*>(p);
      left_ = slab;
    }
    void* p = cur_;
    cur_ += bytes;
    left_ -= bytes;
    return p;
  }
  void release_all(hipStream_t st) {
    for (void* p : own_) (void)hipFreeAsync(p, st);
    for (void* p : slabs_) (void)hipFreeAsync(p, st);
    own_.clear();
    slabs_.clear();
    cur_ = nullptr;
    left_ = bytes_ = 0;
  }
  size_t bytes() const { return bytes_; }  // of device memory held
  // takes over the buffers of another arena of the same device
  void take(PoolArena& o) {
    if (empty()) dev_ = o.dev_;
    own_.insert(own_.end(), o.own_.begin(), o.own_.end());
    own_.insert(own_.end(), o.slabs_.begin(), o.slabs_.end());
    bytes_ += o.bytes_;
    o.own_.clear();
    o.slabs_.clear();
    o.cur_ = nullptr;
    o.left_ = o.bytes_ = 0;
  }
  bool empty() const { return own_.empty() && slabs_.empty(); }
  // Gives everything back at the end of an object whose work may still run on any stream: waits for the device of
  // the buffers, whichever one is current, and hands what the pool does not keep to the device before it returns.
  void close() {
    if (empty()) return;
    int cur = dev_;
    (void)hipGetDevice(&cur);
    if (cur != dev_) (void)hipSetDevice(dev_);
    (void)hipDeviceSynchronize();
    release_all(nullptr);
    (void)hipStreamSynchronize(nullptr);
    (void)pool_trim(kPoolKeep);
    if (cur != dev_) (void)hipSetDevice(cur);
  }

 private:
  int dev_ = 0;  // of the buffers
  std::vector<void*> own_, slabs_;
  char* cur_ = nullptr;  // of the newest slab
  size_t left_ = 0, bytes_ = 0;
};

}  // namespace ddf
