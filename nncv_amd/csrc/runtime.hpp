// Thin HIP runtime layer under the C ABI: device selection, one stream, owned device buffers,
// a grow-only bump arena for activations and transform workspaces, pinned staging buffers.
// The reference has no counterpart (its object runs in host memory); the only device code it
// contains are cudaMalloc/cudaFree wrappers (src/nncv/vm/cuda/vm_alloc_cuda.cu:6-10).
#pragma once
#include <algorithm>
#include <memory>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace nncv_hip {

class DevicePool;

class DeviceBuffer {
 public:
  DeviceBuffer() = default;
  explicit DeviceBuffer(size_t bytes) { reset(bytes); }
  DeviceBuffer(const DeviceBuffer&) = delete;
  DeviceBuffer& operator=(const DeviceBuffer&) = delete;
  DeviceBuffer(DeviceBuffer&& o) noexcept : p_(o.p_), n_(o.n_), owned_(o.owned_) { o.p_ = nullptr; o.n_ = 0; }
  DeviceBuffer& operator=(DeviceBuffer&& o) noexcept {
    if (this != &o) { release(); p_ = o.p_; n_ = o.n_; owned_ = o.owned_; o.p_ = nullptr; o.n_ = 0; }
    return *this;
  }
  ~DeviceBuffer() { release(); }
  void reset(size_t bytes) {
    release();
    if (bytes) NNCV_HIP_CHECK(hipMalloc(&p_, bytes));
    n_ = bytes;
    owned_ = true;
  }
  // from `pool` (which outlives this), or an allocation of its own where there is none
  void reset(size_t bytes, DevicePool* pool);
  void borrow(void* p, size_t bytes) {  // memory of another buffer, which outlives this one
    release();
    p_ = p;
    n_ = bytes;
    owned_ = false;
  }
  void release() {
    if (p_ && owned_) (void)hipFree(p_);
    p_ = nullptr;
    n_ = 0;
  }
  void* get() const { return p_; }
  template <typename T> T* as() const { return static_cast<T*>(p_); }
  size_t bytes() const { return n_; }

 private:
  void* p_ = nullptr;
  size_t n_ = 0;
  bool owned_ = true;
};

// Device memory for the weights of one network: handed out from a few large blocks, freed with the network.  A network has
// several hundred small arrays, and creating one spent most of its time in as many hipMalloc calls.  A network that takes
// the place of an idle one can take over its blocks (rewind): mapping and unmapping 100 MB costs the host 4 ms.
class DevicePool {
 public:
  DevicePool(size_t block = size_t(8) << 20) : block_(block) {}
  void* take(size_t bytes) {
    bytes = (bytes + 255) & ~size_t(255);
    while (cur_ < blocks_.size() && off_ + bytes > blocks_[cur_].bytes()) ++cur_, off_ = 0;
    if (cur_ == blocks_.size()) blocks_.emplace_back(std::max(bytes, block_));
    off_ += bytes;
    return blocks_[cur_].as<char>() + off_ - bytes;
  }
  void rewind() { cur_ = off_ = 0; }  // nothing handed out so far is used any more

 private:
  std::vector<DeviceBuffer> blocks_;
  size_t block_, cur_ = 0, off_ = 0;
};

inline void DeviceBuffer::reset(size_t bytes, DevicePool* pool) {
  if (!pool || bytes == 0) return reset(bytes);
  release();
  p_ = pool->take(bytes);
  n_ = bytes;
  owned_ = false;
}

class PinnedBuffer {
 public:
  ~PinnedBuffer() { if (p_) (void)hipHostFree(p_); }
  void* ensure(size_t bytes) {
    if (bytes > n_) {
      if (p_) (void)hipHostFree(p_);
      p_ = nullptr;
      NNCV_HIP_CHECK(hipHostMalloc(&p_, bytes, hipHostMallocDefault));
      n_ = bytes;
    }
    return p_;
  }

 private:
  void* p_ = nullptr;
  size_t n_ = 0;
};

// Bump allocator over one device allocation.  `plan` first (no memory touched), then `reserve`
// grows the backing store if the plan does not fit; pointers are handed out 256-byte aligned.
class Arena {
 public:
  // true when the backing store was replaced (pointers handed out before are gone)
  bool reserve(size_t bytes, hipStream_t s) {
    bool grown = false;
    if (bytes > buf_.bytes()) {
      NNCV_HIP_CHECK(hipStreamSynchronize(s));  // nobody may still be using the old block
      buf_.reset(bytes + bytes / 8);
      grown = true;
    }
    off_ = 0;
    return grown;
  }
  void* take(size_t bytes) {
    const size_t a = (off_ + 255) & ~size_t(255);
    NNCV_REQUIRE(a + bytes <= buf_.bytes(), "arena overflow: workspace plan and use disagree");
    off_ = a + bytes;
    return static_cast<char*>(buf_.get()) + a;
  }
  size_t capacity() const { return buf_.bytes(); }

 private:
  DeviceBuffer buf_;
  size_t off_ = 0;
};

inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// The device array behind nncv_hip_conv_forward_noalloc (noalloc.hip).  noalloc_scratch() is its address on the current
// device (resolved once per device).
constexpr size_t kNoAllocWorkspaceBytes = size_t(4) << 20;
void* noalloc_scratch();

// stream_probe.hip: up to `want` library-owned streams, the first *found of which were measured to overlap pairwise
std::vector<hipStream_t> pick_streams(int want, int* found);

// Orders calls that share device memory (the library's arena, a handle's workspace) across streams: a call on another
// stream than the previous one makes its stream wait for what that one left pending, and for nothing else.  The event it
// waits for belongs to the previous call: its last launch completes it (TailEvent, common.hpp), or it is recorded behind them
// while their stream is certainly alive and not being captured.  A later call never touches the earlier stream, which may be
// gone by then, and never waits for the device: another stream may be waiting for something the caller does next, and
// a device-wide wait ends any capture that is open elsewhere.  What that costs a program that stays on one stream: nothing
// behind a 15 us layer or a 28 us product; 2.4 us a pass where the last launch, which completes the event, is therefore not part
// of the replayed graph (ResNet-18 fp16, one image: 101.5 -> 103.9 us; 3.2 for MobileNetV3, 32 images: 227.8 -> 231.0); and host time where the
// host is what a call costs (a 20 x 30 x 40 product, called from Python: 4.1 -> 7.0 us a call; 9.1 with an event record).
class StreamOrder {
 public:
  StreamOrder() = default;
  StreamOrder(const StreamOrder&) = delete;
  StreamOrder& operator=(const StreamOrder&) = delete;
  ~StreamOrder();
  void create();                       // makes the event; no call does that later
  void after_previous(hipStream_t s);  // s waits for the previous call
  // the call that ends here left work in flight on s, or none; covered: its last launch completes event()
  void note(hipStream_t s, bool pending, bool covered);
  hipEvent_t event() const { return ev_; }

 private:
  hipStream_t tail_ = nullptr;  // stream of the previous call
  bool pending_ = false;        // it was left with work in flight
  hipEvent_t ev_ = nullptr;
};

// Process-wide state.  All public entry points serialise on `mu`.
class Context {
 public:
  static Context& get();
  void init(int device);  // idempotent; device < 0 keeps the current one
  hipStream_t stream() const { return stream_; }
  hipEvent_t event(size_t i);  // kept events of the host-buffer calls
  int device() const { return device_; }
  const std::string& arch() const { return arch_; }
  Arena arena;
  PinnedBuffer pin_in, pin_out;
  std::recursive_mutex mu;
  StreamOrder order;  // of consecutive calls, which share the arena: see Sync in capi.cpp

 private:
  bool ready_ = false;
  int device_ = -1;
  hipStream_t stream_ = nullptr;
  std::vector<hipEvent_t> events_;
  std::string arch_;
};

}  // namespace nncv_hip
