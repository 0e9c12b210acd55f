// HIP runtime helpers for the host engine: error checks that throw, RAII device
// and pinned host buffers, and a per-thread stream bound to a device.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <utility>

namespace kodama_hip {

struct DeviceError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

inline void check(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
  }
}

// Device memory kept from one call for the next (device_pool.cpp). hipFree
// waits for the whole device and its cost is not bounded by the size: the ten
// frees of a batch's table build took 1.8 ms, 14 ms once a process had freed
// some thousand blocks. A block freed under a stream may still be read or
// written by work queued there, so it goes only to allocations under the same
// stream until that stream has been settled (its work done); then to any.
// At most kPoolBytes per device stay in the pool: a block that comes back to a
// full pool takes the place of the settled blocks unused the longest, so what
// stays follows the sizes that calls ask for now; where those do not make room
// it is freed. A failed allocation empties the pool first.
constexpr size_t kPoolBytes = size_t(2) << 30;
struct PoolBlock {
  void* p = nullptr;
  size_t bytes = 0;         // of the block
  int device = -1;
  hipStream_t tag = nullptr;  // null: not from the pool
  uint64_t given = 0;         // order of return, of kept blocks
};
// hipMalloc on the current device (`device`); on failure the pool of that
// device is emptied and the request repeated. Throws DeviceError.
void* device_alloc(size_t bytes, int device);
PoolBlock pool_take(size_t bytes, int device, hipStream_t tag);
void pool_give(const PoolBlock& block);
void pool_empty(int device);  // frees everything kept (hipFree waits for its work)
void pool_settle(int device, hipStream_t tag);  // every block of this tag is idle
void pool_drop(int device, hipStream_t tag);    // free them instead (their work is unknown)

// The stream under which the calling thread's DeviceBuffers allocate; scopes
// nest. Without one they use device_alloc and hipFree.
class Stream;
class StreamScope {
 public:
  explicit StreamScope(const Stream& s);
  ~StreamScope();
  StreamScope(const StreamScope&) = delete;
  StreamScope& operator=(const StreamScope&) = delete;
  static hipStream_t current();
  static int current_device();

 private:
  hipStream_t before_;
  int before_device_;
};

// All work on a buffer that is not yet done when it is released must be on
// the stream it was allocated under.
template <class T>
class DeviceBuffer {
 public:
  DeviceBuffer() = default;
  explicit DeviceBuffer(size_t n) { resize(n); }
  ~DeviceBuffer() { release(); }
  DeviceBuffer(const DeviceBuffer&) = delete;
  DeviceBuffer& operator=(const DeviceBuffer&) = delete;
  DeviceBuffer(DeviceBuffer&& o) noexcept : block_(o.block_), n_(o.n_) { o.block_ = PoolBlock(); o.n_ = 0; }
  DeviceBuffer& operator=(DeviceBuffer&& o) noexcept {
    if (this != &o) {
      release();
      block_ = o.block_; n_ = o.n_;
      o.block_ = PoolBlock(); o.n_ = 0;
    }
    return *this;
  }
  void resize(size_t n) {
    if (n == n_) return;
    release();
    if (n > 0) {
      if (StreamScope::current() != nullptr) {
        block_ = pool_take(n * sizeof(T), StreamScope::current_device(), StreamScope::current());
      } else {
        int device = 0;
        check(hipGetDevice(&device), "hipGetDevice");
        block_.p = device_alloc(n * sizeof(T), device);
      }
    }
    n_ = n;
  }
  void release() {
    if (block_.tag != nullptr) pool_give(block_);
    else if (block_.p != nullptr) (void)hipFree(block_.p);
    block_ = PoolBlock();
    n_ = 0;
  }
  T* get() const { return static_cast<T*>(block_.p); }
  size_t size() const { return n_; }
  void upload(const T* src, size_t n, hipStream_t s, size_t offset = 0) {
    if (n) check(hipMemcpyAsync(get() + offset, src, n * sizeof(T), hipMemcpyHostToDevice, s), "upload");
  }
  void download(T* dst, size_t n, hipStream_t s, size_t offset = 0) const {
    if (n) check(hipMemcpyAsync(dst, get() + offset, n * sizeof(T), hipMemcpyDeviceToHost, s), "download");
  }

 private:
  PoolBlock block_;
  size_t n_ = 0;
};

// One pool block under a given stream.
class PoolBuffer {
 public:
  PoolBuffer() = default;
  ~PoolBuffer() { release(); }
  PoolBuffer(const PoolBuffer&) = delete;
  PoolBuffer& operator=(const PoolBuffer&) = delete;
  void allocate(size_t bytes, int device, hipStream_t s) {
    release();
    block_ = pool_take(bytes, device, s);
    bytes_ = bytes;
  }
  void release() {
    if (block_.p != nullptr) pool_give(block_);
    block_ = PoolBlock();
    bytes_ = 0;
  }
  unsigned char* get() const { return static_cast<unsigned char*>(block_.p); }
  size_t size() const { return bytes_; }

 private:
  PoolBlock block_;
  size_t bytes_ = 0;
};

template <class T>
class PinnedBuffer {
 public:
  PinnedBuffer() = default;
  explicit PinnedBuffer(size_t n) { resize(n); }
  ~PinnedBuffer() { release(); }
  PinnedBuffer(const PinnedBuffer&) = delete;
  PinnedBuffer& operator=(const PinnedBuffer&) = delete;
  void resize(size_t n) {
    if (n == n_) return;
    release();
    if (n > 0) check(hipHostMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T), hipHostMallocDefault), "hipHostMalloc");
    n_ = n;
  }
  void release() {
    if (p_ != nullptr) (void)hipHostFree(p_);
    p_ = nullptr;
    n_ = 0;
  }
  T* get() const { return p_; }
  T& operator[](size_t i) { return p_[i]; }
  const T& operator[](size_t i) const { return p_[i]; }
  size_t size() const { return n_; }

 private:
  T* p_ = nullptr;
  size_t n_ = 0;
};

// Idle streams kept for the next call on their device (creating and destroying
// one takes 0.24 ms, a small call a few times that): at most kIdleStreams per
// device, the rest destroyed. A stream comes back when its work is done, and
// its pool blocks are settled then.
constexpr size_t kIdleStreams = 8;
hipStream_t take_stream(int device);
void give_stream(int device, hipStream_t s);

// A stream on a chosen device, default priority.
class Stream {
 public:
  explicit Stream(int device) : device_(device) {
    check(hipSetDevice(device), "hipSetDevice");
    s_ = take_stream(device);
  }
  ~Stream() {
    if (s_ != nullptr) give_stream(device_, s_);
  }
  Stream(const Stream&) = delete;
  Stream& operator=(const Stream&) = delete;
  hipStream_t get() const { return s_; }
  int device() const { return device_; }
  void sync() const { check(hipStreamSynchronize(s_), "hipStreamSynchronize"); }

 private:
  hipStream_t s_ = nullptr;
  int device_ = 0;
};

// Event-timed region on a stream (milliseconds).
class EventTimer {
 public:
  EventTimer() {
    check(hipEventCreate(&a_), "hipEventCreate");
    check(hipEventCreate(&b_), "hipEventCreate");
  }
  ~EventTimer() {
    (void)hipEventDestroy(a_);
    (void)hipEventDestroy(b_);
  }
  void start(hipStream_t s) { check(hipEventRecord(a_, s), "hipEventRecord"); }
  void stop(hipStream_t s) { check(hipEventRecord(b_, s), "hipEventRecord"); }
  void wait() { check(hipEventSynchronize(b_), "hipEventSynchronize"); }
  float ms() {
    check(hipEventSynchronize(b_), "hipEventSynchronize");
    float v = 0.0f;
    check(hipEventElapsedTime(&v, a_, b_), "hipEventElapsedTime");
    return v;
  }

 private:
  hipEvent_t a_ = nullptr, b_ = nullptr;
};

}  // namespace kodama_hip
