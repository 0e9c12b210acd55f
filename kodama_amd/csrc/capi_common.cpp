// Library-level entry points of the C ABI and the helpers of capi_common.h.
#include "capi_common.h"

#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace kodama_hip {

namespace {
thread_local std::string g_last_error;
thread_local int g_knn_fallbacks = -1;
std::mutex g_arch_mutex;
std::vector<int> g_arch_ok;  // -1 unknown, 0 not gfx950, 1 gfx950

// Idle streams by device; never destroyed at exit (the runtime may be gone).
struct IdleStreams {
  std::mutex mutex;
  std::map<int, std::vector<hipStream_t>> by_device;
};
IdleStreams& idle_streams() {
  static IdleStreams* const pool = new IdleStreams;
  return *pool;
}
}  // namespace

hipStream_t take_stream(int device) {
  IdleStreams& pool = idle_streams();
  {
    std::lock_guard<std::mutex> lock(pool.mutex);
    std::vector<hipStream_t>& idle = pool.by_device[device];
    if (!idle.empty()) {
      const hipStream_t s = idle.back();
      idle.pop_back();
      return s;
    }
  }
  hipStream_t s = nullptr;
  check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
  return s;
}

void give_stream(int device, hipStream_t s) {
  // A call that failed may leave work behind: wait for it. A stream that
  // cannot be waited for (a broken capture, a device error) is not used again.
  const bool idle_now = hipStreamSynchronize(s) == hipSuccess;
  if (idle_now) {
    pool_settle(device, s);
    IdleStreams& pool = idle_streams();
    std::lock_guard<std::mutex> lock(pool.mutex);
    std::vector<hipStream_t>& idle = pool.by_device[device];
    if (idle.size() < kIdleStreams) {
      idle.push_back(s);
      return;
    }
  } else {
    pool_drop(device, s);
  }
  (void)hipStreamDestroy(s);
}

void set_last_error(const std::string& msg) { g_last_error = msg; }

int& last_knn_fallbacks() { return g_knn_fallbacks; }

void select_device(int device) {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
    throw NoDevice("no HIP device is visible; the HIP backend requires an MI355X (gfx950).");
  }
  if (device < 0 || device >= count) throw NoDevice("gpu_device is outside the visible HIP devices.");
  {
    std::lock_guard<std::mutex> lock(g_arch_mutex);
    if (g_arch_ok.size() != static_cast<size_t>(count)) g_arch_ok.assign(static_cast<size_t>(count), -1);
    if (g_arch_ok[device] < 0) {
      hipDeviceProp_t prop;
      check(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties");
      g_arch_ok[device] = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
    }
    if (g_arch_ok[device] != 1) throw NoDevice("the HIP backend is built for gfx950 (MI355X) only.");
  }
  check(hipSetDevice(device), "hipSetDevice");
}

}  // namespace kodama_hip

extern "C" {

const char* kodama_hip_last_error(void) { return kodama_hip::g_last_error.c_str(); }

const char* kodama_hip_version(void) { return "kodama_hip 0.1.0 gfx950"; }

int kodama_hip_last_knn_fallbacks(void) { return kodama_hip::g_knn_fallbacks; }

int kodama_hip_release_memory(int32_t device) {
  return kodama_hip::guarded([&] {
    kodama_hip::select_device(device);
    kodama_hip::pool_empty(device);
  });
}

int kodama_hip_device_count(int32_t* count) {
  return kodama_hip::guarded([&] {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    int ok = 0;
    for (int d = 0; d < n; ++d) {
      hipDeviceProp_t prop;
      if (hipGetDeviceProperties(&prop, d) == hipSuccess && std::strncmp(prop.gcnArchName, "gfx950", 6) == 0) ++ok;
    }
    *count = ok;
  });
}

}  // extern "C"
