// The device memory pool (device.h).
#include <map>
#include <mutex>
#include <vector>

#include "device.h"

namespace kodama_hip {

namespace {

// Blocks are whole multiples of this; smaller requests share it.
constexpr size_t kGrain = size_t(64) << 10;

struct Pool {
  std::mutex mutex;
  struct PerDevice {
    std::multimap<size_t, PoolBlock> blocks;  // by size; tag null once settled
    size_t bytes = 0;
    uint64_t returns = 0;
  };
  std::map<int, PerDevice> devices;
};
// Never destroyed: at exit the runtime may be gone before it.
Pool& pool() {
  static Pool* const p = new Pool;
  return *p;
}

thread_local hipStream_t g_scope = nullptr;
thread_local int g_scope_device = -1;

}  // namespace

StreamScope::StreamScope(const Stream& s) : before_(g_scope), before_device_(g_scope_device) {
  g_scope = s.get();
  g_scope_device = s.device();
}
StreamScope::~StreamScope() {
  g_scope = before_;
  g_scope_device = before_device_;
}
hipStream_t StreamScope::current() { return g_scope; }
int StreamScope::current_device() { return g_scope_device; }

void pool_empty(int device) {
  Pool& pl = pool();
  std::vector<void*> kept;
  {
    std::lock_guard<std::mutex> lock(pl.mutex);
    Pool::PerDevice& d = pl.devices[device];
    for (auto& kv : d.blocks) kept.push_back(kv.second.p);
    d.blocks.clear();
    d.bytes = 0;
  }
  for (void* p : kept) (void)hipFree(p);
}

void* device_alloc(size_t bytes, int device) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  pool_empty(device);
  const hipError_t e = hipMalloc(&p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();  // not to be found by the next launch
  check(e, "hipMalloc");
  return p;
}

PoolBlock pool_take(size_t bytes, int device, hipStream_t tag) {
  const size_t need = (bytes + kGrain - 1) / kGrain * kGrain;
  Pool& pl = pool();
  {
    std::lock_guard<std::mutex> lock(pl.mutex);
    Pool::PerDevice& d = pl.devices[device];
    // The smallest block that fits and wastes at most a quarter (small ones:
    // up to a MiB).
    const size_t most = need + need / 4 + (size_t(1) << 20);
    for (auto it = d.blocks.lower_bound(need); it != d.blocks.end() && it->first <= most; ++it) {
      if (it->second.tag != nullptr && it->second.tag != tag) continue;
      PoolBlock b = it->second;
      d.blocks.erase(it);
      d.bytes -= b.bytes;
      b.tag = tag;
      return b;
    }
  }
  PoolBlock b;
  b.bytes = need;
  b.device = device;
  b.tag = tag;
  b.p = device_alloc(need, device);
  return b;
}

void pool_give(const PoolBlock& block) {
  Pool& pl = pool();
  std::vector<void*> out;  // freed without the lock: hipFree waits for the device
  {
    std::lock_guard<std::mutex> lock(pl.mutex);
    Pool::PerDevice& d = pl.devices[block.device];
    bool keep = true;
    if (d.bytes + block.bytes > kPoolBytes) {
      size_t settled = 0;
      for (const auto& kv : d.blocks) settled += kv.second.tag == nullptr ? kv.first : 0;
      keep = d.bytes - settled + block.bytes <= kPoolBytes;
    }
    while (keep && d.bytes + block.bytes > kPoolBytes) {
      auto oldest = d.blocks.end();
      for (auto it = d.blocks.begin(); it != d.blocks.end(); ++it) {
        if (it->second.tag != nullptr) continue;
        if (oldest == d.blocks.end() || it->second.given < oldest->second.given) oldest = it;
      }
      out.push_back(oldest->second.p);
      d.bytes -= oldest->first;
      d.blocks.erase(oldest);
    }
    if (keep) {
      PoolBlock kept = block;
      kept.given = ++d.returns;
      d.blocks.emplace(kept.bytes, kept);
      d.bytes += kept.bytes;
    } else {
      out.push_back(block.p);
    }
  }
  for (void* p : out) (void)hipFree(p);
}

void pool_settle(int device, hipStream_t tag) {
  Pool& pl = pool();
  std::lock_guard<std::mutex> lock(pl.mutex);
  for (auto& kv : pl.devices[device].blocks) {
    if (kv.second.tag == tag) kv.second.tag = nullptr;
  }
}

void pool_drop(int device, hipStream_t tag) {
  std::vector<PoolBlock> dropped;
  {
    Pool& pl = pool();
    std::lock_guard<std::mutex> lock(pl.mutex);
    Pool::PerDevice& d = pl.devices[device];
    for (auto it = d.blocks.begin(); it != d.blocks.end();) {
      if (it->second.tag == tag) {
        dropped.push_back(it->second);
        d.bytes -= it->second.bytes;
        it = d.blocks.erase(it);
      } else {
        ++it;
      }
    }
  }
  for (const PoolBlock& b : dropped) (void)hipFree(b.p);
}

}  // namespace kodama_hip
