// MADV_POPULATE_WRITE in a few threads (Linux 5.14; elsewhere a no-op).
#include "host_pages.h"

#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <cstdint>
#include <system_error>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace kodama_hip {

namespace {
constexpr size_t kSmall = size_t(4) << 20;
constexpr size_t kPart = size_t(16) << 20;  // bytes per thread at least
constexpr size_t kMaxThreads = 4;           // per buffer
}  // namespace

void PageWarmer::add(void* p, size_t bytes) {
  if (p == nullptr || bytes < kSmall) return;
  const size_t page = static_cast<size_t>(sysconf(_SC_PAGESIZE));
  const uintptr_t begin = (reinterpret_cast<uintptr_t>(p) + page - 1) / page * page;
  const uintptr_t end = (reinterpret_cast<uintptr_t>(p) + bytes) / page * page;
  const size_t parts = std::min(kMaxThreads, std::max<size_t>(1, bytes / kPart));
  const size_t step = ((end - begin) / parts + page - 1) / page * page;
  for (uintptr_t at = begin; at < end; at += step) {
    const size_t len = std::min<size_t>(step, end - at);
    try {
      threads_.emplace_back([at, len] { (void)madvise(reinterpret_cast<void*>(at), len, MADV_POPULATE_WRITE); });
    } catch (const std::system_error&) {
      return;  // no thread to spare: the download faults its pages in
    }
  }
}

void PageWarmer::wait() {
  for (std::thread& t : threads_) t.join();
  threads_.clear();
}

}  // namespace kodama_hip
