// An exception must not leave a parallel region (the process would end): the
// iterations of a loop run through this, and its first exception is thrown
// again after the region.
#pragma once

#include <exception>
#include <mutex>

namespace kodama_hip {

class LoopErrors {
 public:
  template <class F>
  void run(F&& body) noexcept {
    try {
      body();
    } catch (...) {
      std::lock_guard<std::mutex> lock(mutex_);
      if (!first_) first_ = std::current_exception();
    }
  }
  void rethrow() const {
    if (first_) std::rethrow_exception(first_);
  }

 private:
  std::mutex mutex_;
  std::exception_ptr first_;
};

}  // namespace kodama_hip
