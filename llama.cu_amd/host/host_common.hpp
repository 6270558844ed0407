// Internal helpers of the host layer.
#pragma once
#include <signal.h>
#include <stdio.h>

#include <mutex>
#include <utility>

#include "llama_cu_hip.h"
#include "llama_cu_host.hpp"

// A failing device call is fatal, as the reference's CHECK_CUDA (llama_cu.h:48-56): print, raise.
#define LCU_CHECK(expr)                                                                              \
  do {                                                                                               \
    int lcu_status__ = (expr);                                                                       \
    if (lcu_status__ != 0) {                                                                         \
      fprintf(stderr, "%s(%d): gpu error %d: %s (source: " #expr ")\n", __func__, __LINE__,        \
              lcu_status__, lcu_last_error());                                                       \
      raise(SIGSEGV);                                                                                \
    }                                                                                                \
  } while (0)

#define RETURN_UNLESS(x) \
  if (!(x)) {            \
    return false;        \
  }

namespace llama_cu {
// Several host threads may drive contexts of one process.  Kernel launches and copies from several
// threads are everyday use of the runtime; what changes the device's set of streams, allocations
// and graphs is done by one thread at a time: stream creation and destruction, device allocation
// and release (both wait for the whole device), and everything about a graph (its capture runs in
// the capturing thread's own capture mode, and nobody allocates, frees or creates a stream under
// it; instantiation; launch; destruction).  Recursive: a context's constructor takes it around
// members that take it themselves.
inline std::recursive_mutex& device_structure_mutex() {
  static std::recursive_mutex m;
  return m;
}
using device_structure_lock = std::lock_guard<std::recursive_mutex>;

// Page-locked memory that launches read and write: what a step takes from the host and gives back.  A copy of a few bytes costs
// the host and the device more than a launch.
class pinned_buffer {
 public:
  pinned_buffer() {}
  explicit pinned_buffer(size_t size) : size_(size) {
    device_structure_lock lock(device_structure_mutex());
    LCU_CHECK(lcu_host_alloc(&ptr_, size));
  }
  pinned_buffer(pinned_buffer&& other) : ptr_(std::exchange(other.ptr_, nullptr)), size_(std::exchange(other.size_, 0)) {}
  pinned_buffer& operator=(pinned_buffer&& other) {
    std::swap(ptr_, other.ptr_);
    std::swap(size_, other.size_);
    return *this;
  }
  ~pinned_buffer() {
    if (ptr_) {
      device_structure_lock lock(device_structure_mutex());
      LCU_CHECK(lcu_host_free(ptr_));
    }
  }
  void* data() const { return ptr_; }
  size_t size() const { return size_; }

 private:
  void* ptr_{nullptr};
  size_t size_{0};
};

inline size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }
inline size_t round_up(size_t a, size_t b) { return ceil_div(a, b) * b; }
}  // namespace llama_cu
