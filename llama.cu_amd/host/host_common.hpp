// Internal helpers of the host layer.
#pragma once
#include <signal.h>
#include <stdio.h>

#include <chrono>
#include <mutex>
#include <thread>
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

// What the last launch of a one-token step leaves in page-locked memory, none of it ever -1, is watched for instead of waiting for the stream: expect()
// before the launch, await() for the words.  hipStreamSynchronize returns 5 to 10 us after the word is there (a graph of 11 small launches
// 36.7 us with it and 26.5 so, of 36 launches 76.5 and 68.6).  Calls of several tokens wait for the stream: whoever waits for it again afterwards, as
// clear_tokens does, pays for that wait then (requests of one prompt of 512 tokens, width 512, 174 us with the watch, 150 without).  The words say
// nothing of what else the call's launches wrote: that is read behind them on the same stream, or on another behind a wait for this one; what they
// read (page-locked input, a graph's arguments) is released or freed behind such a wait too.
// A watching thread is as busy as one in hipStreamSynchronize, which looks at the stream's signal all the while (1.2 cores either way), but gives its
// core up to any other thread between two looks.  A launch that takes longer than `patience`, or failed, is left to the stream's own wait and its error.
class awaited_words {
 public:
  awaited_words(pinned_buffer const& words, size_t count) : at_(static_cast<int*>(words.data())), count_(count) {}
  void expect() const {
    for (size_t i = 0; i < count_; ++i) __atomic_store_n(at_ + i, -1, __ATOMIC_RELAXED);
    __atomic_thread_fence(__ATOMIC_SEQ_CST);
  }
  void await(void* stream) const {
    using clock = std::chrono::steady_clock;
    constexpr auto patience = std::chrono::milliseconds(20);  // steps of 2.6 ms still gain 7 us (0.3 %)
    const auto until = clock::now() + patience;
    size_t i = 0;
    do {
      while (i < count_ && __atomic_load_n(at_ + i, __ATOMIC_ACQUIRE) != -1) ++i;
      if (i == count_) return;
      std::this_thread::yield();
    } while (clock::now() < until);
    LCU_CHECK(lcu_sync(stream));
  }

 private:
  int* at_;
  size_t count_;
};

inline size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }
inline size_t round_up(size_t a, size_t b) { return ceil_div(a, b) * b; }
}  // namespace llama_cu
