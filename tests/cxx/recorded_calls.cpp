// The device functions of llama_cu_hip.h without a device: they note their name and stream and succeed.  Loaded in front of the library they stand in for
// its own, so that the host layer's calls can be looked at.  Device memory is addresses that nobody follows; page-locked memory is memory.
// A call's last launch leaves its token (7) and count (0) at once, or when its stream is waited for, `lateness` us after the wait began.
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <map>
#include <utility>
#include <vector>

#include "llama_cu_hip.h"

namespace {
struct noted {
  const char* name;
  void* stream;
};
std::vector<noted> calls;
std::vector<std::pair<int*, int>> answers, of_graph;
bool capturing = false;
long lateness = -1;
std::map<void*, size_t> weights;
size_t next_address = 4096;

int note(const char* name, void* stream) {
  if (!capturing) calls.push_back({name, stream});
  return 0;
}
void leave_answers() {
  for (auto& [at, count] : answers) {
    for (int i = 0; i < count; ++i) __atomic_store_n(at + i, i == 1 && count == 2 ? 0 : 7, __ATOMIC_RELEASE);
  }
  answers.clear();
}
void answer(void* at, int count) {
  (capturing ? of_graph : answers).push_back({(int*)at, count});
  if (!capturing && lateness < 0) leave_answers();
}
}  // namespace

extern "C" {
void recorded_lateness(long us) { lateness = us; }
void recorded_clear() { calls.clear(); }
int recorded_count() { return (int)calls.size(); }
const char* recorded_name(int i) { return calls[i].name; }
void* recorded_stream(int i) { return calls[i].stream; }

size_t recorded_weights(void* stream) { return weights.count(stream) ? weights[stream] : 0; }

const char* lcu_last_error(void) { return ""; }
int lcu_malloc(void** out, size_t bytes) {
  *out = (void*)next_address;
  next_address += (bytes + 4095) / 4096 * 4096 + 4096;
  return 0;
}
int lcu_host_alloc(void** out, size_t bytes) {
  *out = calloc(1, bytes + 16);
  return 0;
}
int lcu_host_free(void* p) {
  free(p);
  return 0;
}
int lcu_stream_create(void** out) { return lcu_malloc(out, 1); }
int lcu_device_get_props(int, lcu_device_props* p) {
  memset(p, 0, sizeof(*p));
  p->compute_units = 256;
  return 0;
}
int lcu_stream_weights(void* stream, size_t bytes) {
  weights[stream] = bytes;
  return 0;
}
int lcu_sync_timeouts(void*, unsigned* out) {
  *out = 0;
  return 0;
}
int lcu_graph_begin_capture(void*) {
  capturing = true;
  of_graph.clear();
  return 0;
}
int lcu_graph_end_capture(void*, void** out) {
  capturing = false;
  return lcu_malloc(out, 1);
}
int lcu_graph_launch(void*, void* stream) {
  for (auto& a : of_graph) answer(a.first, a.second);
  return note("lcu_graph_launch", stream);
}
int lcu_sync(void* stream) {
  if (!answers.empty()) {
    usleep((useconds_t)(lateness > 0 ? lateness : 0));
    leave_answers();
  }
  return note("lcu_sync", stream);
}
int lcu_softmax_argmax_status(void*, void* out, const void*, int, float, void* stream) {
  answer(out, 2);
  return note("lcu_softmax_argmax_status", stream);
}
int lcu_softmax_argmax_rows(void*, void* out, const void*, int rows, int, float, void* stream) {
  answer(out, rows);
  return note("lcu_softmax_argmax_rows", stream);
}
#include "other_calls.inc"  // every other function of the header
}
