// A stand-in for the device behind the host runtime: memory is the host's, copies and fills happen at once, kernels do nothing
// (their entry points, which return 0, are written beside this file from the declared ones).  It watches what a runtime
// may be asked and when, and keeps a line for everything that may not be: a wait for a stream that is being recorded, a recorded
// graph given back while a launch of it may be under way or after the stream it was launched on.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

#include "cavs_hip.h"

namespace {
uintptr_t g_next = 16;
std::set<void *> g_streams;
std::map<void *, void *> g_launched;  // graph -> the stream of its last launch
std::set<void *> g_under_way;         // graphs whose last launch nobody has waited for
void *g_recording = nullptr;
std::string g_faults;
int g_recorded = 0, g_replayed = 0;

void *handle() { return reinterpret_cast<void *>(g_next += 16); }
void fault(const char *what) { g_faults += std::string(what) + "\n"; }
int waited(void *stream) {
  if (stream == g_recording && stream) {
    fault("a wait for the stream that is being recorded");
    return CAVS_EHIP;
  }
  for (auto it = g_under_way.begin(); it != g_under_way.end();) it = g_launched[*it] == stream ? g_under_way.erase(it) : std::next(it);
  return CAVS_OK;
}
}  // namespace

extern "C" {
const char *standin_faults() { return g_faults.c_str(); }
int standin_recorded() { return g_recorded; }
int standin_replayed() { return g_replayed; }

const char *cavs_last_error(void) { return "the stand-in refused"; }
int cavs_malloc(void **p, size_t n) {
  *p = n ? aligned_alloc(256, (n + 255) / 256 * 256) : nullptr;
  if (*p) std::memset(*p, 0, n);
  return CAVS_OK;
}
int cavs_free(void *p) {
  std::free(p);
  return CAVS_OK;
}
int cavs_host_alloc(void **p, size_t n) { return cavs_malloc(p, n); }
int cavs_host_free(void *p) { return cavs_free(p); }
int cavs_memcpy_h2d(void *d, const void *s, size_t n, void *) {
  std::memcpy(d, s, n);
  return CAVS_OK;
}
int cavs_memcpy_d2h(void *d, const void *s, size_t n, void *) { return cavs_memcpy_h2d(d, s, n, nullptr); }
int cavs_memcpy_d2d(void *d, const void *s, size_t n, void *) { return cavs_memcpy_h2d(d, s, n, nullptr); }
int cavs_zero(void *p, size_t n, void *) {
  std::memset(p, 0, n);
  return CAVS_OK;
}
int cavs_stream_create(void **s) {
  g_streams.insert(*s = handle());
  return CAVS_OK;
}
int cavs_stream_destroy(void *s) {
  if (s && !g_streams.erase(s)) fault("a stream is given back twice");
  return waited(s);
}
int cavs_stream_sync(void *s) { return waited(s); }
int cavs_event_create(void **e) {
  *e = handle();
  return CAVS_OK;
}
int cavs_event_create_device(void **e) { return cavs_event_create(e); }
int cavs_graph_capture_begin(void *s) {
  g_recording = s;
  return CAVS_OK;
}
int cavs_graph_capture_end(void *, void **exec) {
  g_recording = nullptr;
  if (!exec) return CAVS_OK;
  g_launched[*exec = handle()] = nullptr;
  g_recorded++;
  return CAVS_OK;
}
int cavs_graph_launch(void *exec, void *s) {
  g_launched[exec] = s;
  g_under_way.insert(exec);
  g_replayed++;
  return CAVS_OK;
}
int cavs_graph_destroy(void *exec) {
  auto it = g_launched.find(exec);
  if (it == g_launched.end()) {
    fault("a graph is given back twice");
    return CAVS_OK;
  }
  if (it->second && !g_streams.count(it->second)) fault("a graph is given back after the stream it was launched on");
  if (g_under_way.erase(exec)) fault("a graph is given back while a launch of it may be under way");
  g_launched.erase(it);
  return CAVS_OK;
}
int cavs_profile_disarm(int *launched) {
  if (launched) *launched = 0;
  return CAVS_OK;
}
}
