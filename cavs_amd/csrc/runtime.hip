// Runtime services of the C ABI: device memory, copies, streams, events, fills.
#include "common.h"

#include <cstring>
#include <mutex>
#include <set>

namespace cavs {

static thread_local char g_err[512] = "";
static int g_cus = 0;

int set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

LaunchProbe &launch_probe() {
  static thread_local LaunchProbe probe;
  return probe;
}

int num_cus() {
  if (g_cus == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      g_cus = prop.multiProcessorCount;
    if (g_cus <= 0) g_cus = 256;
  }
  return g_cus;
}

namespace {
constexpr int kOrderDevices = 64;
struct ResidentState {
  std::mutex m;                     // held around every ordered launch
  std::set<hipStream_t> own;        // streams of cavs_stream_create: known to live until stream_gone
  struct PerDevice {
    hipStream_t last = nullptr;     // stream of the last ordered launch (null: none, or it is over)
    hipEvent_t ev = nullptr;
    bool recorded = false;          // ev stands behind that launch
  } dev[kOrderDevices];
};
ResidentState &resident_state() {
  static ResidentState *s = new ResidentState;  // (outlives every static destructor)
  return *s;
}
bool mark(ResidentState::PerDevice &d) {
  if (!d.ev && hipEventCreateWithFlags(&d.ev, hipEventDisableTiming) != hipSuccess) return false;
  if (hipEventRecord(d.ev, d.last) != hipSuccess) return false;
  return d.recorded = true;
}
}  // namespace

ResidentOrder::ResidentOrder(hipStream_t stream) : stream_(stream) {
  ResidentState &s = resident_state();
  s.m.lock();
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipGetDevice(&dev_) != hipSuccess || dev_ < 0 || dev_ >= kOrderDevices) {
    rc_ = set_error(CAVS_EHIP, "ordering a resident launch: no usable device");
    return;
  }
  captured_ = stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
  if (captured_) return;
  ResidentState::PerDevice &d = s.dev[dev_];
  if (!d.last || d.last == stream) return;
  if ((!d.recorded && !mark(d)) || hipStreamWaitEvent(stream, d.ev, 0) != hipSuccess)
    rc_ = set_error(CAVS_EHIP, "ordering a resident launch behind another stream's: %s", hipGetErrorString(hipGetLastError()));
}

ResidentOrder::~ResidentOrder() {
  ResidentState &s = resident_state();
  if (rc_ == 0 && !captured_) {
    ResidentState::PerDevice &d = s.dev[dev_];
    d.last = stream_;
    d.recorded = false;
    if (!s.own.count(stream_)) (void)mark(d);  // a caller's stream may be gone before the next launch asks
  }
  s.m.unlock();
}

void ResidentOrder::stream_created(hipStream_t st) {
  ResidentState &s = resident_state();
  std::lock_guard<std::mutex> lock(s.m);
  s.own.insert(st);
}

void ResidentOrder::stream_gone(hipStream_t st) {
  ResidentState &s = resident_state();
  std::lock_guard<std::mutex> lock(s.m);
  s.own.erase(st);
  for (auto &d : s.dev)
    if (d.last == st) {
      if (!d.recorded) (void)hipStreamSynchronize(st);
      d.last = nullptr;
    }
}

void ResidentOrder::capture_begins(hipStream_t st) {
  ResidentState &s = resident_state();
  std::lock_guard<std::mutex> lock(s.m);
  for (auto &d : s.dev)
    if (d.last == st && !d.recorded) (void)mark(d);
}

__global__ void fill_kernel(float *p, float v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

__global__ void fill4_kernel(float4 *p, float v, size_t n4) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  float4 x = make_float4(v, v, v, v);
  for (; i < n4; i += stride) p[i] = x;
}

static int fill_impl(float *ptr, float value, size_t n, hipStream_t st) {
  if (n == 0) return CAVS_OK;
  size_t head = 0;
  // align to 16 bytes, then vector stores, then the tail
  while (head < n && !aligned16(ptr + head)) head++;
  if (head) {
    launch(fill_kernel, 1, 64, 0, st, ptr, value, head);
  }
  size_t n4 = (n - head) / 4;
  if (n4) {
    size_t blocks = (n4 + 255) / 256;
    size_t cap = (size_t)num_cus() * 8;
    launch(fill4_kernel, (unsigned)(blocks < cap ? blocks : cap), 256, 0, st, 
        reinterpret_cast<float4 *>(ptr + head), value, n4);
  }
  size_t done = head + n4 * 4;
  if (done < n) launch(fill_kernel, 1, 64, 0, st, ptr + done, value, n - done);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

}  // namespace cavs

using namespace cavs;

extern "C" {

const char *cavs_last_error(void) { return g_err; }
int cavs_abi_version(void) { return CAVS_ABI_VERSION; }

int cavs_init(int device) {
  CAVS_HIP_TRY(hipSetDevice(device));
  g_cus = 0;
  num_cus();
  // The entry point that allocates nothing finds its scratch here, with this device current.  A
  // device on which the lookup fails keeps everything else: that entry point reports it.
  (void)static_scratch_setup(nullptr);
  return CAVS_OK;
}

int cavs_device_name(char *buf, size_t len) {
  CAVS_REQUIRE(buf && len > 0, "cavs_device_name: null buffer");
  int dev = 0;
  hipDeviceProp_t prop;
  CAVS_HIP_TRY(hipGetDevice(&dev));
  CAVS_HIP_TRY(hipGetDeviceProperties(&prop, dev));
  snprintf(buf, len, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
  return CAVS_OK;
}

int cavs_device_bus_id(int device, char *buf, size_t len) {
  CAVS_REQUIRE(buf && len >= 13, "cavs_device_bus_id: a buffer of 13 bytes needed");
  CAVS_HIP_TRY(hipDeviceGetPCIBusId(buf, (int)len, device));
  return CAVS_OK;
}

int cavs_malloc(void **ptr, size_t bytes) {
  CAVS_REQUIRE(ptr, "cavs_malloc: null out pointer");
  *ptr = nullptr;
  if (bytes == 0) return CAVS_OK;
  hipError_t e = hipMalloc(ptr, bytes);
  if (e == hipErrorOutOfMemory) return set_error(CAVS_ENOMEM, "hipMalloc(%zu) out of memory", bytes);
  CAVS_HIP_TRY(e);
  return CAVS_OK;
}

int cavs_free(void *ptr) {
  if (ptr) CAVS_HIP_TRY(hipFree(ptr));
  return CAVS_OK;
}

int cavs_host_alloc(void **ptr, size_t bytes) {
  CAVS_REQUIRE(ptr, "cavs_host_alloc: null out pointer");
  *ptr = nullptr;
  if (bytes == 0) return CAVS_OK;
  CAVS_HIP_TRY(hipHostMalloc(ptr, bytes, hipHostMallocDefault));
  return CAVS_OK;
}

int cavs_host_free(void *ptr) {
  if (ptr) CAVS_HIP_TRY(hipHostFree(ptr));
  return CAVS_OK;
}

int cavs_memcpy_h2d(void *dst, const void *src, size_t bytes, void *stream) {
  if (bytes == 0) return CAVS_OK;
  CAVS_REQUIRE(dst && src, "cavs_memcpy_h2d: null pointer");
  CAVS_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
  return CAVS_OK;
}

int cavs_memcpy_d2h(void *dst, const void *src, size_t bytes, void *stream) {
  if (bytes == 0) return CAVS_OK;
  CAVS_REQUIRE(dst && src, "cavs_memcpy_d2h: null pointer");
  CAVS_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
  return CAVS_OK;
}

int cavs_memcpy_d2d(void *dst, const void *src, size_t bytes, void *stream) {
  if (bytes == 0) return CAVS_OK;
  CAVS_REQUIRE(dst && src, "cavs_memcpy_d2d: null pointer");
  CAVS_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
  return CAVS_OK;
}

int cavs_zero(void *ptr, size_t bytes, void *stream) {
  if (bytes == 0) return CAVS_OK;
  CAVS_REQUIRE(ptr && bytes % 4 == 0 && (reinterpret_cast<uintptr_t>(ptr) & 3u) == 0,
               "cavs_zero: pointer and size must be multiples of 4 bytes");
  return fill_impl(static_cast<float *>(ptr), 0.f, bytes / 4, as_stream(stream));
}

int cavs_fill(float *ptr, float value, size_t n, void *stream) {
  if (n == 0) return CAVS_OK;
  CAVS_REQUIRE(ptr, "cavs_fill: null pointer");
  return fill_impl(ptr, value, n, as_stream(stream));
}

int cavs_stream_create(void **stream) {
  CAVS_REQUIRE(stream, "cavs_stream_create: null out pointer");
  hipStream_t s;
  CAVS_HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  *stream = s;
  ResidentOrder::stream_created(s);
  return CAVS_OK;
}

int cavs_stream_destroy(void *stream) {
  if (stream) {
    ResidentOrder::stream_gone(as_stream(stream));
    CAVS_HIP_TRY(hipStreamDestroy(as_stream(stream)));
  }
  return CAVS_OK;
}

int cavs_stream_sync(void *stream) {
  CAVS_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
  return CAVS_OK;
}

int cavs_event_create(void **event) {
  CAVS_REQUIRE(event, "cavs_event_create: null out pointer");
  hipEvent_t e;
  CAVS_HIP_TRY(hipEventCreate(&e));
  *event = e;
  return CAVS_OK;
}

int cavs_event_create_device(void **event) {
  CAVS_REQUIRE(event, "cavs_event_create_device: null out pointer");
  hipEvent_t e;
  CAVS_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableSystemFence));
  *event = e;
  return CAVS_OK;
}

int cavs_event_destroy(void *event) {
  if (event) CAVS_HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)));
  return CAVS_OK;
}

int cavs_event_record(void *event, void *stream) {
  CAVS_REQUIRE(event, "cavs_event_record: null event");
  CAVS_HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)));
  return CAVS_OK;
}

int cavs_stream_wait_event(void *stream, void *event) {
  CAVS_REQUIRE(event, "cavs_stream_wait_event: null event");
  CAVS_HIP_TRY(hipStreamWaitEvent(as_stream(stream), static_cast<hipEvent_t>(event), 0));
  return CAVS_OK;
}

int cavs_event_sync(void *event) {
  CAVS_REQUIRE(event, "cavs_event_sync: null event");
  CAVS_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(event)));
  return CAVS_OK;
}

int cavs_event_elapsed_ms(float *ms, void *start, void *stop) {
  CAVS_REQUIRE(ms && start && stop, "cavs_event_elapsed_ms: null argument");
  CAVS_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(stop)));
  CAVS_HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
  return CAVS_OK;
}

int cavs_graph_capture_begin(void *stream) {
  CAVS_REQUIRE(stream, "cavs_graph_capture_begin: the default stream cannot be captured");
  ResidentOrder::capture_begins(as_stream(stream));
  // relaxed: other threads of the process (an allocator, another session) may go on calling the runtime
  CAVS_HIP_TRY(hipStreamBeginCapture(as_stream(stream), hipStreamCaptureModeRelaxed));
  return CAVS_OK;
}

int cavs_graph_capture_end(void *stream, void **graph_exec) {
  CAVS_REQUIRE(stream, "cavs_graph_capture_end: null stream");
  hipGraph_t graph = nullptr;
  const hipError_t rc = hipStreamEndCapture(as_stream(stream), &graph);
  if (!graph_exec) {  // the caller gives the capture up
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    // (an invalidated capture is supposed to end here; if the stream is still in it, say so)
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(as_stream(stream), &status) != hipSuccess || status != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      return cavs::set_error(CAVS_EHIP, "cavs_graph_capture_end: the stream is still in a capture (%s, status %d)", hipGetErrorString(rc),
                             (int)status);
    }
    return CAVS_OK;
  }
  *graph_exec = nullptr;
  if (rc != hipSuccess || !graph) {
    (void)hipGetLastError();
    if (graph) (void)hipGraphDestroy(graph);
    return cavs::set_error(CAVS_EHIP, "cavs_graph_capture_end: the capture was invalidated (%s)", hipGetErrorString(rc));
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t ri = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (ri != hipSuccess) {
    (void)hipGetLastError();
    return cavs::set_error(CAVS_EHIP, "cavs_graph_capture_end: hipGraphInstantiate: %s", hipGetErrorString(ri));
  }
  *graph_exec = exec;
  return CAVS_OK;
}

int cavs_graph_launch(void *graph_exec, void *stream) {
  CAVS_REQUIRE(graph_exec, "cavs_graph_launch: null graph");
  ResidentOrder order(as_stream(stream));  // (it may hold such launches)
  if (order.rc()) return order.rc();
  CAVS_HIP_TRY(hipGraphLaunch(static_cast<hipGraphExec_t>(graph_exec), as_stream(stream)));
  return CAVS_OK;
}

int cavs_graph_destroy(void *graph_exec) {
  if (graph_exec) CAVS_HIP_TRY(hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph_exec)));
  return CAVS_OK;
}

int cavs_profile_arm(void *start_event, void *stop_event) {
  CAVS_REQUIRE(start_event && stop_event, "cavs_profile_arm: null event");
  LaunchProbe &p = launch_probe();
  p.start = static_cast<hipEvent_t>(start_event);
  p.stop = static_cast<hipEvent_t>(stop_event);
  p.armed = true;
  p.started = false;
  return CAVS_OK;
}

int cavs_stop_event_arm(void *event) {
  CAVS_REQUIRE(event, "cavs_stop_event_arm: null event");
  LaunchProbe &p = launch_probe();
  p.start = nullptr;
  p.stop = static_cast<hipEvent_t>(event);
  p.armed = true;
  p.started = false;
  return CAVS_OK;
}

int cavs_profile_disarm(int *launched) {
  LaunchProbe &p = launch_probe();
  if (launched) *launched = p.armed && p.started;
  p = LaunchProbe{};
  return CAVS_OK;
}

}  // extern "C"
