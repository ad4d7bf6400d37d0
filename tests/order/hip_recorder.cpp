// Stands in for the HIP runtime in CPU tests of stream ordering: it runs
// nothing, and records for every operation that the library enqueues (kernel
// or copy) which earlier operations it follows by its stream and the events
// that stream has waited for.  Loaded with RTLD_GLOBAL before the library, in
// a process of its own without torch, so that the library's calls come here.
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <map>
#include <set>
#include <string>
#include <vector>

namespace {

typedef std::set<int> Ops;

struct Op {
  std::string name;
  Ops after;
};

std::vector<Op> g_ops;
std::map<void*, Ops> g_streams, g_events;
std::map<void*, bool> g_capturing;
std::map<const void*, std::string> g_names;
std::map<uintptr_t, size_t> g_pinned;
Ops g_host;            // operations the host has waited for
int g_unwaited = 0;    // operations not waited for when device memory was first freed
bool g_freed = false;
uintptr_t g_next = uintptr_t(1) << 40;

void* make(size_t bytes) {
  void* p = reinterpret_cast<void*>(g_next);
  g_next += (bytes + 4095) / 4096 * 4096;
  return p;
}

void add(const std::string& name, hipStream_t stream) {
  Ops& s = g_streams[stream];
  g_ops.push_back(Op{name, s});
  s.insert(static_cast<int>(g_ops.size()) - 1);
}

}  // namespace

extern "C" {

// ---------------------------------------------------------------- the test's side
int rec_count(void) { return static_cast<int>(g_ops.size()); }
const char* rec_name(int op) { return g_ops[op].name.c_str(); }
int rec_follows(int op, int earlier) { return static_cast<int>(g_ops[op].after.count(earlier)); }
int rec_stream_follows(void* stream, int op) { return static_cast<int>(g_streams[stream].count(op)); }
int rec_unwaited_at_free(void) { return g_freed ? g_unwaited : -1; }
void rec_pinned(void* p, int64_t bytes) { g_pinned[reinterpret_cast<uintptr_t>(p)] = static_cast<size_t>(bytes); }
void rec_capture(void* stream, int on) { g_capturing[stream] = on != 0; }

// ---------------------------------------------------------------- the runtime's side
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(make(1)); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, void*, void*,
                           int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = make(n);
  return hipSuccess;
}
hipError_t hipFree(void*) {
  if (!g_freed) g_unwaited = static_cast<int>(g_ops.size() - g_host.size());
  g_freed = true;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) {
  *s = static_cast<hipStream_t>(make(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  g_host.insert(g_streams[s].begin(), g_streams[s].end());
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status) {
  *status = g_capturing[s] ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned int) {
  *e = static_cast<hipEvent_t>(make(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  g_events[e] = g_streams[s];
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  g_host.insert(g_events[e].begin(), g_events[e].end());
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int) {
  const Ops& before = g_events[e];
  g_streams[s].insert(before.begin(), before.end());
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind kind, hipStream_t s) {
  add(kind == hipMemcpyDeviceToHost ? "copy D2H" : "copy H2D", s);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3, dim3, void**, size_t, hipStream_t s) {
  add(g_names[fn], s);
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void* fn, dim3, dim3, void**, size_t, hipStream_t s, hipEvent_t, hipEvent_t stop,
                              int) {
  add(g_names[fn], s);
  if (stop != nullptr) g_events[stop] = g_streams[s];
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(p);
  auto it = g_pinned.upper_bound(at);
  if (it == g_pinned.begin()) return hipErrorInvalidValue;
  --it;
  if (at - it->first >= it->second) return hipErrorInvalidValue;
  a->type = hipMemoryTypeHost;
  a->devicePointer = const_cast<void*>(p);
  a->hostPointer = const_cast<void*>(p);
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* start, size_t* size, hipDeviceptr_t p) {
  auto it = g_pinned.upper_bound(reinterpret_cast<uintptr_t>(p));
  if (it == g_pinned.begin()) return hipErrorInvalidValue;
  --it;
  *start = reinterpret_cast<hipDeviceptr_t>(it->first);
  *size = it->second;
  return hipSuccess;
}

}  // extern "C"
