// A stand-in for the HIP runtime on the host, so that the library's host code
// (streams, events, allocations, launches, error paths) runs without a GPU.
// Loaded before libocr.so with global symbols, it answers the library's HIP
// calls: memory is host memory (reserved, touched only when written), kernels
// are logged and not run, work is finished at once unless its stream is held.
//
// host_*: what the tests use.  The log has a line per call that matters:
//   launch <kernel> <stream>     record <event> <stream>
//   wait <stream> <event>        graph <stream>
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {

struct Stream {
  int id = 0;
  bool held = false, capturing = false;
};
struct Event {
  int id = 0;
  Stream* on = nullptr;   // the held stream it was recorded on
};

std::recursive_mutex g_mu;
#define LOCK std::lock_guard<std::recursive_mutex> lk(g_mu)
Stream g_null;
std::map<hipStream_t, Stream*> g_streams;
std::set<Event*> g_events;
std::map<const void*, std::string> g_kernels;
std::map<const void*, void*> g_vars;
std::map<void*, size_t> g_mem;
std::string g_log;
int g_next = 1, g_fail_launch = -1;
size_t g_room = ~(size_t)0, g_bytes = 0;
hipError_t g_last = hipSuccess;
struct { dim3 grid, block; size_t shared; hipStream_t st; } g_call;

Stream* at(hipStream_t s) { return s ? g_streams.at(s) : &g_null; }
void put(const char* what, const std::string& a, const std::string& b) {
  g_log += std::string(what) + " " + a + (b.empty() ? "" : " " + b) + "\n";
}
std::string num(int i) { return std::to_string(i); }
hipError_t bad(hipError_t e) { return g_last = e; }
void* reserve(size_t n) {
  void* p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : p;
}

}  // namespace

extern "C" {

const char* host_log() { return g_log.c_str(); }
void host_clear() { LOCK; g_log.clear(); }
// The n-th launch from now fails (0: the next); -1: none.
void host_fail_launch(int n) { g_fail_launch = n; }
// Device allocations that take more than `bytes` from now on fail.
void host_limit_device(size_t bytes) { g_room = bytes == ~(size_t)0 ? bytes : g_bytes + bytes; }
size_t host_device_bytes() { return g_bytes; }
int host_live_events() { return (int)g_events.size(); }
// A held stream's work is not finished until it is let go.
void host_hold(void* s, int on) {
  LOCK;
  Stream* st = at((hipStream_t)s);
  st->held = on != 0;
  if (!on)
    for (Event* e : g_events)
      if (e->on == st) e->on = nullptr;
}
void host_capture(void* s, int on) { LOCK; at((hipStream_t)s)->capturing = on != 0; }
int host_stream_id(void* s) { LOCK; return at((hipStream_t)s)->id; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_kernels[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { g_vars[var] = reserve(size); }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t st) {
  g_call = {grid, block, shared, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* st) {
  *grid = g_call.grid;
  *block = g_call.block;
  *shared = g_call.shared;
  *st = g_call.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t s) {
  LOCK;
  if (g_fail_launch == 0) {
    g_fail_launch = -1;
    return bad(hipErrorLaunchFailure);
  }
  if (g_fail_launch > 0) g_fail_launch--;
  put("launch", g_kernels.count(f) ? g_kernels[f] : "?", num(at(s)->id));
  return hipSuccess;
}
hipError_t hipGetLastError() { hipError_t e = g_last; g_last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "host stand-in error"; }

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) { *p = g_vars.at(sym); return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)288 << 30; return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
  LOCK;
  *p = g_bytes + n > g_room ? nullptr : reserve(n);
  if (!*p) return bad(hipErrorOutOfMemory);
  g_mem[*p] = n;
  g_bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  LOCK;
  if (!p) return hipSuccess;
  g_bytes -= g_mem.at(p);
  munmap(p, g_mem[p] ? g_mem[p] : 1);
  g_mem.erase(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return *p ? hipSuccess : bad(hipErrorOutOfMemory); }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) {
  if (v || n < ((size_t)1 << 30)) memset(p, v, n);   // fresh memory is zero
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  LOCK;
  Stream* st = new Stream;
  st->id = g_next++;
  *s = (hipStream_t)st;
  g_streams[*s] = st;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { LOCK; g_streams.erase(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { LOCK; (void)at(s); return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { LOCK; return at(s)->held ? bad(hipErrorNotReady) : hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  LOCK;
  put("wait", num(at(s)->id), num(((Event*)e)->id));
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
  LOCK;
  *c = at(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)&g_null; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = (hipGraphExec_t)&g_null;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { LOCK; put("graph", num(at(s)->id), ""); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  LOCK;
  Event* ev = new Event;
  ev->id = g_next++;
  g_events.insert(ev);
  *e = (hipEvent_t)ev;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { LOCK; g_events.erase((Event*)e); delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  LOCK;
  Event* ev = (Event*)e;
  ev->on = at(s)->held ? at(s) : nullptr;
  put("record", num(ev->id), num(at(s)->id));
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { LOCK; return ((Event*)e)->on ? bad(hipErrorNotReady) : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }

}  // extern "C"
