#include "hip_on_host.hpp"

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <condition_variable>
#include <mutex>

namespace onhost {
std::function<bool(const char*)> refuse;
namespace {
std::mutex mu;
std::condition_variable cv;
thread_local int device = 0;
struct Stream {
  int device = 0;
  bool held = false;
};
struct Event {
  int device = 0;
  Stream* on = nullptr;
};
Stream* of(hipStream_t st) { return (Stream*) st; }
Event* of(hipEvent_t e) { return (Event*) e; }
bool refused(const char* name) { return refuse && refuse(name); }
void wait(Stream* s) {
  std::unique_lock<std::mutex> lk(mu);
  cv.wait(lk, [&] { return !s || !s->held; });
}
}  // namespace
void hold(hipStream_t st, bool on) {
  std::lock_guard<std::mutex> lk(mu);
  of(st)->held = on;
  cv.notify_all();
}
}  // namespace onhost
using namespace onhost;

#define ASK \
  if (refused(__func__)) return hipErrorUnknown

extern "C" {
int hydro_amd_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vfprintf(stderr, fmt, ap);
  va_end(ap);
  fputc('\n', stderr);
  return -1;
}

hipError_t hipMalloc(void** p, size_t n) {
  ASK;
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) {
  ASK;
  return hipMalloc(p, n);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ASK;
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) { return hipFree(p); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  ASK;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  ASK;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t) {
  ASK;
  for (size_t r = 0; r < h; r++) memcpy((char*) d + r * dp, (const char*) s + r * sp, w);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  ASK;
  memset(p, v, n);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  device = d;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* st, unsigned) {
  ASK;
  Stream* s = new Stream;
  s->device = device;
  *st = (hipStream_t) s;
  return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t st, hipDevice_t* d) {
  ASK;
  *d = of(st)->device;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t st) {
  delete of(st);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  ASK;
  wait(of(st));
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  ASK;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  ASK;
  Event* v = new Event;
  v->device = device;
  *e = (hipEvent_t) v;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  ASK;
  return hipEventCreateWithFlags(e, 0);
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete of(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  ASK;
  if (st && of(e)->device != of(st)->device) return hipErrorInvalidHandle;
  of(e)->on = of(st);
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  ASK;
  wait(of(e)->on);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  ASK;
  *ms = 1.0f;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t*, int) { return hipErrorNotSupported; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
// (nothing is captured here)
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return hipErrorNotSupported;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
}
