// A model of the part of the HIP runtime that the library's host code uses:
// streams, events and graphs as host objects, kernels and copies as nothing.
// Linked instead of the runtime, it lets host code run without a device and
// counts what a device would get wrong only now and then:
//   foreign waits   a thread waits for an event that another thread recorded
//                   after it;
//   busy releases   a graph or stream is destroyed while launched work on it
//                   has not been waited for.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <thread>

#include "runtime.hpp"

struct ihipStream_t {
  std::set<hipGraphExec *> busy;  // launched here and not waited for
  std::set<ihipStream_t *> after;
};
struct ihipEvent_t {
  std::thread::id by;
  ihipStream_t *on = nullptr;
  int records = 0;
};
struct ihipGraph {
  int nodes = 1;
};
struct hipGraphExec {
  int launches = 0;
};

namespace {
std::mutex mu;
std::condition_variable cv;
Model m;
std::set<ihipStream_t *> streams;

void wait_for(ihipStream_t *s) {
  for (hipGraphExec *e : s->busy) e->launches = 0;
  for (ihipStream_t *t : streams)
    if (t != s)
      for (hipGraphExec *e : s->busy) t->busy.erase(e);
  s->busy.clear();
}
ihipStream_t *known(ihipStream_t *s) {
  static ihipStream_t null_stream;
  if (!s) s = &null_stream;
  streams.insert(s);
  return s;
}
}  // namespace

Model &model() { return m; }
hipStream_t model_stream() { return new ihipStream_t; }

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) {
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) {
  return *s = new ihipStream_t, hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> l(mu);
  if (!known(s)->busy.empty()) ++m.busy_releases;
  streams.erase(s);
  delete s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> l(mu);
  wait_for(known(s));
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  std::lock_guard<std::mutex> l(mu);
  for (ihipStream_t *s : std::set<ihipStream_t *>(streams)) wait_for(s);
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = new ihipGraph, hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::unique_lock<std::mutex> l(mu);
  e->by = std::this_thread::get_id();
  e->on = known(s);
  const int mine = ++e->records;
  cv.notify_all();
  // let another thread record the same event now, if it can
  if (m.yield_ms > 0)
    cv.wait_for(l, std::chrono::milliseconds(m.yield_ms), [&] { return e->records != mine; });
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned int) {
  std::lock_guard<std::mutex> l(mu);
  ++m.waits;
  if (e->by != std::this_thread::get_id()) ++m.foreign_waits;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> l(mu);
  if (e->on) wait_for(e->on);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return *x = reinterpret_cast<hipGraphExec_t>(new hipGraphExec), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  std::lock_guard<std::mutex> l(mu);
  auto *e = reinterpret_cast<hipGraphExec *>(x);
  ++e->launches;
  ++m.launches;
  known(s)->busy.insert(e);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  std::lock_guard<std::mutex> l(mu);
  auto *e = reinterpret_cast<hipGraphExec *>(x);
  if (e->launches) ++m.busy_releases;
  for (ihipStream_t *t : streams) t->busy.erase(e);
  delete e;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete g, hipSuccess; }

// kernel launches and the registration of device code
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned int, void *, void *,
                           void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}
