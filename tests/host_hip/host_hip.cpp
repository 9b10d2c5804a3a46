#include "host_hip.h"

#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>
#include <vector>

namespace {
typedef std::map<void *, size_t> Clock;  // stream -> launches known to be done before

struct Call {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
};
struct State {
  std::set<void *> memory;
  std::map<void *, Clock> streams, events;
  Clock host;
  std::vector<Call> calls;
  hipError_t last = hipSuccess;
  int graphs = 0;
};
State &state() {
  static State s;
  return s;
}
long malloc_left = -1, launch_left = -1, new_left = -1;
int inside = 0;  // the runtime's own allocations do not count
struct Inside {
  Inside() { inside++; }
  ~Inside() { inside--; }
};

// true when the armed countdown reaches its call
bool due(long *left) {
  if (*left < 0) return false;
  return (*left)-- == 0;
}
hipError_t ret(hipError_t e) {
  if (e != hipSuccess) state().last = e;
  return e;
}
void join(Clock *to, const Clock &from) {
  for (auto &e : from)
    if (e.second > (*to)[e.first]) (*to)[e.first] = e.second;
}
hipError_t launch(void *s) {
  Inside guard;
  if (due(&launch_left)) return ret(hipErrorLaunchFailure);
  state().streams[s][s]++;
  return hipSuccess;
}
template <class T>
T handle() {
  return reinterpret_cast<T>(std::malloc(1));
}
}  // namespace

void *operator new(size_t n) {
  if (!inside && due(&new_left)) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

namespace host_hip {
void fail_malloc(long n) { malloc_left = n; }
void fail_launch(long n) { launch_left = n; }
void fail_new(long n) { new_left = n; }
bool all_used() { return malloc_left < 0 && launch_left < 0 && new_left < 0; }
void clear_error() { state().last = hipSuccess; }
size_t live() { return state().memory.size(); }
size_t outstanding(void *stream) {
  Inside guard;
  Clock known = state().host;
  join(&known, state().streams[stream]);
  size_t n = 0;
  for (auto &s : state().streams) n += s.second[s.first] - known[s.first];
  return n;
}
}  // namespace host_hip

extern "C" {
char __hip_fatbin[64];
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  Inside guard;
  state().calls.push_back({g, b, m, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
  const Call c = state().calls.back();
  state().calls.pop_back();
  *g = c.grid;
  *b = c.block;
  *m = c.shmem;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s) {
  return launch(s);
}
hipError_t hipMalloc(void **p, size_t n) {
  Inside guard;
  if (due(&malloc_left)) return ret(hipErrorOutOfMemory);
  *p = std::calloc(n ? n : 1, 1);
  state().memory.insert(*p);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  if (!state().memory.erase(p)) std::abort();  // not ours, or freed before
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  Inside guard;
  std::memcpy(d, s, n);
  state().streams[st][st]++;
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return ret(hipErrorNotFound); }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = state().last;
  state().last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipDeviceSynchronize(void) {
  Inside guard;
  for (auto &s : state().streams) join(&state().host, s.second);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  Inside guard;
  join(&state().host, state().streams[s]);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
  *c = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  Inside guard;
  join(&state().streams[s], state().events[e]);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = handle<hipEvent_t>();
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  Inside guard;
  state().events[e] = state().streams[s];
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
// a captured stream's launches count as work: nothing outstanding is missed
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = handle<hipGraph_t>();
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *x = handle<hipGraphExec_t>();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return launch(s); }
}
