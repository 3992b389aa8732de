// A stand-in for the HIP runtime that runs nothing: memory is the host's, copies
// happen at once, kernels not at all, an event has happened at its first or
// second query.  For the host logic of the served form, whose waits it can
// make endless: with STUB_STALL=event events recorded after the first
// STUB_AFTER never happen, with STUB_STALL=sync synchronisations and copies to
// the host after the first STUB_AFTER synchronisations do not return.
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <thread>

typedef int E;
typedef void* P;
struct Dim {
  unsigned x, y, z;
};
struct Event {
  std::atomic<int> state{0};  // 0 never recorded, 1 and 2 recorded, 3 happened, -1 never will
};

static bool stalls(const char* what, long n) {
  static const char* kind = getenv("STUB_STALL");
  static const long after = getenv("STUB_AFTER") ? atol(getenv("STUB_AFTER")) : 0;
  return kind && !strcmp(kind, what) && n >= after;
}
static void wait() {
  static std::atomic<long> n{0};
  if (stalls("sync", n++))
    for (;;) std::this_thread::sleep_for(std::chrono::seconds(1));
}

extern "C" {
E __hipPopCallConfiguration(Dim* g, Dim* b, size_t* s, P* st) {
  *g = *b = Dim{1, 1, 1};
  *s = 0;
  *st = nullptr;
  return 0;
}
E __hipPushCallConfiguration(Dim, Dim, size_t, P) { return 0; }
P* __hipRegisterFatBinary(const void*) {
  static P x;
  return &x;
}
void __hipRegisterFunction(P*, const void*, char*, const char*, unsigned, P, P, P, P, int*) {}
void __hipRegisterVar(P*, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(P*) {}
E hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
E hipDeviceSynchronize() {
  wait();
  return 0;
}
E hipEventCreate(P* e) {
  *e = new Event;
  return 0;
}
E hipEventCreateWithFlags(P* e, unsigned) { return hipEventCreate(e); }
E hipEventDestroy(P e) {
  delete static_cast<Event*>(e);
  return 0;
}
E hipEventElapsedTime(float* f, P, P) {
  *f = 1.0f;
  return 0;
}
E hipEventRecord(P e, P) {
  static std::atomic<long> n{0};
  static_cast<Event*>(e)->state = stalls("event", n++) ? -1 : 1;
  return 0;
}
E hipEventQuery(P e) {
  std::atomic<int>& s = static_cast<Event*>(e)->state;
  if (s == -1) return 600;  // not ready
  if (s == 1) {
    s = 2;
    return 600;
  }
  s = 3;
  return 0;
}
E hipEventSynchronize(P e) {
  while (static_cast<Event*>(e)->state == -1) std::this_thread::sleep_for(std::chrono::milliseconds(10));
  return 0;
}
E hipFree(P p) {
  free(p);
  return 0;
}
E hipFuncGetAttributes(P a, const void*) {
  memset(a, 0, 56);
  return 0;
}
E hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
E hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
const char* hipGetErrorString(E) { return "error"; }
E hipGetLastError() { return 0; }
E hipGetSymbolAddress(P* p, const void* s) {
  *p = const_cast<P>(s);
  return 0;
}
E hipGraphDestroy(P) { return 0; }
E hipGraphExecDestroy(P) { return 0; }
E hipGraphInstantiate(P* g, P, P*, char*, size_t) {
  *g = nullptr;
  return 0;
}
E hipGraphLaunch(P, P) { return 0; }
E hipHostFree(P p) { return hipFree(p); }
E hipMalloc(P* p, size_t n) {
  *p = malloc(n);
  return *p ? 0 : 2;
}
E hipHostMalloc(P* p, size_t n, unsigned) { return hipMalloc(p, n); }
E hipLaunchCooperativeKernel(const void*, Dim, Dim, P*, unsigned, P) { return 0; }
E hipLaunchKernel(const void*, Dim, Dim, P*, size_t, P) { return 0; }
E hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = size_t(8) << 30;
  return 0;
}
E hipMemcpyAsync(P d, const void* s, size_t n, int kind, P) {
  if (kind == 2) memset(d, 0, n);  // to the host: what no kernel has computed
  else memcpy(d, s, n);
  return 0;
}
E hipMemsetAsync(P d, int v, size_t n, P) {
  memset(d, v, n);
  return 0;
}
E hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return 0;
}
E hipSetDevice(int) { return 0; }
E hipStreamBeginCapture(P, int) { return 0; }
E hipStreamCreateWithFlags(P* s, unsigned) {
  *s = malloc(8);
  return 0;
}
E hipStreamDestroy(P s) { return hipFree(s); }
E hipStreamEndCapture(P, P* g) {
  *g = nullptr;
  return 0;
}
E hipStreamSynchronize(P) {
  wait();
  return 0;
}
}
