// A host stand-in for the HIP runtime calls that libcueva.so makes, loaded
// ahead of the runtime (LD_PRELOAD), so that the host side of its transfers
// runs without a GPU.  "Device" and "pinned" memory are host memory.  Work on
// a stream is only queued; it runs when something waits for it (a stream or
// event wait), which is the latest that a GPU could run it: whatever the
// library does without the wait it needs shows as a wrong value or as work
// still queued.  Of the kernels, the two that place and gather rows run; the
// others do nothing.  Calls can be told to fail, and each thread has a current
// device, with the rules of HIP's multi-device guide: an event is recorded only
// on a stream of its own device, a kernel launched only on a stream of the
// current one, a copy is taken on any.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>

struct FakeStream {
  int dev;
  unsigned long long queued = 0, done = 0;
  std::deque<std::function<void()>> work;
};
struct FakeEvent {
  int dev;
  FakeStream* on = nullptr;
  unsigned long long at = 0;
};

static std::recursive_mutex mu;
static std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> m;
  return m;
}
static std::map<std::string, std::pair<int, int>> fail;  // call -> (successes left, failures after that)
static std::map<char*, size_t> device_memory;
static unsigned long long pending;
static thread_local int current = 0;
static thread_local hipError_t last = hipSuccess;

#define LOCK std::lock_guard<std::recursive_mutex> guard(mu)

static hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
static bool fails(const char* call) {
  auto it = fail.find(call);
  if (it == fail.end()) return false;
  if (it->second.first > 0) return it->second.first--, false;
  return it->second.second > 0 && it->second.second--;
}
static FakeStream* S(hipStream_t s) { return (FakeStream*)s; }
static hipError_t put(hipStream_t s, std::function<void()> f) {
  S(s)->work.push_back(std::move(f));
  S(s)->queued++;
  pending++;
  return hipSuccess;
}
static void run_to(FakeStream* s, unsigned long long n) {
  while (s->done < n) {
    s->work.front()();
    s->work.pop_front();
    s->done++;
    pending--;
  }
}

extern "C" {
// for the test
void fake_fail(const char* call, int after, int times) { LOCK; fail[call] = {after, times}; }
unsigned long long fake_pending() { LOCK; return pending; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  LOCK;
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static thread_local struct { dim3 g, b; size_t m; hipStream_t s; } cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) { cfg = {g, b, m, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = cfg.g; *b = cfg.b; *m = cfg.m; *s = cfg.s;
  return hipSuccess;
}

hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }
hipError_t hipGetSymbolAddress(void**, const void*) { return ret(hipErrorInvalidSymbol); }

hipError_t hipMalloc(void** p, size_t n) {
  LOCK;
  if (fails("hipMalloc")) return ret(hipErrorOutOfMemory);
  *p = calloc(1, n);
  device_memory[(char*)*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) { LOCK; device_memory.erase((char*)p); free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  LOCK;
  if (fails("hipHostMalloc")) return ret(hipErrorOutOfMemory);
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  LOCK;
  memset(a, 0, sizeof(*a));
  auto it = device_memory.upper_bound((char*)p);
  if (it == device_memory.begin()) return ret(hipErrorInvalidValue);
  --it;
  if ((char*)p >= it->first + it->second) return ret(hipErrorInvalidValue);
  a->type = hipMemoryTypeDevice;
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  FakeStream* f = new FakeStream;
  f->dev = current;
  *s = (hipStream_t)f;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { LOCK; run_to(S(s), S(s)->queued); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { hipStreamSynchronize(s); delete S(s); return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  LOCK;
  if (fails("hipEventCreateWithFlags")) return ret(hipErrorOutOfMemory);
  FakeEvent* f = new FakeEvent;
  f->dev = current;
  *e = (hipEvent_t)f;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (FakeEvent*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  LOCK;
  FakeEvent* f = (FakeEvent*)e;
  if (fails("hipEventRecord")) return ret(hipErrorUnknown);
  if (f->dev != S(s)->dev) return ret(hipErrorInvalidHandle);
  f->on = S(s);
  f->at = S(s)->queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  LOCK;
  FakeEvent* f = (FakeEvent*)e;
  if (f->on) run_to(f->on, f->at);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }

hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  LOCK;
  return put(s, [=]() { memset(p, v, n); });
}
hipError_t hipMemcpyAsync(void* d, const void* a, size_t n, hipMemcpyKind, hipStream_t s) {
  LOCK;
  return put(s, [=]() { memcpy(d, a, n); });
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* a, size_t ap, size_t w, size_t h, hipMemcpyKind,
                            hipStream_t s) {
  LOCK;
  if (fails("hipMemcpy2DAsync")) return ret(hipErrorUnknown);
  return put(s, [=]() {
    for (size_t r = 0; r < h; r++) memcpy((char*)d + r * dp, (const char*)a + r * ap, w);
  });
}

hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s) {
  LOCK;
  if (S(s)->dev != current) return ret(hipErrorInvalidHandle);
  const std::string& name = kernels()[f];
  const bool up = name.find("k_rows_to_planes") != std::string::npos;
  if (!up && name.find("k_planes_to_rows") == std::string::npos) return put(s, []() {});
  // (buffer, list of planes (the pointers come first), w, hh, pitch, r0, rows)
  double* buf = *(double**)args[0];
  struct { double* a[32]; } pl;
  memcpy(&pl, args[1], sizeof(pl));
  const int w = *(int*)args[2], hh = *(int*)args[3], pitch = *(int*)args[4], r0 = *(int*)args[5], rows = *(int*)args[6];
  return put(s, [=]() {
    for (int r = 0; r < rows; r++) {
      double* row = pl.a[(r0 + r) / hh] + (long)((r0 + r) % hh) * pitch + FIRST_COLUMN;
      if (up) memcpy(row, buf + (long)r * w, sizeof(double) * w);
      else memcpy(buf + (long)r * w, row, sizeof(double) * w);
    }
  });
}
}
