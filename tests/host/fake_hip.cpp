// Stand-in for the HIP runtime on the host: memory is host memory filled with
// a pattern, copies are memcpy, kernel launches do nothing.  Loaded before the
// library (RTLD_GLOBAL), so that the library's calls bind to it; for tests of
// what the host side allocates, copies, launches and leaves behind, in
// processes of their own without a GPU.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {
const int kOk = 0, kOutOfMemory = 2;
struct Counts {
  long allocs, alloc_bytes, host_allocs, launches, copies, live;
} g;
long g_fail_at = 0;  // the n-th stream-ordered allocation from now on fails
int g_last = kOk;    // kept until it is asked for
std::map<void*, size_t> g_mem;
std::mutex g_mu;

int take(void** p, size_t n, long& count) {
  std::lock_guard<std::mutex> lk(g_mu);
  ++count;
  *p = nullptr;
  if (g_fail_at > 0 && --g_fail_at == 0) return g_last = kOutOfMemory;
  *p = malloc(n ? n : 1);
  memset(*p, 0xA5, n);
  g_mem[*p] = n;
  ++g.live;
  return kOk;
}
int give(void* p) {
  if (!p) return kOk;
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_mem.erase(p)) --g.live;
  free(p);
  return kOk;
}
struct Dim3 {
  unsigned x, y, z;
};
}  // namespace

extern "C" {
void fake_fail_alloc(long n) { g_fail_at = n; }
void fake_counts(long* out) { memcpy(out, &g, sizeof(g)); }

int hipGetDeviceCount(int* n) { return *n = 1, kOk; }
int hipGetDevice(int* d) { return *d = 0, kOk; }
int hipSetDevice(int) { return kOk; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 160 * 1024, kOk; }
int hipDeviceGetDefaultMemPool(void** p, int) { return *p = nullptr, kOk; }
int hipMemPoolSetAttribute(void*, int, void*) { return kOk; }
int hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = size_t(1) << 38, kOk; }
int hipGetLastError() {
  const int e = g_last;
  g_last = kOk;
  return e;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipMalloc(void** p, size_t n) { return g.alloc_bytes += (long)n, take(p, n, g.allocs); }
int hipMallocAsync(void** p, size_t n, void*) { return g.alloc_bytes += (long)n, take(p, n, g.allocs); }
int hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n, g.host_allocs); }
int hipFree(void* p) { return give(p); }
int hipFreeAsync(void* p, void*) { return give(p); }
int hipHostFree(void* p) { return give(p); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return ++g.copies, memmove(d, s, n), kOk; }
int hipStreamCreate(void** s) { return *s = (void*)1, kOk; }
int hipStreamDestroy(void*) { return kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamBeginCapture(void*, int) { return 1; }
int hipStreamEndCapture(void*, void** gr) { return *gr = nullptr, 1; }
int hipGraphInstantiate(void**, void*, void**, char*, size_t) { return 1; }
int hipGraphLaunch(void*, void*) { return 1; }
int hipGraphDestroy(void*) { return kOk; }
int hipGraphExecDestroy(void*) { return kOk; }
int hipEventCreate(void** e) { return *e = (void*)1, kOk; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = (void*)1, kOk; }
int hipEventDestroy(void*) { return kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventQuery(void*) { return kOk; }
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.0f, kOk; }
int hipFuncSetAttribute(const void*, int, int) { return kOk; }
int hipGetSymbolAddress(void** p, const void*) {
  static double scratch[4096];
  return *p = scratch, kOk;
}
int hipLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*) { return ++g.launches, kOk; }
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return kOk; }
int __hipPopCallConfiguration(Dim3* a, Dim3* b, size_t* c, void** d) {
  *a = *b = Dim3{1, 1, 1};
  *c = 0;
  *d = nullptr;
  return kOk;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
