// A HIP runtime that runs on the CPU, for tests of the library's host code: memory is host
// memory, copies are done at once, kernels are counted and not run.  Loaded with RTLD_GLOBAL
// before the library, its symbols are found before the real runtime's.  A test can make
// device allocations and operator new fail.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
struct Dim { unsigned x, y, z; };
std::mutex mu;
std::map<const void *, std::string> &names() { static std::map<const void *, std::string> m; return m; }
constexpr long LOG = 1 << 18;
const char *launched[LOG];                         // takes no memory of the kind it counts
long nlaunched = 0;
long mallocs = 0, malloc_ok = -1, events = 0;      // malloc_ok: allocations that still succeed, -1 all
int last = 0;
std::atomic<long> news{0}, new_fail{0};            // the new_fail-th operator new from now on fails
thread_local struct { Dim g, b; size_t sh; void *s; } cfg;
int ret(int e) { if (e) last = e; return e; }
constexpr int INVALID = 1, NOMEM = 2;
}  // namespace

void *operator new(size_t n) {
  ++news;
  if (new_fail > 0 && --new_fail == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
long stub_mallocs() { return mallocs; }
long stub_events() { return events; }
void stub_malloc_ok(long n) { malloc_ok = n; }
long stub_news() { return news; }
void stub_new_fail(long n) { new_fail = n; }
long stub_launches() { return nlaunched; }
const char *stub_launch(long i) { return launched[i]; }

void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim g, Dim b, size_t sh, void *s) { cfg = {g, b, sh, s}; return 0; }
int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *sh, void **s) { *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *s = cfg.s; return 0; }
int hipLaunchKernel(const void *f, Dim, Dim, void **, size_t, void *) {
  std::lock_guard<std::mutex> l(mu);
  const auto k = names().find(f);
  if (nlaunched == LOG || k == names().end()) std::abort();
  launched[nlaunched++] = k->second.c_str();
  return 0;
}
int hipGetLastError() { const int e = last; last = 0; return e; }
const char *hipGetErrorString(int e) { return e == NOMEM ? "out of memory" : "error"; }
int hipSetDevice(int) { return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 163840; return 0; }
int hipGetSymbolAddress(void **p, const void *) { static double mem[1 << 17]; *p = mem; return 0; }
int hipMalloc(void **p, size_t n) {
  ++mallocs;
  *p = nullptr;
  if (malloc_ok == 0) return ret(NOMEM);
  if (malloc_ok > 0) --malloc_ok;
  *p = std::calloc(1, n);
  return *p ? 0 : ret(NOMEM);
}
int hipFree(void *p) { std::free(p); return 0; }
int hipHostMalloc(void **p, size_t n, unsigned) { *p = std::calloc(1, n); return *p ? 0 : ret(NOMEM); }
int hipHostFree(void *p) { std::free(p); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  if (n && (!d || !s)) return ret(INVALID);
  std::memcpy(d, s, n);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
  if (n && !d) return ret(INVALID);
  std::memset(d, v, n);
  return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned) { *s = std::malloc(1); return 0; }
int hipStreamDestroy(void *s) { std::free(s); return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { ++events; *e = std::malloc(1); return 0; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { std::free(e); return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 0.f; return 0; }
}
