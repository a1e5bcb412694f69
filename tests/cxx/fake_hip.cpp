// A HIP runtime that only keeps books: what libawk_hip.so allocates, launches and
// records, in order, on memory that does not exist.  Loaded ahead of the real runtime
// (tests/fake_hip.py), it shows on the CPU what the host code does at an allocation or
// a launch that fails, under capture, and with which pointers and grids it launches.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <new>
#include <map>
#include <string>
#include <vector>

namespace {
struct Pool {
  std::multimap<size_t, uintptr_t> idle;
};
struct Block {
  size_t size;
  Pool *pool;  // null: hipMalloc, or the runtime's own pool (which keeps nothing)
};
bool g_no_host_memory = false;
struct Own {  // the books themselves do not run out
  bool was = g_no_host_memory;
  Own() { g_no_host_memory = false; }
  ~Own() { g_no_host_memory = was; }
};
size_t g_budget = SIZE_MAX, g_used = 0;
uintptr_t g_next = 0x100000000ull;
std::map<uintptr_t, Block> g_live;
std::map<const void *, std::string> g_names;
std::string g_log, g_fail_name;
int g_fail_skip = 0;
bool g_capturing = false, g_strict = false;  // strict: calls that no capture but a relaxed one allows fail
hipError_t g_last = hipSuccess;
std::vector<void *> g_call;
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_stream;
uintptr_t g_handle = 0x1000;

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
void note(const std::string &s) {
  Own own;
  g_log += s + "\n";
}
std::string num(uintptr_t v) { return std::to_string((unsigned long long)v); }
template <class T>
std::string num(T *p) {
  return num(reinterpret_cast<uintptr_t>(p));
}

hipError_t take(void **p, size_t n, Pool *pool) {
  Own own;
  if (pool) {
    auto it = pool->idle.lower_bound(n);
    if (it != pool->idle.end()) {
      *p = reinterpret_cast<void *>(it->second);
      g_live[it->second] = Block{it->first, pool};
      pool->idle.erase(it);
      return hipSuccess;
    }
  }
  if (n > g_budget || g_used > g_budget - n) return ret(hipErrorOutOfMemory);
  g_used += n;
  *p = reinterpret_cast<void *>(g_next);
  g_live[g_next] = Block{n, pool};
  g_next += (n + 0xffff) / 0x10000 * 0x10000 + 0x10000;
  return hipSuccess;
}
hipError_t give(void *p) {
  Own own;
  if (!p) return hipSuccess;
  auto it = g_live.find(reinterpret_cast<uintptr_t>(p));
  if (it == g_live.end()) return ret(hipErrorInvalidValue);
  if (it->second.pool) it->second.pool->idle.emplace(it->second.size, it->first);
  else g_used -= it->second.size;
  g_live.erase(it);
  return hipSuccess;
}
hipError_t launch(const void *f, dim3 g, dim3 b, void **args, hipStream_t s) {
  const std::string &name = g_names[f];
  if (!g_fail_name.empty() && name.find(g_fail_name) != std::string::npos && g_fail_skip-- == 0) {
    note("failed " + name);
    return ret(hipErrorLaunchFailure);
  }
  // the documented limit: fewer than 2^32 threads along an axis
  if ((unsigned long long)g.x * b.x >> 32 || (unsigned long long)g.y * b.y >> 32 || (unsigned long long)g.z * b.z >> 32)
    return ret(hipErrorInvalidConfiguration);
  note("launch " + name + " " + num((uintptr_t)g.x) + " " + num((uintptr_t)g.y) + " " + num((uintptr_t)b.x) + " " +
       num(s) + " " + num(*static_cast<uintptr_t *>(args[0])));
  return hipSuccess;
}
}  // namespace

// host memory that runs out on demand
void *operator new(std::size_t n) {
  void *p = g_no_host_memory ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

extern "C" {

// ---- the test's side
void fake_no_host_memory(int on) { g_no_host_memory = on != 0; }
void fake_budget(unsigned long long bytes) { g_budget = bytes; }
unsigned long long fake_used() { return g_used; }
void fake_fail(const char *name, int skip) {
  g_fail_name = name;
  g_fail_skip = skip;
}
void fake_capture(int mode) {  // 0 none, 1 global, 2 relaxed
  g_capturing = mode != 0;
  g_strict = mode == 1;
}
const char *fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }

// ---- the runtime's side
void **__hipRegisterFatBinary(const void *) {
  static void *module = nullptr;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
  g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, hipStream_t s) {
  g_grid = g;
  g_block = b;
  g_shmem = shmem;
  g_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shmem, hipStream_t *s) {
  *g = g_grid;
  *b = g_block;
  *shmem = g_shmem;
  *s = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t s) {
  return launch(f, g, b, args, s);
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t s, hipEvent_t, hipEvent_t,
                              int) {
  return launch(f, g, b, args, s);
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipDeviceSynchronize() {
  note(g_capturing ? "invalidated" : "sync");  // whatever the capture's mode
  return g_capturing ? ret(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  if (g_strict) return ret(hipErrorStreamCaptureUnsupported);
  return take(p, n, nullptr);
}
hipError_t hipFree(void *p) {  // waits for the device
  note("free");
  return give(p);
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return take(p, n, nullptr); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return give(p); }
hipError_t hipMemPoolCreate(hipMemPool_t *p, const hipMemPoolProps *) {
  *p = reinterpret_cast<hipMemPool_t>(new Pool());
  return hipSuccess;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipMallocFromPoolAsync(void **p, size_t n, hipMemPool_t pool, hipStream_t) {
  return take(p, n, reinterpret_cast<Pool *>(pool));
}
hipError_t hipMemPoolTrimTo(hipMemPool_t pool, size_t) {  // (to zero: all that is asked here)
  Pool *q = reinterpret_cast<Pool *>(pool);
  for (const auto &b : q->idle) g_used -= b.first;
  q->idle.clear();
  return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *, size_t n, hipMemcpyKind k) {
  if (k == hipMemcpyDeviceToHost) std::memset(dst, 0, n);
  note("sync");
  return g_strict ? ret(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k == hipMemcpyDeviceToHost) std::memset(dst, 0, n);
  return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) {  // returns before it is done, unlike hipMemcpy
  note("memset");
  return g_strict ? ret(hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = reinterpret_cast<void *>(uintptr_t{0x10000});
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(g_handle += 16);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (!s) note("sync");
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
  *c = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  note("wait " + num(s) + " " + num(e));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(g_handle += 16);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  note("record " + num(e) + " " + num(s));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}

}  // extern "C"
