// Test-only stand-in for the HIP runtime, preloaded into a CPU process: device
// memory is host memory, copies are made at once, and launches, copies, event
// records and waits are only written to a log, one line each. A launch of a
// kernel whose name contains the string given to fake_fail_launch fails with
// hipErrorLaunchFailure.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

namespace {

char g_log[1 << 16];
size_t g_log_len = 0;
char g_fail[64];
unsigned long g_news = 0;
hipError_t g_last = hipSuccess;

void note(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  const int n = vsnprintf(g_log + g_log_len, sizeof(g_log) - g_log_len, fmt, ap);
  va_end(ap);
  if (n > 0 && g_log_len + static_cast<size_t>(n) < sizeof(g_log)) g_log_len += n;
}

struct Kernel {
  const void* host;
  char name[192];
};
Kernel g_kernels[4096];
int g_kernel_count = 0;

const char* name_of(const void* host) {
  for (int i = 0; i < g_kernel_count; ++i)
    if (g_kernels[i].host == host) return g_kernels[i].name;
  return "?";
}

struct Var {
  const void* host;
  void* mem;
};
Var g_vars[16];
int g_var_count = 0;

struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} g_config;

}  // namespace

// Allocations by C++ code (the stand-in itself makes none this way).
void* operator new(size_t n) {
  ++g_news;
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {

void fake_fail_launch(const char* part) { snprintf(g_fail, sizeof(g_fail), "%s", part); }
const char* fake_log() { return g_log; }
// Leaves the error of an earlier call behind, as any failed HIP call does.
void fake_leave_error() { g_last = hipErrorOutOfMemory; }
void fake_clear_log() { g_log[g_log_len = 0] = 0; }
unsigned long fake_news() { return g_news; }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  if (g_kernel_count == 4096) std::abort();
  Kernel& k = g_kernels[g_kernel_count++];
  k.host = host;
  snprintf(k.name, sizeof(k.name), "%s", name);
}
void __hipRegisterVar(void**, void* host, char*, char*, int, size_t size, int, int) {
  if (g_var_count == 16) std::abort();
  g_vars[g_var_count++] = Var{host, std::calloc(1, size)};
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_config = Config{grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared,
                                     hipStream_t* stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *shared = g_config.shared;
  *stream = g_config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3, void**, size_t, hipStream_t s) {
  const char* name = name_of(host);
  const bool fails = g_fail[0] && std::strstr(name, g_fail);
  note("%s %s %u %p\n", fails ? "failed" : "launch", name, grid.x, static_cast<void*>(s));
  if (fails) g_last = hipErrorLaunchFailure;
  return fails ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorLaunchFailure ? "launch failure" : "error";
}

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
  for (int i = 0; i < g_var_count; ++i)
    if (g_vars[i].host == symbol) {
      *p = g_vars[i].mem;
      return hipSuccess;
    }
  return hipErrorInvalidSymbol;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
  *free_bytes = *total = size_t(1) << 38;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
// No memory pool: ray ordering finds no memory, and says so in the log.
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t*, int) {
  return g_last = hipErrorNotSupported;
}
hipError_t hipMallocAsync(void**, size_t n, hipStream_t s) {
  note("nopool %zu %p\n", n, static_cast<void*>(s));
  return g_last = hipErrorOutOfMemory;
}
hipError_t hipFreeAsync(void*, hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  note("copy %p %p %zu %p\n", d, s, n, static_cast<void*>(st));
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = static_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  note("syncstream %p\n", static_cast<void*>(s));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = static_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  note("record %p %p\n", static_cast<void*>(e), static_cast<void*>(s));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  note("sync %p\n", static_cast<void*>(e));
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  note("wait %p %p\n", static_cast<void*>(e), static_cast<void*>(s));
  return hipSuccess;
}

}  // extern "C"
