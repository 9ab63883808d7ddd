// A stand-in for the HIP runtime that runs nothing: loaded before libbellman.so
// (tests/test_host_calls.py), it answers the library's runtime calls and keeps a
// list of them, so that what the library asks of the GPU, and in which order, can
// be read on a machine without one.  Memory is addresses that nobody reads:
// device d's start at (32 + d) TiB.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>

namespace {

std::string g_log;
std::map<const void *, std::string> g_kernels;
uintptr_t g_next = uintptr_t(32) << 40, g_handle = 0x1000;
size_t g_largest = SIZE_MAX;                   // larger allocations fail
size_t g_free = size_t(200) << 30, g_total = size_t(256) << 30;
std::string g_fail;                            // launches of this kernel (or of a host function) fail
hipError_t g_error = hipSuccess;

struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} g_config;

template <class... A> void note(const char *format, A... a) {
  char line[512];
  snprintf(line, sizeof line, format, a...);
  g_log += line;
  g_log += '\n';
}

unsigned long long n(const void *p) { return (unsigned long long)(uintptr_t)p; }

hipError_t allocate(const char *what, void **p, size_t bytes, hipStream_t s) {
  if (bytes > g_largest) {
    note("%s refused %zu", what, bytes);
    return g_error = hipErrorOutOfMemory;
  }
  *p = reinterpret_cast<void *>(g_next);
  g_next += (bytes + 4095) & ~size_t(4095);
  note("%s %llx %zu s=%llx", what, n(*p), bytes, n(s));
  return hipSuccess;
}

template <class T> hipError_t handle(const char *what, T *h) {
  *h = reinterpret_cast<T>(g_handle);
  g_handle += 16;
  note("%s %llx", what, n(*h));
  return hipSuccess;
}

} // namespace

extern "C" {

const char *fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
void fake_largest(size_t bytes) { g_largest = bytes; }
void fake_memory(size_t free, size_t total) { g_free = free, g_total = total; }
void fake_fail(const char *kernel) { g_fail = kernel; }

void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(&g_log); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) { g_kernels[host] = name; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  g_config = {grid, block, lds, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  *grid = g_config.grid, *block = g_config.block, *lds = g_config.lds, *stream = g_config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t s) {
  const std::string &name = g_kernels[f];
  if (!g_fail.empty() && name.find(g_fail) != std::string::npos)
    return g_error = hipErrorLaunchFailure;
  note("launch %s %u s=%llx", name.c_str(), grid.x, n(s));
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_error;
  g_error = hipSuccess;
  return e;
}

hipError_t hipGetDeviceCount(int *c) { return *c = 2, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return note("device synchronize"), hipSuccess; }
hipError_t hipDeviceEnablePeerAccess(int, unsigned) { return hipSuccess; }
hipError_t hipDeviceDisablePeerAccess(int) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *free, size_t *total) { return *free = g_free, *total = g_total, hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes) { return allocate("malloc", p, bytes, nullptr); }
hipError_t hipMallocAsync(void **p, size_t bytes, hipStream_t s) { return allocate("malloc_async", p, bytes, s); }
hipError_t hipMallocFromPoolAsync(void **p, size_t bytes, hipMemPool_t, hipStream_t s) { return allocate("malloc_async", p, bytes, s); }
hipError_t hipFree(void *p) { return note("free %llx", n(p)), hipSuccess; }
hipError_t hipFreeAsync(void *p, hipStream_t s) { return note("free_async %llx s=%llx", n(p), n(s)), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t, unsigned) { return *p = nullptr, hipErrorOutOfMemory; }
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipHostRegister(void *, size_t, unsigned) { return hipErrorInvalidValue; }
hipError_t hipHostUnregister(void *) { return hipErrorInvalidValue; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = reinterpret_cast<void *>(uintptr_t(32) << 40), hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  const uintptr_t d = reinterpret_cast<uintptr_t>(p) >> 40;
  if (d != 32 && d != 33)
    return g_error = hipErrorInvalidValue;
  memset(a, 0, sizeof *a);
  a->type = hipMemoryTypeDevice;
  a->device = (int)d - 32;
  return hipSuccess;
}
hipError_t hipMemPoolCreate(hipMemPool_t *p, const hipMemPoolProps *) { return handle("pool", p); }
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }
hipError_t hipMemPoolSetAccess(hipMemPool_t, const hipMemAccessDesc *, size_t) { return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }

hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t s) {
  return note("memcpy %llx %llx %zu s=%llx", n(dst), n(src), bytes, n(s)), hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }

hipError_t hipStreamCreate(hipStream_t *s) { return handle("stream", s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle("stream", s); }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { return *d = 0, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return note("synchronize s=%llx", n(s)), hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return note("wait %llx s=%llx", n(e), n(s)), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status) { return *status = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = nullptr, hipSuccess; }
hipError_t hipLaunchHostFunc(hipStream_t s, hipHostFn_t, void *) {
  if (g_fail == "host_func")
    return g_error = hipErrorUnknown;
  return note("host_func s=%llx", n(s)), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return handle("event", e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle("event", e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return note("record %llx s=%llx", n(e), n(s)), hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
}
