// hip_stub.cpp -- a HIP runtime that launches nothing, for host-code tests without a GPU: two gfx950
// devices, and a launch with more than 64 KiB of dynamic LDS fails unless the kernel's attribute
// was raised on the device that is current, as each device holds a kernel's attributes of its own.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <utility>

namespace {
int g_dev = 0, g_launches = 0, g_refused = 0, g_mallocs = 0, g_frees = 0, g_copies = 0;
std::map<std::pair<int, const void *>, int> g_lds;
double g_scratch[2][4096];
hipError_t g_last = hipSuccess;
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} g_call;
}  // namespace

extern "C" {
int stub_launches() { return g_launches; }
int stub_refused() { return g_refused; }
int stub_mallocs() { return g_mallocs; }
int stub_frees() { return g_frees; }
int stub_copies() { return g_copies; }

hipError_t hipGetDeviceCount(int *n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = g_dev, hipSuccess; }
hipError_t hipSetDevice(int d) { return g_dev = d, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = g_scratch[g_dev], hipSuccess; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) {
  if (a == hipFuncAttributeMaxDynamicSharedMemorySize) g_lds[{g_dev, f}] = v;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 2, hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  g_call = Call{g, b, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = g_call.grid, *b = g_call.block, *lds = g_call.lds, *s = g_call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t lds, hipStream_t) {
  ++g_launches;
  const auto it = g_lds.find({g_dev, f});
  if (lds > 65536 && (it == g_lds.end() || (size_t)it->second < lds)) {
    ++g_refused;
    return g_last = hipErrorInvalidValue;
  }
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
// device memory is host memory
hipError_t hipMalloc(void **p, size_t n) {
  ++g_mallocs;
  return (*p = calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  g_frees += p != nullptr;
  free(p);
  return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  ++g_copies;
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)&g_call, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)&g_call, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
}
