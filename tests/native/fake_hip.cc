// fake_hip.cc -- the HIP calls of libdfrg.so's host code on host memory, for tests of its failure paths
// without a GPU: loaded into the global scope before the library, so the library's calls land here.
// Kernels are not run.  Calls that matter to such a test are logged by letter, and two can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <string>

namespace
{
  std::string log_; // L launch, S stream synchronisation, M pinned allocation, C graph captured, D graph destroyed
  bool fail_host_malloc = false, fail_instantiate = false;
  alignas(256) char scratch[64 << 20];
} // namespace

extern "C" {
const char *fake_log() { return log_.c_str(); }
void fake_clear() { log_.clear(); }
void fake_fail(int host_malloc, int instantiate)
{
  fail_host_malloc = host_malloc;
  fail_instantiate = instantiate;
}

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
  std::memset(p, 0, sizeof(*p));
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = scratch, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "forced"; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return *p = std::calloc(n, 1), hipSuccess; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return hipFree(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
  log_ += 'M';
  if (fail_host_malloc) return hipErrorOutOfMemory;
  return *p = std::calloc(n, 1), hipSuccess;
}
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return p == scratch ? p : std::memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return log_ += 'S', hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shm, hipStream_t *s)
{
  return *g = *b = dim3(1), *shm = 0, *s = nullptr, hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return log_ += 'L', hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return log_ += 'C', *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
  if (fail_instantiate) return hipErrorOutOfMemory;
  return *e = (hipGraphExec_t)1, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return log_ += 'D', hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
