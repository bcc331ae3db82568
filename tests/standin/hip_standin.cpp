// CPU stand-in for the HIP runtime calls of plan creation, execution and serving:
// device addresses that nobody reads, launches that do nothing.  Preloaded ahead
// of the runtime in a process of its own (tests/standin/plans.py), it lets CPU
// tests see which launches a plan makes and what it takes in workspace.
// standin_limit > 0: device memory ends there (hipErrorOutOfMemory past it).
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

extern "C" {
long long standin_limit = 0, standin_live = 0, standin_launches = 0;
}

namespace {
std::mutex mu;
std::map<void *, size_t> live;
size_t next_addr = size_t{0x700000000000};
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  if (standin_limit > 0 && standin_live + static_cast<long long>(bytes) > standin_limit) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void *>(next_addr);
  next_addr += (bytes + 8191) / 4096 * 4096;
  live[*p] = bytes;
  standin_live += static_cast<long long>(bytes);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = live.find(p);
  if (it != live.end()) {
    standin_live -= static_cast<long long>(it->second);
    live.erase(it);
  }
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  ++standin_launches;
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *st) {
  *grid = *block = dim3(1);
  *lds = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;  // compute units
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned) {
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  *p = reinterpret_cast<void *>(size_t{0x600000000000});
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}
