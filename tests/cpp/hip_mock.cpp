// A HIP runtime of two devices that runs no kernel: it counts what is alive,
// refuses the call of a chosen number or the device memory beyond a capacity.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>

namespace {
std::map<void*, size_t> size;
size_t used = 0, capacity = 0;
int syncs = 0;
int device = 1, streams = 0, events = 0, buffers = 0, calls = 0, refuse = 0;
bool refused() { return ++calls == refuse; }
template <class T>
hipError_t make(T* out, int& alive, hipError_t error) {
  if (refused()) return error;
  *out = reinterpret_cast<T>(std::malloc(1));
  ++alive;
  return hipSuccess;
}
template <class T>
hipError_t drop(T h, int& alive) {
  std::free(reinterpret_cast<void*>(h));
  --alive;
  return hipSuccess;
}
}  // namespace

extern "C" {
void mock_refuse(int n) { calls = 0; refuse = n; }
int mock_calls() { return calls; }
int mock_device() { return device; }
int mock_alive() { return streams + events + buffers; }

hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return make(s, streams, hipErrorUnknown);
}
hipError_t hipStreamDestroy(hipStream_t s) { return drop(s, streams); }
int mock_syncs() { return syncs; }
hipError_t hipStreamSynchronize(hipStream_t) { ++syncs; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return make(e, events, hipErrorUnknown); }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e, events); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  const hipError_t e = make(p, buffers, hipErrorOutOfMemory);
  if (e == hipSuccess) *p = std::realloc(*p, n), std::memset(*p, 0, n);
  return e;
}
hipError_t hipHostFree(void* p) { return drop(p, buffers); }
hipError_t hipMalloc(void** p, size_t n) {
  if (capacity && used + n > capacity) return hipErrorOutOfMemory;
  const hipError_t e = make(p, buffers, hipErrorOutOfMemory);
  if (e == hipSuccess) used += size[*p] = n;
  return e;
}
hipError_t hipFree(void* p) {
  used -= size[p];
  size.erase(p);
  return drop(p, buffers);
}

void mock_capacity(size_t bytes) { capacity = bytes; }
size_t mock_used() { return used; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  return make(e, events, hipErrorUnknown);
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
// device memory holds zeros
hipError_t hipMemcpy(void* d, const void*, size_t n, hipMemcpyKind k) {
  if (k == hipMemcpyDeviceToHost) std::memset(d, 0, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) {
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  return hipSuccess;
}
}
