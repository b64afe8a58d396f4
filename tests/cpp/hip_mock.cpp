// A HIP runtime of two devices that counts what is alive and refuses the
// call of a chosen number, for the creation and destruction of a context.
#include <hip/hip_runtime_api.h>

#include <cstdlib>

namespace {
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
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return make(e, events, hipErrorUnknown); }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e, events); }
hipError_t hipHostMalloc(void** p, size_t, unsigned) {
  return make(p, buffers, hipErrorOutOfMemory);
}
hipError_t hipHostFree(void* p) { return drop(p, buffers); }
hipError_t hipMalloc(void** p, size_t) { return make(p, buffers, hipErrorOutOfMemory); }
hipError_t hipFree(void* p) { return drop(p, buffers); }
}
