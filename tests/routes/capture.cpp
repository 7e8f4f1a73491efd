// Convolutions enqueued while their stream is, or is not, being captured, on
// a device that is stubbed out (linked with --wrap for the calls below): it
// counts launches and allocations.  Input: one step a line, "what capturing
// nx ny nz kx ky kz", what = 0 a convolution, 1 a PSF gradient, 2 a plan made
// and destroyed (in a caller's workspace), 3 a batch made and destroyed;
// output: "launches allocations" of the step, or "error <code>".
#include <cstdio>
#include <cstdlib>

#include "../../include/fourierconvolution_amd.h"
#include "conv_driver.hpp"

using namespace fcamd;

static int g_capturing, g_launches, g_allocations;

extern "C" {
hipError_t __wrap_hipMalloc(void** p, size_t) {
  ++g_allocations;
  *p = std::malloc(16);
  return hipSuccess;
}
hipError_t __wrap_hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t __wrap_hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t __wrap_hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t __wrap_hipGetLastError() { return hipSuccess; }
hipError_t __wrap_hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t __wrap___hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) {
  return hipSuccess;
}
hipError_t __wrap___hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) {
  return hipSuccess;
}
hipError_t __wrap_hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  ++g_launches;
  return hipSuccess;
}
hipError_t __wrap_hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t __wrap_hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t __wrap_hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return hipSuccess;
}
hipError_t __wrap_hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(16);
  return hipSuccess;
}
hipError_t __wrap_hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t __wrap_hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(16);
  return hipSuccess;
}
hipError_t __wrap_hipEventDestroy(hipEvent_t) { return hipSuccess; }
}

int main() {
  int what, n[3], k[3];
  // (addresses that nothing reads)
  float* a = reinterpret_cast<float*>(1 << 20);
  void* ws = reinterpret_cast<void*>(1 << 24);
  void* st = reinterpret_cast<void*>(16);
  const long long room = 1LL << 50;
  while (std::scanf("%d %d %d %d %d %d %d %d", &what, &g_capturing, n, n + 1, n + 2, k, k + 1,
                    k + 2) == 8) {
    g_launches = g_allocations = 0;
    int rc = 0;
    if (what == 0) {
      rc = fcamd_convolve3d_device(a, a, n, a, k, FCAMD_CONVOLVE, ws, room, st);
    } else if (what == 1) {
      rc = fcamd_conv_grad_kernel_device(a, a, a, n, k, ws, room, st);
    } else if (what == 2) {
      void* p = fcamd_conv_plan_create(n, k, a, FCAMD_CONVOLVE, ws, room, st);
      rc = p ? 0 : fcamd_last_error();
      fcamd_conv_plan_destroy(p);
    } else {
      float* outs[] = {a};
      const float* ins[] = {a};
      void* p = fcamd_batch_create(1, n, k, outs, ins, ins, FCAMD_CONVOLVE, ws, room);
      rc = p ? 0 : fcamd_last_error();
      fcamd_batch_destroy(p);
    }
    if (rc)
      std::printf("error %d\n", rc);
    else
      std::printf("%d %d\n", g_launches, g_allocations);
  }
  return 0;
}
