// host_stage.cpp -- the pinned slots of synchronous transfers (api.cpp) over a
// runtime of stubs in host memory, for failures that a GPU does not give on
// demand: no memory to pin, and a capture query that is refused.  Built with
// api.cpp by tests/test_host_stage.py; no GPU code runs.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../xmp_amd/csrc/internal.hpp"
#include "../../xmp_amd/csrc/kernels.hpp"

static hipError_t last = hipSuccess;
static int pins = 0, copies = 0;
static hipError_t pin_result = hipSuccess, capture_result = hipSuccess;
static hipError_t fail(hipError_t e) { return last = e; }

extern "C" {
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipPeekAtLastError(void) { return last; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->totalGlobalMem = (size_t)1 << 30;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) {
  pins++;
  if (pin_result != hipSuccess) return fail(pin_result);
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  if (capture_result != hipSuccess) return fail(capture_result);
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  copies++;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
int roctxRangePushA(const char *) { return 0; }
int roctxRangePop(void) { return 0; }
}

namespace xmp {
bool transfer_in_words(uint32_t, int32_t, int32_t, uint32_t, uint32_t, uint32_t) { return true; }
hipError_t launch_copy(void *d, const void *s, size_t n, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t launch_import(uint32_t *d, uint32_t st, uint32_t nl, const uint8_t *s, uint32_t c, uint32_t, int32_t, int32_t,
                         uint32_t, uint32_t, const uint32_t *, uint32_t, hipStream_t) {
  for (uint32_t i = 0; i < c; i++)
    for (uint32_t j = 0; j < nl; j++) std::memcpy(d + (size_t)j * st + i, s + 4 * ((size_t)i * nl + j), 4);
  return hipSuccess;
}
hipError_t launch_export(uint8_t *d, const uint32_t *s, uint32_t st, uint32_t nl, uint32_t c, uint32_t, int32_t, int32_t,
                         uint32_t, uint32_t, const uint32_t *, uint32_t, hipStream_t) {
  for (uint32_t i = 0; i < c; i++)
    for (uint32_t j = 0; j < nl; j++) std::memcpy(d + 4 * ((size_t)i * nl + j), s + (size_t)j * st + i, 4);
  return hipSuccess;
}
hipError_t launch_set(uint32_t *, uint32_t, uint32_t, const uint32_t *, uint32_t, uint32_t, uint32_t, uint32_t,
                      const uint32_t *, uint32_t, const uint32_t *, uint32_t, hipStream_t) { return hipSuccess; }
}  // namespace xmp

#define CHECK(x) \
  if (!(x)) return std::printf("line %d: %s (%d pins, %d copies)\n", __LINE__, #x, pins, copies), 1

// three imports and exports on a new handle, whose results are right
static int round_trips(void) {
  const uint32_t n = 40, limbs = 8;
  xmpHandle_t h;
  xmpIntegers_t x;
  CHECK(xmpHandleCreate(&h) == xmpErrorSuccess);
  CHECK(xmpIntegersCreate(h, &x, 32 * limbs, n) == xmpErrorSuccess);
  for (uint32_t k = 0; k < 3; k++) {
    uint32_t a[n * limbs], b[n * limbs] = {}, words;
    for (uint32_t j = 0; j < n * limbs; j++) a[j] = 77 * j + k;
    CHECK(xmpIntegersImport(h, x, limbs, -1, 4, 0, 0, a, n) == xmpErrorSuccess);
    CHECK(xmpIntegersExport(h, b, &words, -1, 4, 0, 0, x, n) == xmpErrorSuccess);
    CHECK(words == limbs && std::memcmp(a, b, sizeof a) == 0);
  }
  CHECK(xmpIntegersDestroy(h, x) == xmpErrorSuccess);
  CHECK(xmpHandleDestroy(h) == xmpErrorSuccess);
  CHECK(last == hipSuccess);
  return 0;
}

int main() {
  if (round_trips()) return 1;
  CHECK(pins == 1 && copies == 0);
  // no memory to pin: asked for once, and the runtime's copies instead
  pins = 0;
  pin_result = hipErrorOutOfMemory;
  if (round_trips()) return 1;
  CHECK(pins == 1 && copies == 6);
  // a refusal that passes (another thread's capture) is no reason to stop asking
  pins = copies = 0;
  pin_result = hipErrorStreamCaptureUnsupported;
  if (round_trips()) return 1;
  CHECK(pins >= 6 && copies == 6);
  // the capture query refused: the runtime's path, and no error left behind
  pins = copies = 0;
  pin_result = hipSuccess;
  capture_result = hipErrorStreamCaptureImplicit;
  if (round_trips()) return 1;
  CHECK(pins == 0 && copies == 6);
  std::printf("host stage ok\n");
  return 0;
}
