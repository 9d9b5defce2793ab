// Host-side runtime helpers of the bitexact HIP library: error text, launch checks, device properties.
#include <cstdarg>
#include <cstdio>

#include "bx_common.h"

namespace bx {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: %s", what, hipGetErrorString(e));
    return BX_EHIP;
  }
  return BX_OK;
}

int device_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

}  // namespace bx

extern "C" const char* bx_last_error(void) { return bx::g_err; }
extern "C" int bx_version(void) { return 1; }

extern "C" int64_t bx_capture_id(bx_stream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo((hipStream_t)stream, &status, &id) != hipSuccess) {
    (void)hipGetLastError();                         // (a launch check after this call sees its own errors only)
    return 0;
  }
  return status == hipStreamCaptureStatusActive ? (int64_t)id : 0;
}
