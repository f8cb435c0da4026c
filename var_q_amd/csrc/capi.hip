// Error reporting and version query of the C ABI (varq.h), and what the rules of the launches ask of the device.
#include "varq_common.h"

static thread_local char g_err[512] = "";

int varq_set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cus[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

extern "C" const char *varq_last_error(void) { return g_err; }
extern "C" int varq_abi_version(void) { return VARQ_ABI_VERSION; }
