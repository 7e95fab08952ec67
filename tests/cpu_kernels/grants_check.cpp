// CPU check of the dynamic LDS that the fully reorthogonalised step's kernels
// are granted on each device (ed_reorth.hip's host code on the runtime calls
// defined here; no kernel runs).  Arguments: devices to ask on, in turn, "-d" for
// a device that refuses.  Output per argument: "device available grants".
#include <map>
#include <string>

#include <hip/hip_runtime.h>

static int g_device = 0, g_grants = 0;
static bool g_refuse = false;
static hipError_t test_get_device(int* d) {
  *d = g_device;
  return hipSuccess;
}
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize = 8 };
static hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) {
  if (g_refuse || bytes < 128 * 1024) return hipErrorInvalidValue;
  ++g_grants;
  return hipSuccess;
}
#define hipGetDevice test_get_device
#undef __shared__  // declared, not run
#define __shared__
#include "cmpy_amd/csrc/ed_reorth.cpp"

namespace ed {
double tile[1];
HvArgs make_hv_args(const ed_op*) { return {}; }
int set_error(int code, const char*, ...) { return code; }
}  // namespace ed

int main(int argc, char** argv) {
  for (int i = 1; i < argc; ++i) {
    g_refuse = argv[i][0] == '-';
    g_device = std::atoi(argv[i] + g_refuse);
    g_grants = 0;
    const bool ok = ed::reorth_available();
    std::printf("%d %d %d\n", g_device, (int)ok, g_grants);
  }
  return 0;
}
