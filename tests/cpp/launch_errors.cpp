// The launchers of calls with two kernels, linked from the built library, with
// this program's stand-ins in front of the HIP launch calls: the first kernel's
// launch is refused, the last one's is not (tests/test_launch_errors.py).
// Runs on the CPU; no kernel starts.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>

#include "../../plainmp_amd/csrc/launch.h"

static hipError_t g_last = hipSuccess;
static int g_refused = 0, g_taken = 0;

extern "C" {
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = *b = dim3(1);
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  ++g_refused;
  return g_last = hipErrorInvalidConfiguration;
}
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
  ++g_taken;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
}

int main() {
  using namespace pmp;
  static char event;
  KinArgs<float> k32{};
  KinArgs<double> k64{};
  SceneArgs<float> s32{};
  SceneArgs<double> s64{};
  k32.n_items = k32.n_cols = k64.n_cols = 1;
  k32.lds_limit = k64.lds_limit = 65536;
  EdgeArgs ea{};
  ea.E = 100000;
  for (int waits = 0; waits < 2; ++waits) {  // without and with a stop event for the last kernel
    call_end.ask = waits ? (hipEvent_t)&event : nullptr;
    call_end.done = nullptr;
    const hipError_t e = launch_edges(k32, k64, s32, s64, ea, 1e-5f, 256, 256, nullptr);
    std::printf("edges %d %d %d\n", (int)e, g_refused, g_taken);
    g_last = hipSuccess;
    call_end.ask = waits ? (hipEvent_t)&event : nullptr;
    call_end.done = nullptr;
    const hipError_t v = launch_vjp(k32, s32, nullptr, 64, 64, nullptr, nullptr, nullptr, 0, nullptr);
    std::printf("vjp %d %d %d\n", (int)v, g_refused, g_taken);
    g_last = hipSuccess;
  }
  return 0;
}
