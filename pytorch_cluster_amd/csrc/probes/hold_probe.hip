// Holds compute units for some time, for tests of what other calls do beside such work:
// more LDS than half a unit has, so a workgroup takes one of its own.  (Bounded by the
// clock and, if that stood still, by the number of looks at it.)
#include <hip/hip_runtime.h>

namespace {
__global__ __launch_bounds__(64) void hold_kernel(long long ticks) {
  __shared__ volatile int room[24 * 1024];
  room[threadIdx.x] = 0;
  const long long begin = wall_clock64();
  for (int i = 0; i < 100000 && wall_clock64() - begin < ticks; ++i)
    __builtin_amdgcn_s_sleep(8);
}
} // namespace

// `us`: at most 10,000 (a tick of the clock is 10 ns).
extern "C" int pca_probe_hold(int units, int us, void *stream) {
  if (units < 1 || units > 256 || us < 1 || us > 10000)
    return -1;
  hipLaunchKernelGGL(hold_kernel, dim3(units), dim3(64), 0,
                     static_cast<hipStream_t>(stream), 100ll * us);
  return (int)hipGetLastError();
}
