// launch_fps with another patience than its own, for the tests of what happens when
// a workgroup does not hear from the others of its example in time, or the others do
// not come.  (Every wait is bounded, with any patience.)  `states`: the examples' words
// after a call that shares them (bit 30: sampled by one workgroup after all).
#include "../launchers.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

extern "C" int pca_probe_fps(const float *src, const int64_t *ptr,
                             const int64_t *out_ptr, int64_t n, int64_t d,
                             int64_t num_segments, int64_t max_rows, int told,
                             int came, int64_t *out, void *workspace,
                             size_t workspace_bytes, uint32_t *states) {
  if (workspace_bytes < pca::fps_scratch_bytes(0, (int)n, (int)d,
                                               (int)num_segments, max_rows))
    return -1;
  pca::FpsPatience patience;
  if (told >= 0)
    patience.told = told;
  if (came >= 0)
    patience.came = came;
  const hipError_t err =
      pca::launch_fps(0, src, ptr, out_ptr, nullptr, (int)n, (int)d,
                      (int)num_segments, max_rows, workspace, false, out,
                      nullptr, patience);
  if (err != hipSuccess)
    return (int)err;
  return (int)hipMemcpyAsync(
      states,
      static_cast<char *>(workspace) +
          pca::fps_states_at((int)n, (int)num_segments),
      sizeof(uint32_t) * (size_t)num_segments, hipMemcpyDeviceToDevice,
      nullptr);
}
