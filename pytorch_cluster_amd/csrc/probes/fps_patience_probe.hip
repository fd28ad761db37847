// launch_fps with another patience than its own, for the test of what happens when
// a workgroup does not hear from the others of its example in time.  (Every wait is
// bounded, with any patience.)
#include "../launchers.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

extern "C" int pca_probe_fps(const float *src, const int64_t *ptr,
                             const int64_t *out_ptr, int64_t n, int64_t d,
                             int64_t num_segments, int64_t max_rows,
                             int patience, int64_t *out, void *workspace,
                             size_t workspace_bytes) {
  if (workspace_bytes < pca::fps_scratch_bytes(0, (int)n, (int)d,
                                               (int)num_segments, max_rows))
    return -1;
  return (int)pca::launch_fps(0, src, ptr, out_ptr, nullptr, (int)n, (int)d,
                              (int)num_segments, max_rows, workspace, false,
                              out, nullptr, patience);
}
