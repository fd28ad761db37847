// Preparation and dispatch of the feature-space `nearest` search (see
// nearest_feat_impl.hpp).
#include "nearest_feat_impl.hpp"

#include <algorithm>
#include <cstdlib>

namespace pca {

#define PCA_DECLARE_BLOCKS(NB)                                                 \
  template <>                                                                  \
  hipError_t launch_nearest_feat_blocks<NB>(const NearestFeatParams &, int,    \
                                            int, hipStream_t);
PCA_DECLARE_BLOCKS(1)
PCA_DECLARE_BLOCKS(2)
PCA_DECLARE_BLOCKS(3)
PCA_DECLARE_BLOCKS(4)
PCA_DECLARE_BLOCKS(5)
PCA_DECLARE_BLOCKS(6)
PCA_DECLARE_BLOCKS(7)
PCA_DECLARE_BLOCKS(8)
#undef PCA_DECLARE_BLOCKS

// 16 lanes per row; few workgroups, as each ends with adds to the same words.
__global__ __launch_bounds__(kBlock) void nearest_feat_rows_kernel(
    const float *__restrict__ x, int n, int d, float *__restrict__ weight,
    NearestFeatGlobals *__restrict__ globals) {
  constexpr int W = kBlock / kWave;
  __shared__ unsigned s_bits[W], s_rows[W];
  __shared__ double s_sum[W], s_log[W];
  const int tid = threadIdx.x;
  const int part = tid & 15;
  unsigned bits = 0, rows = 0;
  double sum = 0.0, logs = 0.0;
  for (int row = blockIdx.x * (kBlock / 16) + (tid >> 4); row < n;
       row += gridDim.x * (kBlock / 16)) {
    const float *p = x + (size_t)row * d;
    float sq = 0.0f;
    unsigned top = 0;
    for (int c = part; c < d; c += 16) {
      const float v = p[c];
      sq = __builtin_fmaf(v, v, sq);
      top = max(top, __float_as_uint(v) & 0x7fffffffu);
    }
#pragma unroll
    for (int sh = 1; sh < 16; sh <<= 1) {
      sq += __shfl_xor(sq, sh);
      top = max(top, (unsigned)__shfl_xor((int)top, sh));
    }
    const bool finite = top < 0x7f800000u;
    const bool moderate = finite && sq <= kFilterNormLimit;
    if (part == 0) {
      weight[row] = moderate ? sq : finite ? -1.0f : -2.0f;
      if (moderate && sq > 0.0f) {
        bits = max(bits, top);
        sum += (double)sq;
        logs += (double)__builtin_log2f(sq);
        ++rows;
      }
    }
  }
#pragma unroll
  for (int sh = 16; sh < kWave; sh <<= 1) { // (part 0 of a row holds them)
    bits = max(bits, (unsigned)__shfl_xor((int)bits, sh));
    rows += (unsigned)__shfl_xor((int)rows, sh);
    sum += __shfl_xor(sum, sh);
    logs += __shfl_xor(logs, sh);
  }
  if ((tid & (kWave - 1)) == 0) {
    s_bits[tid / kWave] = bits;
    s_rows[tid / kWave] = rows;
    s_sum[tid / kWave] = sum;
    s_log[tid / kWave] = logs;
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < W; ++w) {
      bits = max(bits, s_bits[w]);
      rows += s_rows[w];
      sum += s_sum[w];
      logs += s_log[w];
    }
    if (rows != 0) {
      atomicMax(&globals->max_bits, bits);
      atomicAdd(&globals->rows, rows);
      atomicAdd(&globals->sum_sq, sum);
      atomicAdd(&globals->sum_log, logs);
    }
  }
}

namespace {

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

int blocks_of(int d) { return (d + 15) / 16; }

size_t pack_bytes(int n, int d) {
  return align256(sizeof(uint4) * ((size_t)n + kNfTileRows) *
                  (2 * blocks_of(d) + 1));
}

// 1,048,576 queries x 4,096 rows, call (knn_mfma / this kernel, us): 16
// components 1,271 / 396, 32: 1,540 / 453, 64: 2,208 / 679, 128: 4,094 / 1,274.
// At 64 components the kernel takes 695 us under the profiler, 790 TFLOP/s
// (hipBLASLt reaches 1,160 on 8,192^3 in fp16).  Vector ALU / matrix cores busy,
// of the SIMD-cycles: 16 components 67 / 18 %, 32: 61 / 30, 64: 50 / 43, 128:
// 36 / 44; two waves per SIMD wait for a tile, LDS or a barrier in the rest.
//
// Sets of queries per wave: all that fit the registers once that gives every
// CU a workgroup, else one, for four times the workgroups.
int sets_of(int m, int d) {
  const int most = nearest_feat_sets(blocks_of(d));
  return m / (most * 128) >= 256 ? most : 1;
}

// Work items of the segments, and the globals' start values.
__global__ __launch_bounds__(kPlanThreads) void nearest_feat_plan_kernel(
    const int64_t *__restrict__ ptr_y, int m, int num_segments, int per_item,
    int *__restrict__ work_start, NearestFeatGlobals *__restrict__ globals) {
  __shared__ int partial[kPlanThreads];
  if (threadIdx.x == 0) {
    globals->max_bits = 0;
    globals->rows = 0;
    globals->sum_sq = 0.0;
    globals->sum_log = 0.0;
  }
  plan_segments(ptr_y, m, num_segments, per_item, work_start, partial);
}

} // namespace

bool nearest_feat_supported(int n, int m, int d, int num_segments) {
  if (d <= 8 || d > 128)
    return false;
  if (const char *env = std::getenv("PCA_NEAREST_FEAT")) {
    if (env[0] == '0')
      return false;
    if (env[0] == '1')
      return true;
  }
  // A tile of queries scans its whole segment: long segments need enough tiles
  // to fill the device, the kernel behind knn_mfma_impl.hpp slices them
  // instead.  Measured, us (knn_mfma / this one): 1,000 queries x 200,000 rows
  // x 64 components 475 / 2,164, 10,000 x 200,000 1,016 / 2,097, 60,000 x
  // 200,000 4,646 / 2,557; 1,000 x 4,096 x 64 207 / 96, 10,000 x 64 x 16
  // 65 / 54, 100,000 x 1,000 x 48 255 / 83.
  return m / 128 + num_segments >= 192 || n / num_segments <= 8192;
}

size_t nearest_feat_scratch_bytes(int n, int d) {
  return pack_bytes(n, d) + align256(sizeof(float) * (size_t)n) +
         align256(sizeof(NearestFeatGlobals));
}

hipError_t launch_nearest_feat(const SearchInput &in, int *work_start,
                               void *scratch, int64_t *out,
                               hipEvent_t time_start, hipEvent_t time_stop,
                               hipStream_t stream) {
  char *base = static_cast<char *>(scratch);
  NearestFeatParams p;
  p.x = static_cast<const float *>(in.x);
  p.y = static_cast<const float *>(in.y);
  p.ptr_x = in.ptr_x;
  p.ptr_y = in.ptr_y;
  p.n = in.n;
  p.m = in.m;
  p.d = in.d;
  p.num_segments = in.num_segments;
  p.work_start = work_start;
  p.pack = reinterpret_cast<const uint4 *>(base);
  base += pack_bytes(in.n, in.d);
  float *weight = reinterpret_cast<float *>(base);
  base += align256(sizeof(float) * (size_t)in.n);
  NearestFeatGlobals *globals = reinterpret_cast<NearestFeatGlobals *>(base);
  p.weight = weight;
  p.globals = globals;
  p.out = out;
  const int sets = sets_of(in.m, in.d);
  const int per_item = sets * 128;
  hipLaunchKernelGGL(nearest_feat_plan_kernel, dim3(1), dim3(kPlanThreads), 0,
                     stream, in.ptr_y, in.m, in.num_segments, per_item,
                     work_start, globals);
  const int row_blocks =
      std::max(1, std::min(128, (in.n + kBlock / 16 - 1) / (kBlock / 16)));
  hipLaunchKernelGGL(nearest_feat_rows_kernel, dim3(row_blocks), dim3(kBlock),
                     0, stream, p.x, in.n, in.d, weight, globals);
  const int grid = plan_upper_bound(in.m, in.num_segments, per_item);
  if (time_start)
    (void)hipEventRecord(time_start, stream);
  hipError_t err;
  switch (blocks_of(in.d)) {
  case 1:
    err = launch_nearest_feat_blocks<1>(p, sets, grid, stream);
    break;
  case 2:
    err = launch_nearest_feat_blocks<2>(p, sets, grid, stream);
    break;
  case 3:
    err = launch_nearest_feat_blocks<3>(p, sets, grid, stream);
    break;
  case 4:
    err = launch_nearest_feat_blocks<4>(p, sets, grid, stream);
    break;
  case 5:
    err = launch_nearest_feat_blocks<5>(p, sets, grid, stream);
    break;
  case 6:
    err = launch_nearest_feat_blocks<6>(p, sets, grid, stream);
    break;
  case 7:
    err = launch_nearest_feat_blocks<7>(p, sets, grid, stream);
    break;
  default:
    err = launch_nearest_feat_blocks<8>(p, sets, grid, stream);
    break;
  }
  if (time_stop)
    (void)hipEventRecord(time_stop, stream);
  return err;
}

} // namespace pca
