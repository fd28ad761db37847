// Euclidean kNN for small calls (fp32, up to 4 dimensions, k <= 64): one wave
// per query.  Results are those of the reference's scalar loop
// (csrc/cuda/knn_cuda.cu:52-78), bit for bit.
//
// The kernels that scan for 128 queries per workgroup take the time of one
// scan however few queries there are: 30 us for a cloud of 1,024 points, on 8
// of 256 CUs.  Here a wave looks at 1,024 rows at a time, 16 distances per lane
// in registers.  Every lane's smallest one goes through a sort across the
// wave; the k-th of these 64 minima bounds the k-th distance (k lanes hold a
// row at or below it) and about k + k / 6 rows lie below it.  Those are handed
// to the lanes through LDS, 64 at a time, sorted by (distance, row) across the
// wave and merged with what earlier rows left: lane i holds the i-th nearest
// row.  No packed rows, no plan, no lists to insert into.
//
// Bound by the latency of its ~30 dependent exchanges and three trips to
// memory with few queries, by vector instructions (about 800 per query and
// 1,024 rows) once there are several waves per SIMD.
//
// One cloud of 1,024 points, k = 17: 6.1 us (set-up and scan before: 4 + 30).
#include "device_utils.hpp"
#include "knn_lowd_impl.hpp"
#include "launchers.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace pca {

namespace {

struct KnnWaveParams {
  const float *x;
  const float *y;
  const int64_t *ptr_x;
  const int64_t *ptr_y;
  int n, m, num_segments, k;
  DenseResult out;
};

// The value of lane `lane ^ M`.
template <int M> __device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
#define PCA_DPP(v, ctrl)                                                       \
  (uint32_t) __builtin_amdgcn_update_dpp((int)(v), (int)(v), ctrl, 0xf, 0xf,   \
                                         false)
  if (M == 1)
    return PCA_DPP(v, 0xb1); // quad_perm 1,0,3,2
  if (M == 2)
    return PCA_DPP(v, 0x4e); // quad_perm 2,3,0,1
  if (M == 4) {
    const uint32_t t = PCA_DPP(v, 0x141); // row_half_mirror: lane ^ 7
    return PCA_DPP(t, 0x1b);              // quad_perm 3,2,1,0: lane ^ 3
  }
  if (M == 8)
    return PCA_DPP(v, 0x128); // row_ror:8
#undef PCA_DPP
  const int lane = threadIdx.x & (kWave - 1);
  if (M == 16) {
    const auto both = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return lane & 16 ? both[0] : both[1];
  }
  const auto both = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return lane & 32 ? both[0] : both[1];
}
template <int M> __device__ __forceinline__ float lane_xor(float v) {
  return __uint_as_float(lane_xor<M>(__float_as_uint(v)));
}
template <int M> __device__ __forceinline__ double lane_xor(double v) {
  return __hiloint2double(
      (int)lane_xor<M>((uint32_t)__double2hiint(v)),
      (int)lane_xor<M>((uint32_t)__double2loint(v)));
}

__device__ __forceinline__ float pick(float a, float b, bool low) {
  return low ? __builtin_fminf(a, b) : __builtin_fmaxf(a, b);
}
__device__ __forceinline__ double pick(double a, double b, bool low) {
  return low ? key_min(a, b) : key_max(a, b);
}

// Steps M, M / 2 .. 1 of a bitonic merge; `up`: ascending.
template <int M, typename T>
__device__ __forceinline__ T merge_lanes(T v, int lane, bool up) {
  v = pick(v, lane_xor<M>(v), ((lane & M) == 0) == up);
  if constexpr (M > 1)
    v = merge_lanes<M / 2, T>(v, lane, up);
  return v;
}
// Ascending over the 64 lanes.
template <typename T> __device__ __forceinline__ T sort_lanes(T v, int lane) {
  v = merge_lanes<1, T>(v, lane, (lane & 2) == 0);
  v = merge_lanes<2, T>(v, lane, (lane & 4) == 0);
  v = merge_lanes<4, T>(v, lane, (lane & 8) == 0);
  v = merge_lanes<8, T>(v, lane, (lane & 16) == 0);
  v = merge_lanes<16, T>(v, lane, (lane & 32) == 0);
  return merge_lanes<32, T>(v, lane, true);
}

__device__ __forceinline__ double lane_key(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Largest b with ptr[b] <= q (all lanes the same q), 64 probes per step.
__device__ __forceinline__ int wave_segment(const int64_t *__restrict__ ptr,
                                            int num_segments, int q,
                                            int lane) {
  int lo = 0, hi = num_segments; // ptr[lo] <= q, and q < ptr[hi]
  while (hi - lo > 1) {
    const int step = (hi - lo + kWave) / (kWave + 1);
    const int at = lo + (lane + 1) * step;
    const uint64_t not_above =
        __ballot(at < hi && ptr[min(at, num_segments)] <= (int64_t)q);
    const int steps = __builtin_popcountll(not_above);
    lo += steps * step;
    hi = min(hi, lo + step);
  }
  return lo;
}

constexpr int kWaveRows = 16; // rows per lane and round

template <int D>
__global__ __launch_bounds__(kBlock) void knn_wave_kernel(KnnWaveParams p) {
  constexpr int R = kWaveRows;
  constexpr int W = kBlock / kWave;
  __shared__ double handed[W][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int q = blockIdx.x * W + wave;
  if (q >= p.m)
    return;
  const int k = p.k;
  int x_begin = 0, x_end = p.n;
  if (p.ptr_x != nullptr) {
    const int seg = __builtin_amdgcn_readfirstlane(
        wave_segment(p.ptr_y, p.num_segments, q, lane));
    x_begin = (int)p.ptr_x[seg];
    x_end = (int)p.ptr_x[seg + 1];
  }
  float yq[D];
#pragma unroll
  for (int c = 0; c < D; ++c)
    yq[c] = p.y[(size_t)q * D + c];

  double best = empty_key(); // lane i: the i-th nearest row so far
  // a row can matter if its distance is not above this (the limit itself is
  // not reached: the float below 1e10)
  float reach = __uint_as_float(__float_as_uint(kKnnSentinel) - 1u);
  for (int c0 = x_begin; c0 < x_end; c0 += R * kWave) {
    float dist[R];
    {
      float row[R][D];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int at = min(c0 + i * kWave + lane, x_end - 1);
#pragma unroll
        for (int c = 0; c < D; ++c)
          row[i][c] = p.x[(size_t)at * D + c];
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float t0 = row[i][0] - yq[0];
        float d = t0 * t0;
#pragma unroll
        for (int c = 1; c < D; ++c) {
          const float t = row[i][c] - yq[c];
          d = __builtin_fmaf(t, t, d);
        }
        // (a NaN is no distance either)
        const bool row_there = c0 + i * kWave + lane < x_end;
        dist[i] = row_there && d < kKnnSentinel ? d : __builtin_inff();
      }
    }
    if (c0 == x_begin) {
      float least = dist[0];
#pragma unroll
      for (int i = 1; i < R; ++i)
        least = __builtin_fminf(least, dist[i]);
      least = sort_lanes<float>(least, lane);
      reach = __builtin_fminf(reach, __uint_as_float(
          (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(least),
                                              k - 1)));
    }
    uint32_t left = (1u << R) - 1u;
    for (;;) {
      uint32_t mask = 0;
#pragma unroll
      for (int i = 0; i < R; ++i)
        mask |= dist[i] <= reach ? 1u << i : 0u;
      mask &= left;
      if (!__any(mask != 0))
        break;
      const int own = __builtin_popcount(mask);
      int upto = own; // inclusive sum over the lanes
#pragma unroll
      for (int sh = 1; sh < kWave; sh <<= 1) {
        const int t = __shfl_up(upto, sh);
        upto += lane >= sh ? t : 0;
      }
      const int total = __builtin_amdgcn_readlane(upto, kWave - 1);
      int slot = upto - own;
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (mask & (1u << i)) {
          if (slot < kWave) {
            handed[wave][slot] =
                make_key(dist[i], (uint32_t)(c0 + i * kWave + lane));
            left &= ~(1u << i);
          }
          ++slot;
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      double key = lane < total ? handed[wave][lane] : empty_key();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      key = sort_lanes<double>(key, lane);
      // the smaller half of both sorted sequences, sorted again
      const double turned = __shfl(key, kWave - 1 - lane);
      best = merge_lanes<32, double>(key_min(best, turned), lane, true);
      const double kth = lane_key(best, k - 1);
      if (kth < empty_key())
        reach = __builtin_fminf(reach, key_dist(kth));
      if (total <= kWave)
        break;
    }
  }

  const bool found = lane < k && best < empty_key();
  const int count = __builtin_popcountll(__ballot(found));
  const int row = key_row(best);
  const uint64_t self = __ballot(found && row == q);
  if (found) {
    p.out.idx[(size_t)q * k + lane] = row;
    if (p.out.dist != nullptr)
      p.out.dist[(size_t)q * k + lane] = key_dist(best);
  }
  if (lane == 0) {
    p.out.count[q] = count;
    if (p.out.self_pos != nullptr) {
      p.out.self_pos[q] = self != 0 ? (int)__builtin_ctzll(self) : -1;
      p.out.kept[q] = count - (self != 0 ? 1 : 0);
    }
  }
}

} // namespace

bool knn_wave_supported(int n, int m, int d, int num_segments, int k,
                        bool cosine) {
  if (cosine || d > 4 || k > kWave)
    return false;
  if (const char *env = std::getenv("PCA_KNN_WAVE")) {
    if (env[0] == '0')
      return false;
    if (env[0] == '1')
      return true;
  }
  // us of a call both ways, fitted to 632 calls of one example and of batches
  // (500 - 524,288 rows in all, 1 - 16,384 queries, k = 1 - 32).  The pick costs
  // 0.2 % over the faster path on average and at most 8 % where the examples are
  // of one size (batches with one example a hundred times longer: 28 %).
  // Every query's wave goes through all rows of its example; the scan cuts long
  // examples into slices, so it gains on this path as examples grow.  This path
  // / the scan, us, k = 16: one cloud of 1,024 points 28 / 53, of 4,096 45 / 85,
  // of 8,192 97 / 112, of 16,384 263 / 131; 4,000 queries among 20,000 rows
  // 109 / 133, among 50,000 191 / 154, among 200,000 502 / 249; 64 queries among
  // 16,384 66 / 118, among 200,000 285 / 206.
  const double rows = (double)n / num_segments;
  const double rounds = std::ceil(rows / (kWaveRows * kWave));
  const double thousands = (double)m / 1024.0;
  // Lists beyond 32 entries go through the vector-ALU scan otherwise: k = 33,
  // 1,024 points 27 / 220, 16 x 4,096 316 / 468, 64 x 4,096 1,096 / 925.
  if (k > 32)
    return thousands * (1.0 + rounds) <= 400.0;
  const double here =
      26.0 + (num_segments > 1 ? 3.0 : 0.0) +
      std::max(1.6 * rounds, thousands * (0.55 + 0.95 * rounds));
  // (without its slices, which take a look at the environment)
  const double least = 37.0 + 0.8 * k + (0.038 + 0.0025 * k) * 1e-6 * m * rows;
  if (here <= least)
    return true;
  const int slices =
      knn_lowd_config(d, k, n, m, num_segments, cosine).num_chunks;
  const double scan = least + (4.3 + 0.16 * k) * rows / slices / 1024.0 +
                      (slices > 1 ? 6.0 + 2.2 * k : 0.0);
  return here <= scan;
}

hipError_t launch_knn_wave(const SearchInput &in, int k, const DenseResult &out,
                           hipEvent_t time_start, hipEvent_t time_stop,
                           hipStream_t stream) {
  KnnWaveParams p;
  p.x = static_cast<const float *>(in.x);
  p.y = static_cast<const float *>(in.y);
  p.ptr_x = in.ptr_x;
  p.ptr_y = in.ptr_y;
  p.n = in.n;
  p.m = in.m;
  p.num_segments = in.num_segments;
  p.k = k;
  p.out = out;
  const int per_block = kBlock / kWave;
  const dim3 grid((unsigned)((in.m + per_block - 1) / per_block));
  if (time_start)
    (void)hipEventRecord(time_start, stream);
  switch (in.d) {
  case 1:
    hipLaunchKernelGGL((knn_wave_kernel<1>), grid, dim3(kBlock), 0, stream, p);
    break;
  case 2:
    hipLaunchKernelGGL((knn_wave_kernel<2>), grid, dim3(kBlock), 0, stream, p);
    break;
  case 3:
    hipLaunchKernelGGL((knn_wave_kernel<3>), grid, dim3(kBlock), 0, stream, p);
    break;
  case 4:
    hipLaunchKernelGGL((knn_wave_kernel<4>), grid, dim3(kBlock), 0, stream, p);
    break;
  default:
    return hipErrorInvalidValue;
  }
  if (time_stop)
    (void)hipEventRecord(time_stop, stream);
  return hipGetLastError();
}

} // namespace pca
