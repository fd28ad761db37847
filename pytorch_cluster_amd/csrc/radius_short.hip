// Fixed-radius neighbour search in short examples (fp32, up to 4 dimensions):
// one lane per query.  Computes what radius_kernel of the reference computes
// (csrc/cuda/radius_cuda.cu:9-42): the first max_num_neighbors rows of the
// query's example with dist < r^2, in ascending order.
//
// The other kernels give an example at least one workgroup: with a thousand
// examples of 5 - 65 rows a quarter of their queries are none, and packed rows,
// pointers and the plan are launches of their own in front.  Here 64
// consecutive queries, of whatever examples, are a wave; a lane goes through
// its own example's rows eight at a time.  Example ids are searched directly
// -- the wave finds the rows of its first and last example, its lanes theirs
// between them -- and a workgroup is one block of queries of the compaction,
// whose sum it writes itself: the whole call is this launch and the
// compaction.
//
// Bound by latency: ids, ~15 dependent probes of the searches, then a trip to
// the L2 per eight rows, the eight rows of all lanes in flight together (sixteen
// at a time measured the same: 38.8 / 39.9 us for 1,000 examples).
#include "device_utils.hpp"
#include "launchers.hpp"

#include <cstdlib>

namespace pca {

namespace {

struct RadiusShortParams {
  const float *x;
  const float *y;
  const int64_t *ptr_x; // NULL: one example
  const int64_t *ptr_y;
  SegmentSource src; // example ids instead of pointers (ids_x != NULL)
  int n, m, num_segments;
  float r2;
  int slots, ignore_same_index;
  int *out_idx;
  int *out_count;
  unsigned long long *edge_sums; // per kCompactBlockQueries queries, or NULL
};

constexpr int kShortRound = 8; // rows per lane and round
// a wave that meets a longer example takes its queries one after the other,
// 64 rows at a time
constexpr int kShortRows = 1024;

template <int D>
__device__ __forceinline__ float short_distance(const float (&row)[D],
                                                const float (&q)[D]) {
  const float t0 = row[0] - q[0];
  float dist = t0 * t0;
#pragma unroll
  for (int c = 1; c < D; ++c) {
    const float t = row[c] - q[c];
    dist = __builtin_fmaf(t, t, dist);
  }
  return dist;
}

template <int D>
__global__ __launch_bounds__(kBlock) void radius_short_kernel(
    RadiusShortParams p) {
  constexpr int U = kShortRound;
  __shared__ long long sums[kBlock / kWave];
  static_assert(kBlock == kCompactBlockQueries, "a block writes its own sum");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int q = blockIdx.x * kBlock + tid;
  const bool valid = q < p.m;
  const int q_in = min(q, p.m - 1);

  // ---- the rows of the query's example -------------------------------------
  int x_begin = 0, x_end = p.n;
  if (p.src.ids_x != nullptr) {
    const int64_t *ids = p.src.ids_x;
    // (rows with ids beyond the number of examples search the last one, as in
    // pointers_from_ids; rows with negative ids are in none)
    const int64_t id =
        min(p.src.ids_y[q_in], (int64_t)(p.num_segments - 1));
    const int64_t ends[2] = {__shfl(id, 0), __shfl(id, kWave - 1) + 1};
    int at[2];
    wave_rows_below(ids, p.n, ends, lane, at);
    int lo0 = at[0], hi0 = max(at[1], at[0]), lo1 = lo0, hi1 = hi0;
    while (__any(lo0 < hi0 || lo1 < hi1)) {
      const int mid0 = (lo0 + hi0) >> 1, mid1 = (lo1 + hi1) >> 1;
      const int64_t v0 = ids[min(mid0, p.n - 1)];
      const int64_t v1 = ids[min(mid1, p.n - 1)];
      if (lo0 < hi0) {
        lo0 = v0 < id ? mid0 + 1 : lo0;
        hi0 = v0 < id ? hi0 : mid0;
      }
      if (lo1 < hi1) {
        lo1 = v1 <= id ? mid1 + 1 : lo1;
        hi1 = v1 <= id ? hi1 : mid1;
      }
    }
    x_begin = lo0;
    x_end = id < 0 ? lo0 : lo1;
    if (p.src.examples_out != nullptr && q == 0)
      *p.src.examples_out =
          max(max(ids[p.n - 1], p.src.ids_y[p.m - 1]), (int64_t)-1) + 1;
  } else if (p.ptr_x != nullptr) {
    const int seg = find_segment64(p.ptr_y, p.num_segments, q_in);
    x_begin = (int)p.ptr_x[seg];
    x_end = (int)p.ptr_x[seg + 1];
  }
  const int len = valid ? max(x_end - x_begin, 0) : 0;

  // ---- the search -----------------------------------------------------------
  float yq[D];
#pragma unroll
  for (int c = 0; c < D; ++c)
    yq[c] = p.y[(size_t)q_in * D + c];
  int count = 0;
  int longest = len;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1)
    longest = max(longest, __shfl_xor(longest, sh));
  if (longest <= kShortRows) {
    int *slot = p.out_idx + (size_t)q_in * p.slots;
    for (int i0 = 0; i0 < longest; i0 += U) {
      if (!__any(i0 < len && count < p.slots))
        break;
      float row[U][D];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int at = min(x_begin + i0 + u, p.n - 1);
#pragma unroll
        for (int c = 0; c < D; ++c)
          row[u][c] = p.x[(size_t)at * D + c];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int g = x_begin + i0 + u;
        const bool hit = short_distance<D>(row[u], yq) < p.r2 &&
                         i0 + u < len && count < p.slots &&
                         !(p.ignore_same_index && g == q);
        if (hit) {
          slot[count] = g;
          ++count;
        }
      }
    }
  } else {
    for (int l = 0; l < kWave; ++l) {
      const int rows = __builtin_amdgcn_readlane(len, l);
      if (rows == 0)
        continue;
      const int first = __builtin_amdgcn_readlane(x_begin, l);
      const int own = __builtin_amdgcn_readlane(q, l);
      float of[D];
#pragma unroll
      for (int c = 0; c < D; ++c)
        of[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
            (int)__float_as_uint(yq[c]), l));
      int found = 0;
      for (int i0 = 0; i0 < rows && found < p.slots; i0 += kWave) {
        const int g = first + i0 + lane;
        float row[D];
#pragma unroll
        for (int c = 0; c < D; ++c)
          row[c] = p.x[(size_t)min(g, p.n - 1) * D + c];
        const bool hit = short_distance<D>(row, of) < p.r2 &&
                         i0 + lane < rows &&
                         !(p.ignore_same_index && g == own);
        const uint64_t hits = __ballot(hit);
        const int at = found + (int)__builtin_amdgcn_mbcnt_hi(
                                   (uint32_t)(hits >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)hits, 0u));
        if (hit && at < p.slots)
          p.out_idx[(size_t)own * p.slots + at] = g;
        found += __builtin_popcountll(hits);
      }
      found = min(found, p.slots);
      count = lane == l ? found : count;
    }
  }

  // ---- counts -----------------------------------------------------------------
  if (valid)
    p.out_count[q] = count;
  if (p.edge_sums == nullptr)
    return;
  long long sum = count;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1)
    sum += __shfl_xor(sum, sh);
  if (lane == 0)
    sums[tid / kWave] = sum;
  __syncthreads();
  if (tid == 0) {
    long long all = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w)
      all += sums[w];
    p.edge_sums[blockIdx.x] = (unsigned long long)all;
  }
}

} // namespace

bool radius_short_supported(int d, int n, int m, int num_segments) {
  if (d < 1 || d > 4)
    return false;
  // PCA_RADIUS_SHORT=0 / 1: never / whenever the dimension fits (tests); a
  // forced choice of the matrix cores stands
  if (const char *env = std::getenv("PCA_RADIUS_SHORT")) {
    if (env[0] == '0')
      return false;
    if (env[0] == '1')
      return true;
  }
  if (std::getenv("PCA_RADIUS_MATRIX_CORES") != nullptr)
    return false;
  // A lane's time grows with its example.  radius_graph, whole calls, us, the
  // kernels before / this one, many and few neighbours: 1,000 examples of 5 -
  // 65 rows 64 / 39 and 52 / 39, 4,000 131 / 59 and 86 / 46, 16 35 / 33 and
  // 38 / 36; of 100 - 156 rows 1,000 examples 105 / 65 and 65 / 52, 300 67 / 50
  // and 51 / 47, but 16 38 / 44 (a wave per eight queries has less to wait for
  // then); of 200 - 312 rows 1,000 examples 153 / 118 and 83 / 83, 100 67 / 63
  // and 50 / 58.
  const int rows = n / num_segments;
  return num_segments > 1 && (rows <= 64 || (rows <= 128 && m >= 16384));
}

hipError_t launch_radius_short(const SearchInput &in, float r2,
                               bool ignore_same_index, const DenseResult &out,
                               hipStream_t stream, const SegmentSource *src) {
  RadiusShortParams p;
  p.x = static_cast<const float *>(in.x);
  p.y = static_cast<const float *>(in.y);
  p.ptr_x = in.ptr_x;
  p.ptr_y = in.ptr_y;
  if (src)
    p.src = *src;
  p.n = in.n;
  p.m = in.m;
  p.num_segments = in.num_segments;
  p.r2 = r2;
  p.slots = out.slots;
  p.ignore_same_index = ignore_same_index ? 1 : 0;
  p.out_idx = out.idx;
  p.out_count = out.count;
  p.edge_sums = out.edge_sums;
  const dim3 grid((unsigned)((in.m + kBlock - 1) / kBlock));
  switch (in.d) {
  case 1:
    hipLaunchKernelGGL((radius_short_kernel<1>), grid, dim3(kBlock), 0, stream,
                       p);
    break;
  case 2:
    hipLaunchKernelGGL((radius_short_kernel<2>), grid, dim3(kBlock), 0, stream,
                       p);
    break;
  case 3:
    hipLaunchKernelGGL((radius_short_kernel<3>), grid, dim3(kBlock), 0, stream,
                       p);
    break;
  case 4:
    hipLaunchKernelGGL((radius_short_kernel<4>), grid, dim3(kBlock), 0, stream,
                       p);
    break;
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

} // namespace pca
