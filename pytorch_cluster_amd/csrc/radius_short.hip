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
//
// The rule that takes a call here knows the mean length only, and of ids only
// the number of examples an earlier call met, so an example may be of any
// length.  Those of more than kShortRows rows are searched by the workgroups
// that hold their queries, one example after the other: 512 rows at a time in
// LDS, the distances of 64 rows x 64 queries of a wave by fp32 matrix
// instructions.  Bound by that wave's chain -- operands from LDS, products,
// gathered signs, the rows that pass one by one -- at one wave per SIMD: 12 ns
// per row of the example (as plain fp32 instructions on broadcast rows the LDS
// alone would take that).  Graphs of 1,000 examples of 35 rows and one of 2,000
// / 20,000 / 60,000, r = 2, us a call (query after query by waves / so / the
// matrix-core kernel with its pointers and plan): 381 / 4,113 / 12,250, now 82 /
// 275 / 681, 232 / 354 / 785.  Only where few short examples share a call with
// a long one that kernel is the faster one still: 300 of 35 rows and one of
// 20,000 275 / 226.
#include "device_utils.hpp"
#include "knn_lowd_impl.hpp"
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
// longest example a lane goes through by itself: 1,000 examples of 5 - 240
// rows, r = 5, take 77 us a call, with those beyond 192 rows searched by their
// workgroups 96 us; one of 1,000 rows among 1,000 of 35 takes 135 us by lanes
// and 72 us by workgroups
constexpr int kShortRows = 256;
constexpr int kLongTile = 512; // rows of a longer one in LDS
// start values of the filter's sum for rows and queries beyond its range
constexpr float kLongNever = 3e38f;
constexpr float kLongAlways = -3e38f;
typedef float long_acc_t __attribute__((ext_vector_type(16)));

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
  constexpr int W = kBlock / kWave;
  constexpr int K = D <= 3 ? 4 : 6;            // x .. | |x|^2 | 0
  constexpr int AT_W = D;                      // plane of |x|^2
  constexpr int STRIDE = kLongTile + 32;       // (both halves: other banks)
  __shared__ float tile[K][STRIDE];
  __shared__ int waiting_rows[W][2];
  __shared__ long long sums[W];
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
  // (no distance is below an r^2 of 0 or NaN, nor from a query that is not
  // finite)
  bool finite_query = true;
#pragma unroll
  for (int c = 0; c < D; ++c)
    finite_query = finite_query && __builtin_fabsf(yq[c]) < __builtin_inff();
  bool is_long = len > kShortRows && finite_query && p.r2 > 0.0f;
  const int own = len > kShortRows ? 0 : len;
  int longest = own;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1)
    longest = max(longest, __shfl_xor(longest, sh));
  int *slot = p.out_idx + (size_t)q_in * p.slots;
  for (int i0 = 0; i0 < longest; i0 += U) {
    if (!__any(i0 < own && count < p.slots))
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
                       i0 + u < own && count < p.slots &&
                       !(p.ignore_same_index && g == q);
      if (hit) {
        slot[count] = g;
        ++count;
      }
    }
  }

  // ---- long examples ----------------------------------------------------------
  // With t = |x|^2 - 2 x.y + c, c = |y|^2 - r^2 - margin, from fp32 matrix
  // instructions: a row with a computed distance below r^2 has t < 0.  (Such a
  // row has |x|^2 <= 2 |y|^2 + 2 r^2 (1 + 2^-20); the roundings of |x|^2, |y|^2,
  // c and of a sum of six terms are each within 2^-24 of |x|^2 + 2 |x| |y| +
  // |y|^2 + r^2, 72 |y|^2 + 60 r^2 of them in all; the margin holds 128 of both,
  // and 1e-36 for what is flushed to zero.)  Whether a row with t < 0 is a
  // neighbour is decided by the distance.
  if (__syncthreads_or(is_long)) {
    const int wave = tid / kWave;
    const int half = lane >> 5;
    const int col = lane & 31;
    // the queries of both halves of the wave: B operands and start values
    float yb[2][K / 2], start[2];
    {
      float sq = 0.0f;
#pragma unroll
      for (int c = 0; c < D; ++c)
        sq = __builtin_fmaf(yq[c], yq[c], sq);
      // (a query beyond 1e30, or such an r^2: every row is looked at)
      const bool moderate = sq <= kFilterNormLimit && p.r2 <= kFilterNormLimit;
      float operand[K];
#pragma unroll
      for (int c = 0; c < K; ++c)
        operand[c] = c < D ? (moderate ? -2.0f * yq[c < D ? c : 0] : 0.0f)
                           : (c == AT_W ? 1.0f : 0.0f);
      const float margin =
          __builtin_fmaf(7.62939453125e-06f, sq + p.r2, 1e-36f);
      const float begin = moderate ? (sq - p.r2) - margin : kLongAlways;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        start[s] = __shfl(begin, 32 * s + col);
#pragma unroll
        for (int i = 0; i < K / 2; ++i) {
          const float lower = __shfl(operand[2 * i], 32 * s + col);
          const float upper = __shfl(operand[2 * i + 1], 32 * s + col);
          yb[s][i] = half ? upper : lower;
        }
      }
    }
    for (;;) {
      // the example of the workgroup's first query that waits (every wave has
      // read the one before: at least one barrier per tile lies between)
      const uint64_t waits = __ballot(is_long);
      const int first = waits != 0 ? (int)__builtin_ctzll(waits) : 0;
      if (lane == first) {
        waiting_rows[wave][0] = x_begin;
        waiting_rows[wave][1] = is_long ? x_end : x_begin;
      }
      __syncthreads();
      int begin = 0, end = 0;
#pragma unroll
      for (int w = W - 1; w >= 0; --w)
        if (waiting_rows[w][1] > waiting_rows[w][0]) {
          begin = __builtin_amdgcn_readfirstlane(waiting_rows[w][0]);
          end = __builtin_amdgcn_readfirstlane(waiting_rows[w][1]);
        }
      if (end <= begin)
        break;
      const bool mine = is_long && x_begin == begin && x_end == end;
      is_long = is_long && !mine;
      // a tile waits in registers while the one before it is searched
      constexpr int PT = kLongTile / kBlock;
      float staged[PT][D];
      auto load = [&](int base) {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          const int at = min(base + i * kBlock + tid, end - 1);
#pragma unroll
          for (int c = 0; c < D; ++c)
            staged[i][c] = p.x[(size_t)at * D + c];
        }
      };
      load(begin);
      for (int base = begin; base < end; base += kLongTile) {
        // (also: nobody reads the tile before any more)
        if (!__syncthreads_or(mine && count < p.slots))
          break;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          const int at = i * kBlock + tid;
          float sq = 0.0f;
          bool finite = true;
#pragma unroll
          for (int c = 0; c < D; ++c) {
            sq = __builtin_fmaf(staged[i][c], staged[i][c], sq);
            finite = finite && __builtin_fabsf(staged[i][c]) < __builtin_inff();
          }
          // (rows that are not finite have no distance below r^2; those
          // beyond 1e30 are always looked at, where they are)
          const bool moderate = sq <= kFilterNormLimit;
#pragma unroll
          for (int c = 0; c < D; ++c)
            tile[c][at] = moderate ? staged[i][c] : 0.0f;
          tile[AT_W][at] = base + at >= end || !finite ? kLongNever
                           : moderate                  ? sq
                                                       : kLongAlways;
#pragma unroll
          for (int c = AT_W + 1; c < K; ++c)
            tile[c][at] = 0.0f;
        }
        __syncthreads();
        if (base + kLongTile < end)
          load(base + kLongTile);
        if (!__any(mine && count < p.slots))
          continue;
        // 64 rows at a time: the chains of four products fill each other's
        // waits
        const int steps = (min(kLongTile, end - base) + 63) / 64;
        for (int step = 0; step < steps; ++step) {
          uint32_t pending[2];
          {
            long_acc_t t[2][2];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                  t[h][s][v] = start[s];
#pragma unroll
            for (int i = 0; i < K / 2; ++i)
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const float a = tile[2 * i + half][step * 64 + 32 * h + col];
#pragma unroll
                for (int s = 0; s < 2; ++s)
                  t[h][s] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                      a, yb[s][i], t[h][s], 0, 0, 0);
              }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              uint32_t rows_of[2];
#pragma unroll
              for (int s = 0; s < 2; ++s) {
                uint32_t mask = 0;
#pragma unroll
                for (int v = 0; v < 16; ++v)
                  mask = __builtin_amdgcn_alignbit(
                      mask, __float_as_uint(t[h][s][v]), 31);
                // the rows of the step in order, the first one in the highest
                // bit: nibbles of the lower and of the upper lane in turn
                uint32_t spread = (mask | (mask << 8)) & 0x00ff00ffu;
                spread = (spread | (spread << 4)) & 0x0f0f0f0fu;
                spread <<= half == 0 ? 4 : 0;
                const auto both = __builtin_amdgcn_permlane32_swap(
                    spread, spread, false, false);
                rows_of[s] = both[0] | both[1];
              }
              pending[h] = half ? rows_of[1] : rows_of[0];
            }
          }
          if (!mine || count >= p.slots)
            pending[0] = pending[1] = 0;
          while (__any((pending[0] | pending[1]) != 0)) {
            const bool later = pending[0] == 0;
            const uint32_t some = later ? pending[1] : pending[0];
            const int v = __builtin_clz(some | 1u);
            const int j = step * 64 + (later ? 32 : 0) + v;
            const int g = base + j;
            float row[D];
#pragma unroll
            for (int c = 0; c < D; ++c)
              row[c] = tile[c][j];
            if (tile[AT_W][j] == kLongAlways) {
#pragma unroll
              for (int c = 0; c < D; ++c)
                row[c] = p.x[(size_t)min(g, end - 1) * D + c];
            }
            const bool hit = some != 0 && g < end &&
                             short_distance<D>(row, yq) < p.r2 &&
                             !(p.ignore_same_index && g == q);
            const uint32_t rest = some & ~(0x80000000u >> v);
            pending[0] = later ? 0 : rest;
            pending[1] = later ? rest : pending[1];
            if (hit) {
              slot[count] = g;
              ++count;
              if (count >= p.slots)
                pending[0] = pending[1] = 0;
            }
          }
        }
      }
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
    for (int w = 0; w < W; ++w)
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
