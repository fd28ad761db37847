// Exact Euclidean kNN over spatially binned rows: fp32 points of up to three
// dimensions, k <= 64 (more than 32 with the matrix-core scan of
// knn_binned_mc_impl.hpp only), and the radius and nearest searches over the
// same bins (further down).  This comment describes the vector-ALU kNN scan,
// the first of them, and the binning all share.  Same results, bit for bit, as the reference's scan of
// every row of the segment (csrc/cuda/knn_cuda.cu:52-78: distances as chains
// of direct differences and fused multiply-adds, neighbours by ascending
// distance, ties by ascending row, strictly below 1e10), but a query looks only
// at rows near it.
//
// Per call: every segment's x rows are ordered along a space-filling curve
// (30-bit places on a Hilbert curve through the segment's bounding box, its
// cells the voxels of the reference's grid clustering,
// csrc/cuda/grid_cuda.cu:10-25, sorted by curve_order.hip), copied in that order together
// with their row numbers, and cut into tiles of 32 rows with a bounding box
// each.  The queries are ordered the same way, so the 64 queries of a wave
// (one per lane) are neighbours in space and share one bounding box.
//
// A wave first scans the tiles around its queries' position in the order of x
// (that fills the lists and gives every query a k-th distance), then goes
// through the segment's groups of 64 tiles outwards from that position: a
// group, and inside it a tile, is looked into only if for SOME lane the
// distance from its query to the box is not above that query's k-th distance.
// Boxes are tested 64 at a time first (one per lane, against the box around
// the wave's queries and the wave's largest k-th distance); the few that pass
// are broadcast lane by lane for the per-query test (a dozen vector
// instructions per box for all 64 queries).  That box distance is
// computed with the operations of the exact chain (one difference per axis,
// product, fused multiply-adds in the same order) applied to per-axis gaps
// that are not above any row's difference: rounding is monotone, so the value
// is never above the computed distance of any row of the box, and a skipped
// tile cannot hold a neighbour.  Testing per query, not per wave, bounds the
// work of a wave whose queries straddle a jump of the curve: it pays for the
// neighbourhoods of its queries, not for the space between them.
// Rows of a scanned tile are uniform over the wave as well; a lane whose
// distance passes its own bound parks (distance, row) in a queue in LDS, and
// the queues are emptied into the sorted lists by all lanes together when one
// fills up, as in the scanning kernels.  Rows arrive out of row order here, so
// a row of EQUAL distance may still displace a neighbour with a larger row
// number: a full list admits d <= its k-th distance and the 64-bit
// (distance, row) keys decide.
//
// The curve decides how many boxes a query meets (hilbert_place).  Calls, us,
// Morton / Hilbert order: kNN of 238,000 queries among 952,000 LiDAR-like rows,
// k = 16, 713 / 649; nearest of 952,000 rows among 119,000 375 / 334.
#include "device_utils.hpp"
#include "knn_binned_mc_impl.hpp"
#include "knn_lowd_impl.hpp"
#include "launchers.hpp"

#include <climits>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace pca {

namespace {

constexpr int kBinQueueCap = 16;  // parked rows per lane

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The first launch of a binned search (a call starts with kernels so short
// that the host's launch rate sets the pace: one launch instead of many): a
// workgroup per plan counts the work items of the segments - tiles and groups of
// tiles of x, tasks of 64 and of 32 queries of y, the sort's -, the others empty
// the segment boxes, the buckets and the extra task slots.  seg_box:
// [num_segments][6] = lower corner, upper corner (ordered integers).
struct BinsSetup {
  struct Plan {
    const int64_t *ptr;
    int rows, per_item;
    int *start;
    int above; // segments of at most so many rows count none
  } plan[10];
  int plans, num_segments;
  int *seg_box;
  uint32_t *total[2]; // the sort's buckets
  int totals[2];
  // task slots (task_spans'; task_extra == 0: no tasks wanted)
  int task_blocks, task_extra;
  int *extra_used;
  int2 *task_desc;

  void add(const int64_t *ptr, int rows, int per_item, int *start,
           int above = 0) {
    plan[plans++] = {ptr, rows, per_item, start, above};
  }
  void add_sort(int side, const int64_t *ptr, int rows, void *scratch) {
    const CurveSortPlan s = curve_sort_plan(scratch, rows, num_segments);
    if (s.buckets == 0)
      return;
    add(ptr, rows, s.bucket_rows, s.bucket_start);
    add(ptr, rows, s.tile_rows, s.tile_start, s.bucket_rows);
    add(ptr, rows, s.chunk_rows, s.chunk_start, s.bucket_rows);
    total[side] = s.total;
    totals[side] = s.buckets;
  }
};
__global__ __launch_bounds__(kPlanThreads) void bins_setup_kernel(BinsSetup s) {
  __shared__ int partial[kPlanThreads];
  const int job = blockIdx.x; // (uniform over the workgroup)
  if (job < s.plans) {
    const BinsSetup::Plan p = s.plan[job];
    plan_segments(p.ptr, p.rows, s.num_segments, p.per_item, p.start, partial,
                  p.above);
  } else {
    const int i = (job - s.plans) * kPlanThreads + (int)threadIdx.x;
    if (i < 6 * s.num_segments)
      s.seg_box[i] = (i % 6) < 3 ? INT_MAX : INT_MIN;
#pragma unroll
    for (int side = 0; side < 2; ++side)
      if (i < s.totals[side])
        s.total[side][i] = 0u;
    // the extra task slots start out unused
    if (i == 0 && s.extra_used != nullptr)
      *s.extra_used = 0;
    if (i < s.task_extra)
      s.task_desc[s.task_blocks + i] = make_int2(0, 0);
  }
}
hipError_t launch_bins_setup(const BinsSetup &s, hipStream_t stream) {
  const int resets = std::max(std::max(6 * s.num_segments, s.task_extra),
                              std::max(s.totals[0], s.totals[1]));
  hipLaunchKernelGGL(
      bins_setup_kernel,
      dim3(s.plans + (resets + kPlanThreads - 1) / kPlanThreads),
      dim3(kPlanThreads), 0, stream, s);
  return hipGetLastError();
}

// Bounding box of the finite coordinates of every segment; grid (parts,
// up to 65,535 segments at a time).
__global__ __launch_bounds__(kBlock) void seg_box_kernel(
    const float *__restrict__ x, const int64_t *__restrict__ ptr_x, int n,
    int d, int seg_count, int *__restrict__ seg_box) {
  __shared__ float part[kBlock / kWave][6];
  for (int seg = blockIdx.y; seg < seg_count; seg += gridDim.y) {
    const int64_t begin = ptr_x ? ptr_x[seg] : 0;
    const int64_t end = ptr_x ? ptr_x[seg + 1] : n;
    float lo[3], hi[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      lo[c] = __builtin_inff();
      hi[c] = -__builtin_inff();
    }
    // (eight rows at a time, the last one again beyond the end)
    const int64_t step = (int64_t)gridDim.x * kBlock;
    for (int64_t i = begin + (int64_t)blockIdx.x * kBlock + threadIdx.x;
         i < end; i += 8 * step) {
      float v[8][3];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          v[u][c] = c < d ? x[(size_t)min(i + u * step, end - 1) * d + c] : 0.0f;
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (__builtin_fabsf(v[u][c]) < __builtin_inff()) {
            lo[c] = __builtin_fminf(lo[c], v[u][c]);
            hi[c] = __builtin_fmaxf(hi[c], v[u][c]);
          }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int sh = 1; sh < kWave; sh <<= 1) {
        lo[c] = __builtin_fminf(lo[c], __shfl_xor(lo[c], sh));
        hi[c] = __builtin_fmaxf(hi[c], __shfl_xor(hi[c], sh));
      }
    }
    // one set of atomic updates per workgroup
    __syncthreads(); // (the previous segment's values have been read)
    if ((threadIdx.x & (kWave - 1)) == 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        part[threadIdx.x / kWave][c] = lo[c];
        part[threadIdx.x / kWave][3 + c] = hi[c];
      }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
      float v = part[0][threadIdx.x];
      for (int w = 1; w < kBlock / kWave; ++w)
        v = threadIdx.x < 3 ? __builtin_fminf(v, part[w][threadIdx.x])
                            : __builtin_fmaxf(v, part[w][threadIdx.x]);
      if (threadIdx.x < 3)
        atomicMin(&seg_box[seg * 6 + threadIdx.x], ordered_int(v));
      else
        atomicMax(&seg_box[seg * 6 + threadIdx.x], ordered_int(v));
    }
  }
}

// Rows in curve order with their row numbers (plain and as the matrix-core
// filter takes them), and the box of every tile of 32: half a wave per tile.
__device__ __forceinline__ void
gather_tiles(int block, const float *__restrict__ x,
             const int64_t *__restrict__ ptr_x, int n, int d, int num_segments,
             const int *__restrict__ tile_start,
             const uint32_t *__restrict__ perm, float4 *__restrict__ rows,
             uint4 *__restrict__ packed, Box *__restrict__ box) {
  const int gt = (block * kBlock + (int)threadIdx.x) / kBinTile;
  const int r = threadIdx.x & (kBinTile - 1);
  // behind the last row a tile of rows that never pass the filter (operand
  // w = NaN), so that a fetch of a whole tile stays inside the copy
  if (block == 0 && threadIdx.x < kBinTile) {
    packed[(size_t)(n + r) * 2] = make_uint4(0u, 0x7fc00000u, 0u, 0u);
    packed[(size_t)(n + r) * 2 + 1] = make_uint4(0u, 0u, 0u, 0u);
  }
  if (gt >= tile_start[num_segments])
    return;
  const int seg = find_segment(tile_start, num_segments, gt);
  const int x_begin = ptr_x ? (int)ptr_x[seg] : 0;
  const int x_end = ptr_x ? (int)ptr_x[seg + 1] : n;
  const int j = x_begin + (gt - tile_start[seg]) * kBinTile + r;
  const bool ok = j < x_end;
  const uint32_t id = ok ? perm[j] : 0u;
  float v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    v[c] = (ok && c < d) ? x[(size_t)id * d + c] : 0.0f;
  if (ok) {
    // (the plain copy is read by the vector-ALU scans only)
    if (rows != nullptr)
      rows[j] = make_float4(v[0], v[1], v[2], __uint_as_float(id));
    // the operand of the matrix-core filter, then coordinates and row number
    uint4 rec[McShape<3>::REC];
    mc_pack_row<3>(v, rec);
    rec[1].w = id;
    packed[(size_t)j * 2] = rec[0];
    packed[(size_t)j * 2 + 1] = rec[1];
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // (fminf / fmaxf drop a NaN operand: a NaN coordinate is in no box, and
    // such a row has no distance below the limit either)
    float lo = ok ? v[c] : __builtin_inff();
    float hi = ok ? v[c] : -__builtin_inff();
#pragma unroll
    for (int sh = 1; sh < kBinTile; sh <<= 1) {
      lo = __builtin_fminf(lo, __shfl_xor(lo, sh));
      hi = __builtin_fmaxf(hi, __shfl_xor(hi, sh));
    }
    if (r == 0) {
      box[gt].lo[c] = lo;
      box[gt].hi[c] = hi;
    }
  }
  uint32_t min_row = ok ? id : 0xffffffffu;
#pragma unroll
  for (int sh = 1; sh < kBinTile; sh <<= 1)
    min_row = min(min_row, (uint32_t)__shfl_xor((int)min_row, sh));
  if (r == 0) {
    box[gt].min_row = min_row;
    box[gt].pad = 0u;
  }
}

// Boxes of the groups of kBinGroup consecutive tiles of a segment: one wave
// per group.
__device__ __forceinline__ void
group_boxes(int block, int num_segments, const int *__restrict__ tile_start,
            const int *__restrict__ group_start, const Box *__restrict__ box,
            Box *__restrict__ group_box) {
  const int gg = (block * kBlock + (int)threadIdx.x) / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (gg >= group_start[num_segments])
    return;
  const int seg = find_segment(group_start, num_segments, gg);
  const int t = (gg - group_start[seg]) * kBinGroup + lane;
  const int tiles = tile_start[seg + 1] - tile_start[seg];
  const bool ok = t < tiles;
  static_assert(kBinGroup == kWave, "one tile per lane");
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float lo = ok ? box[tile_start[seg] + t].lo[c] : __builtin_inff();
    float hi = ok ? box[tile_start[seg] + t].hi[c] : -__builtin_inff();
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      lo = __builtin_fminf(lo, __shfl_xor(lo, sh));
      hi = __builtin_fmaxf(hi, __shfl_xor(hi, sh));
    }
    if (lane == 0) {
      group_box[gg].lo[c] = lo;
      group_box[gg].hi[c] = hi;
    }
  }
  uint32_t min_row = ok ? box[tile_start[seg] + t].min_row : 0xffffffffu;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1)
    min_row = min(min_row, (uint32_t)__shfl_xor((int)min_row, sh));
  if (lane == 0) {
    group_box[gg].min_row = min_row;
    group_box[gg].pad = 0u;
  }
}

// The rows' tiles and the queries' tasks do not need each other: one launch for
// tiles and task classes, one for groups of tiles and task places (952,000
// queries among 119,000 rows: 9 us a call less than four launches).  Workgroups
// from tile_blocks / group_blocks on are the tasks'.
struct BinsRows {
  const float *x;
  const int64_t *ptr_x;
  int n, d, num_segments, tile_blocks, group_blocks;
  const int *tile_start, *group_start;
  const uint32_t *perm;
  float4 *rows;
  uint4 *packed;
  Box *box, *group_box;
};
struct BinsTasks {
  int groups, blocks, extra;
  int *extra_used;
  int2 *desc;
  uint32_t *cls, *order;
  int *hist;
};
__global__ __launch_bounds__(kBlock) void
tiles_and_tasks_kernel(BinsRows r, BinnedParams p, BinsTasks t) {
  const int block = blockIdx.x;
  if (block < r.tile_blocks)
    gather_tiles(block, r.x, r.ptr_x, r.n, r.d, r.num_segments, r.tile_start,
                 r.perm, r.rows, r.packed, r.box);
  else
    task_spans(p, block - r.tile_blocks, t.blocks, t.extra, t.extra_used,
               t.desc, t.cls, t.hist);
}
__global__ __launch_bounds__(kBlock) void
groups_and_tasks_kernel(BinsRows r, BinsTasks t) {
  const int block = blockIdx.x;
  if (block < r.group_blocks)
    group_boxes(block, r.num_segments, r.tile_start, r.group_start, r.box,
                r.group_box);
  else
    task_places(block - r.group_blocks, t.groups, t.blocks, t.extra,
                t.extra_used, t.cls, t.hist, t.order);
}

template <int K>
__global__ __launch_bounds__(kBlock) void knn_binned_kernel(BinnedParams p) {
  // parked rows: distance and row number, [slot][thread]
  __shared__ float queue_d[2 * kBinQueueCap][kBlock];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int task = blockIdx.x * (kBlock / kWave) +
                   __builtin_amdgcn_readfirstlane(tid / kWave);
  if (task >= p.wave_start[p.num_segments])
    return; // (whole waves leave; no barrier below)
  const int seg = find_segment(p.wave_start, p.num_segments, task);
  const int x_begin = p.ptr_x ? (int)p.ptr_x[seg] : 0;
  const int x_end = p.ptr_x ? (int)p.ptr_x[seg + 1] : p.n;
  const int y_begin = p.ptr_y ? (int)p.ptr_y[seg] : 0;
  const int y_end = p.ptr_y ? (int)p.ptr_y[seg + 1] : p.m;
  const int jq = y_begin + (task - p.wave_start[seg]) * kWave + lane;
  const bool valid = jq < y_end;
  const int q = valid ? (int)p.perm_y[jq] : 0;
  const int k = p.k;
  const int d_in = p.d;

  float yq[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    yq[c] = (valid && c < d_in) ? p.y[(size_t)q * d_in + c] : 0.0f;
  // a query with a coordinate that is not finite has no distance below the
  // limit: it looks at nothing and returns nothing
  const bool searching = valid && __builtin_fabsf(yq[0]) < __builtin_inff() &&
                         __builtin_fabsf(yq[1]) < __builtin_inff() &&
                         __builtin_fabsf(yq[2]) < __builtin_inff();

  // the wave's box (lanes that do not search stay out)
  float q_lo[3], q_hi[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float lo = searching ? yq[c] : __builtin_inff();
    float hi = searching ? yq[c] : -__builtin_inff();
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      lo = __builtin_fminf(lo, __shfl_xor(lo, sh));
      hi = __builtin_fmaxf(hi, __shfl_xor(hi, sh));
    }
    q_lo[c] = lo;
    q_hi[c] = hi;
  }

  double best[K];
#pragma unroll
  for (int j = 0; j < K; ++j)
    best[j] = (j < K - k) ? lowest_key() : empty_key();
  // a row is parked when its distance is strictly below `admit`: the limit
  // while the list has room, just above the k-th distance afterwards (a row of
  // equal distance and smaller number still gets in); nothing for a lane
  // that does not search.  `kth`: the k-th distance (the limit while the list
  // has room; below every distance for a lane that does not search): a box
  // farther away than that holds no neighbour of this lane's query.
  float admit = searching ? kKnnSentinel : -__builtin_inff();
  float kth = searching ? kKnnSentinel : -1.0f;
  // byte offset in the queue at which the lane's next row goes
  const int park_first = tid * (int)sizeof(float);
  int park_at = park_first;

  auto drain = [&]() {
    for (;;) {
      const bool has = park_at > park_first;
      if (!__any(has))
        break;
      park_at -= has ? kBlock * (int)sizeof(float) : 0;
      const float *slot = reinterpret_cast<const float *>(
          reinterpret_cast<const char *>(&queue_d[0][0]) + park_at);
      const float d = slot[0];
      const uint32_t id = __float_as_uint(slot[kBinQueueCap * kBlock]);
      // (parked under an older bound: the keys sort it out)
      const double key = (has && d < admit) ? make_key(d, id) : empty_key();
      sorted_insert<K>(best, key);
      const float now = key_dist(best[K - 1]);
      if (searching && now < kKnnSentinel) {
        kth = now;
        admit = next_up_positive(now);
      }
    }
  };

  // rows of one tile against every lane's query, four rows per step (the
  // copy of the rows is padded, so a step may read past the tile's rows;
  // FULL: the tile has all its 32 rows, no step needs a bound)
  auto scan_rows = [&](const float4 *__restrict__ src, int rows,
                       auto full) {
    constexpr bool FULL = decltype(full)::value;
    for (int r = 0; r < (FULL ? kBinTile : rows); r += 4) {
      float4 row[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        row[u] = src[r + u]; // (uniform addresses)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float d0 = row[u].x - yq[0];
        float dd = d0 * d0;
        const float d1 = row[u].y - yq[1];
        dd = __builtin_fmaf(d1, d1, dd);
        const float d2 = row[u].z - yq[2];
        dd = __builtin_fmaf(d2, d2, dd);
        const bool hit = dd < admit && (FULL || r + u < rows);
        if (hit) {
          // (one address for both queues: the row numbers sit a fixed
          // distance behind the distances)
          float *slot = reinterpret_cast<float *>(
              reinterpret_cast<char *>(&queue_d[0][0]) + park_at);
          slot[0] = dd;
          slot[kBinQueueCap * kBlock] = row[u].w;
          park_at += kBlock * (int)sizeof(float);
        }
      }
      if (__any(park_at > park_first + (kBinQueueCap - 4) * kBlock *
                                          (int)sizeof(float)))
        drain();
    }
  };
  auto scan_tile = [&](int tile) {
    const int j0 = x_begin + tile * kBinTile;
    const int rows = min(kBinTile, x_end - j0);
    if (rows == kBinTile)
      scan_rows(p.rows + j0, rows, std::true_type{});
    else
      scan_rows(p.rows + j0, rows, std::false_type{});
  };

  // largest k-th distance among the wave's queries
  auto wave_reach = [&]() {
    float r = kth;
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1)
      r = __builtin_fmaxf(r, __shfl_xor(r, sh));
    return r;
  };
  // Of the 64 boxes the lanes hold (lane l: box l, `mine` = it exists), is
  // the box of lane `src` within reach of some lane's query?  (A NaN - from an
  // infinite or empty box - never rules a box out.)
  auto reachable = [&](const Box &held, int src) {
    float lo[3], hi[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      lo[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(held.lo[c]), src));
      hi[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(held.hi[c]), src));
    }
    return __any(!(box_gap2(lo, hi, yq, yq) > kth));
  };
  const int tile0 = p.tile_start[seg];
  const int num_tiles = p.tile_start[seg + 1] - tile0;
  if (num_tiles > 0) {
    // where the wave's first and last query fall in the order of x
    const int last_lane = min(kWave, y_end - (jq - lane)) - 1;
    const uint32_t key_first =
        p.keys_y[__builtin_amdgcn_readfirstlane(jq - lane)];
    const uint32_t key_last =
        p.keys_y[__builtin_amdgcn_readfirstlane(jq - lane + last_lane)];
    const int pos_first =
        wave_lower_bound(p.keys_x, x_begin, x_end, key_first, lane);
    const int pos_last =
        wave_lower_bound(p.keys_x, x_begin, x_end, key_last, lane);
    const int t_first = min(num_tiles - 1, (pos_first - x_begin) / kBinTile);
    const int t_last = min(num_tiles - 1, (pos_last - x_begin) / kBinTile);
    // tiles seed_lo .. seed_hi are scanned up front
    int seed_lo = max(0, t_first - 1);
    int seed_hi = min(num_tiles - 1, max(t_last, t_first) + 1);
    if (seed_hi - seed_lo + 1 > kBinSeedTiles) {
      // queries far apart in the order of x: the middle of their range
      const int mid = (seed_lo + seed_hi) / 2;
      seed_lo = max(0, mid - kBinSeedTiles / 2);
      seed_hi = min(num_tiles - 1, seed_lo + kBinSeedTiles - 1);
    }
    for (int t = seed_lo; t <= seed_hi; ++t)
      scan_tile(t);
    drain();
    float reach = wave_reach();

    // Groups of tiles, 64 at a time (one box per lane), nearest to the seed
    // tiles first.  A group, then a tile, is looked into if its box is within
    // the wave's largest k-th distance of the box around the wave's queries
    // (all 64 boxes at once), and then within some query's own k-th distance
    // of that query (a dozen instructions per box).
    const int group0 = p.group_start[seg];
    const int num_groups = (num_tiles + kBinGroup - 1) / kBinGroup;
    const int centre = ((seed_lo + seed_hi) / 2) / kBinGroup;
    const int num_rounds = (num_groups + kWave - 1) / kWave;
    const int centre_round = centre / kWave;
    for (int i = 0; i < 2 * num_rounds; ++i) {
      const int round = centre_round + ((i & 1) ? -((i + 1) >> 1) : (i >> 1));
      if (round < 0 || round >= num_rounds)
        continue;
      const int g_mine = round * kWave + lane;
      Box g_box = {};
      if (g_mine < num_groups)
        g_box = p.group_box[group0 + g_mine];
      uint64_t g_todo =
          __ballot(g_mine < num_groups &&
                   !(box_gap2(g_box.lo, g_box.hi, q_lo, q_hi) > reach));
      const int g_at = min(max(centre - round * kWave, 0), kWave - 1);
      while (g_todo != 0) {
        const int g_lane = nearest_bit(g_todo, g_at);
        g_todo &= ~((uint64_t)1 << g_lane);
        if (!reachable(g_box, g_lane))
          continue;
        const int group = round * kWave + g_lane;
        const int t_mine = group * kBinGroup + lane;
        const bool t_ok =
            t_mine < num_tiles && !(t_mine >= seed_lo && t_mine <= seed_hi);
        Box t_box = {};
        if (t_ok)
          t_box = p.box[tile0 + t_mine];
        uint64_t t_todo = __ballot(
            t_ok && !(box_gap2(t_box.lo, t_box.hi, q_lo, q_hi) > reach));
        while (t_todo != 0) {
          const int t_lane = (int)__builtin_ctzll(t_todo);
          t_todo &= t_todo - 1;
          if (!reachable(t_box, t_lane))
            continue;
          scan_tile(group * kBinGroup + t_lane);
        }
        if (__any(park_at > park_first)) {
          drain();
          reach = wave_reach();
        }
      }
    }
    drain();
  }

  if (valid)
    write_dense<K>(best, k, q, p.out_idx, p.out_dist, p.out_count);
}

// The radius search over the same bins (reference: radius_kernel,
// csrc/cuda/radius_cuda.cu:9-42): every row with a squared distance strictly
// below r2, at most `slots` of them - the ones with the smallest row numbers,
// in ascending order.  The radius is known from the start, so there are no
// seed tiles: boxes at r2 or farther from every query are skipped, rows that
// qualify are parked by number, and the lists keep the `slots` smallest
// numbers (as doubles; a full list admits only smaller numbers).
template <int K>
__global__ __launch_bounds__(kBlock) void radius_binned_kernel(
    BinnedParams p, float r2, int ignore_same_index) {
  __shared__ uint32_t queue[kBinQueueCap][kBlock];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int task = blockIdx.x * (kBlock / kWave) +
                   __builtin_amdgcn_readfirstlane(tid / kWave);
  if (task >= p.wave_start[p.num_segments])
    return; // (whole waves leave; no barrier below)
  const int seg = find_segment(p.wave_start, p.num_segments, task);
  const int x_begin = p.ptr_x ? (int)p.ptr_x[seg] : 0;
  const int x_end = p.ptr_x ? (int)p.ptr_x[seg + 1] : p.n;
  const int y_begin = p.ptr_y ? (int)p.ptr_y[seg] : 0;
  const int y_end = p.ptr_y ? (int)p.ptr_y[seg + 1] : p.m;
  const int jq = y_begin + (task - p.wave_start[seg]) * kWave + lane;
  const bool valid = jq < y_end;
  const int q = valid ? (int)p.perm_y[jq] : 0;
  const int slots = p.k;
  const int d_in = p.d;

  float yq[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    yq[c] = (valid && c < d_in) ? p.y[(size_t)q * d_in + c] : 0.0f;
  // (a coordinate that is not finite: no distance below r2)
  const bool searching = valid && __builtin_fabsf(yq[0]) < __builtin_inff() &&
                         __builtin_fabsf(yq[1]) < __builtin_inff() &&
                         __builtin_fabsf(yq[2]) < __builtin_inff();
  float q_lo[3], q_hi[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float lo = searching ? yq[c] : __builtin_inff();
    float hi = searching ? yq[c] : -__builtin_inff();
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      lo = __builtin_fminf(lo, __shfl_xor(lo, sh));
      hi = __builtin_fmaxf(hi, __shfl_xor(hi, sh));
    }
    q_lo[c] = lo;
    q_hi[c] = hi;
  }

  double best[K];
#pragma unroll
  for (int j = 0; j < K; ++j)
    best[j] = (j < K - slots) ? -__builtin_inf() : __builtin_inf();
  // rows with a number below `below` are parked: all while the list has
  // room, those under its largest number afterwards; none for a lane that
  // does not search
  uint32_t below = searching ? 0xffffffffu : 0u;
  const uint32_t self = ignore_same_index ? (uint32_t)q : 0xffffffffu;
  // a lane without a query never passes d < limit
  const float limit = searching ? r2 : -__builtin_inff();
  int parked = 0;

  auto drain = [&]() {
    for (;;) {
      const bool has = parked > 0;
      if (!__any(has))
        break;
      parked -= has ? 1 : 0;
      const uint32_t id = queue[has ? parked : 0][tid];
      const double key = (has && id < below) ? (double)id : __builtin_inf();
      sorted_insert<K>(best, key);
      if (searching && best[K - 1] < __builtin_inf())
        below = (uint32_t)best[K - 1];
    }
  };

  auto scan_tile = [&](int tile) {
    const int j0 = x_begin + tile * kBinTile;
    const int rows = min(kBinTile, x_end - j0);
    const float4 *__restrict__ src = p.rows + j0;
    for (int r = 0; r < rows; r += 4) {
      float4 row[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        row[u] = src[r + u]; // (uniform addresses; the copy is padded)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float d0 = row[u].x - yq[0];
        float dd = d0 * d0;
        const float d1 = row[u].y - yq[1];
        dd = __builtin_fmaf(d1, d1, dd);
        const float d2 = row[u].z - yq[2];
        dd = __builtin_fmaf(d2, d2, dd);
        const uint32_t id = __float_as_uint(row[u].w);
        const bool hit = dd < limit && id < below && id != self &&
                         r + u < rows;
        if (hit) {
          queue[parked][tid] = id;
          ++parked;
        }
      }
      if (__any(parked > kBinQueueCap - 4))
        drain();
    }
  };

  // is the box of lane `src` closer than the radius to some lane's query?
  // (A NaN - from an infinite or empty box - never rules a box out.)
  auto reachable = [&](const Box &held, int src) {
    float lo[3], hi[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      lo[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(held.lo[c]), src));
      hi[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(held.hi[c]), src));
    }
    return __any(searching && !(box_gap2(lo, hi, yq, yq) >= r2));
  };

  const int tile0 = p.tile_start[seg];
  const int num_tiles = p.tile_start[seg + 1] - tile0;
  const int group0 = p.group_start[seg];
  const int num_groups = (num_tiles + kBinGroup - 1) / kBinGroup;
  if (__any(searching)) {
    for (int g_base = 0; g_base < num_groups; g_base += kWave) {
      const int g_mine = g_base + lane;
      Box g_box = {};
      if (g_mine < num_groups)
        g_box = p.group_box[group0 + g_mine];
      uint64_t g_todo =
          __ballot(g_mine < num_groups &&
                   !(box_gap2(g_box.lo, g_box.hi, q_lo, q_hi) >= r2));
      while (g_todo != 0) {
        const int g_lane = (int)__builtin_ctzll(g_todo);
        g_todo &= g_todo - 1;
        if (!reachable(g_box, g_lane))
          continue;
        const int group = g_base + g_lane;
        const int t_mine = group * kBinGroup + lane;
        Box t_box = {};
        if (t_mine < num_tiles)
          t_box = p.box[tile0 + t_mine];
        uint64_t t_todo =
            __ballot(t_mine < num_tiles &&
                     !(box_gap2(t_box.lo, t_box.hi, q_lo, q_hi) >= r2));
        while (t_todo != 0) {
          const int t_lane = (int)__builtin_ctzll(t_todo);
          t_todo &= t_todo - 1;
          if (reachable(t_box, t_lane))
            scan_tile(group * kBinGroup + t_lane);
        }
        if (__any(parked > 0))
          drain();
      }
    }
  }

  if (valid) {
    const size_t row = (size_t)q * slots;
    int found = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int e = j - (K - slots);
      if (e >= 0 && best[j] < __builtin_inf()) {
        p.out_idx[row + e] = (int)best[j];
        ++found;
      }
    }
    p.out_count[q] = found;
  }
}

struct BinnedLayout {
  size_t seg_box, keys_x, keys_y, perm_x, perm_y, rows, packed, box, group_box,
      tile_start, group_start, wave_start, half_start, task_keys, sort_x,
      sort_y;
  int tiles_bound, groups_bound;
  size_t total() const {
    return seg_box + keys_x + keys_y + perm_x + perm_y + rows + packed + box +
           group_box + tile_start + group_start + wave_start + half_start +
           task_keys + sort_x + sort_y;
  }
};

// Keys are 32 bits: the segment above the place on the curve, whose bits per axis
// (at most 10) shrink as the segments get more (and with that smaller).
int segment_bits(int num_segments) {
  int bits = 0;
  while (bits < 31 && ((int64_t)1 << bits) < num_segments)
    ++bits;
  return bits;
}
int axis_bits(int num_segments) {
  return std::min(10, (32 - segment_bits(num_segments)) / 3);
}

// Tasks in a row that one XCD takes, as a power of two: long runs keep what a
// task fetches in the L2 its neighbours fill (256 in a row: 258 MB fetched by
// the search kernel of the 1 M-point workload, 8 in a row: 594 MB, at the
// same speed), but every XCD needs a few runs for its share of the long tasks
// at the front of the order.  PCA_BINNED_XCD_RUN_LOG2 overrides.
int xcd_run_log2(int tasks) {
  static const int fixed = [] {
    const char *text = std::getenv("PCA_BINNED_XCD_RUN_LOG2");
    if (!text)
      return -1;
    const int v = std::atoi(text);
    return v < 0 ? 0 : (v > 12 ? 12 : v);
  }();
  if (fixed >= 0)
    return fixed;
  int log2 = 3;
  while (log2 < 8 && (size_t)(8 << (log2 + 1)) * 3 <= (size_t)tasks)
    ++log2;
  return log2;
}

// Workgroups of a search on matrix cores: whole runs on each of the 8 XCDs.
int xcd_run_grid(int tasks) {
  const int unit = 8 << xcd_run_log2(tasks);
  return (tasks + unit - 1) / unit * unit;
}

// Task slots for `blocks` blocks of 32 queries: one each, and half as many
// again for the parts of split blocks - while the blocks are not many more
// than the waves the device holds at once (256 CUs x 4 SIMDs x 4 waves).  With
// several rounds of waves the long tasks, started first, are covered by the
// others, and splitting only adds work (measured: it gains 15-25 % up to
// ~4,000 blocks and loses 5 % at 8,000).
int task_slots(int blocks) {
  return blocks <= 6144 ? blocks + (blocks / 6) * 3 : blocks;
}

// Words of the task-slot buffer (see TaskBuffers).
size_t task_buffer_words(int m, int num_segments) {
  const int blocks = plan_upper_bound(m, num_segments, kWave / 2);
  const int groups = (blocks + kBlock - 1) / kBlock;
  return 64 + 4 * (size_t)task_slots(blocks) + (size_t)kTaskClasses * groups;
}

BinnedLayout binned_layout(int n, int m, int num_segments) {
  BinnedLayout w;
  w.seg_box = align256(sizeof(int) * 6 * (size_t)num_segments);
  w.keys_x = align256(sizeof(uint32_t) * (size_t)n);
  w.keys_y = align256(sizeof(uint32_t) * (size_t)m);
  w.perm_x = align256(sizeof(uint32_t) * (size_t)n);
  w.perm_y = align256(sizeof(uint32_t) * (size_t)m);
  // (padded: the search reads rows four at a time)
  w.rows = align256(sizeof(float4) * ((size_t)n + kBinTile));
  w.packed = align256(sizeof(uint4) * 2 * ((size_t)n + kBinTile));
  w.tiles_bound = plan_upper_bound(n, num_segments, kBinTile);
  w.groups_bound = plan_upper_bound(n, num_segments, kBinTile * kBinGroup);
  w.box = align256(sizeof(Box) * (size_t)w.tiles_bound);
  w.group_box = align256(sizeof(Box) * (size_t)w.groups_bound);
  w.tile_start = align256(sizeof(int) * (size_t)(num_segments + 1));
  w.group_start = align256(sizeof(int) * (size_t)(num_segments + 1));
  w.wave_start = align256(sizeof(int) * (size_t)(num_segments + 1));
  w.half_start = align256(sizeof(int) * (size_t)(num_segments + 1));
  // per task slot: descriptor (2 words), class, place in the starting order;
  // a histogram of the classes per kBlock blocks
  w.task_keys = align256(sizeof(uint32_t) * task_buffer_words(m, num_segments));
  w.sort_x = curve_sort_bytes(n, num_segments);
  w.sort_y = curve_sort_bytes(m, num_segments);
  return w;
}

// Everything a binned search reads, as prepare_bins leaves it in the scratch.
struct Bins {
  const int *tile_start, *group_start;
  const int *wave_start; // tasks of 64 queries
  const int *half_start; // tasks of 32 queries
  const uint32_t *keys_x, *keys_y, *perm_y;
  const float4 *rows;
  const uint4 *packed;
  const Box *box, *group_box;
  // the tasks of 32 queries in starting order (when asked for)
  const int2 *task_desc;
  const uint32_t *task_order;
  int task_slots; // slots of the order
  int task_grid;  // workgroups that cover them: whole runs of
                  // 2^xcd_run_log2(task_slots) tasks on each of 8 XCDs
  int code_bits;
};

// The pieces of the task-slot buffer.
struct TaskBuffers {
  int blocks, slots, groups; // groups: workgroups of kBlock blocks
  int *extra_used;
  int2 *desc;
  uint32_t *cls, *order;
  int *hist;
};
TaskBuffers task_buffers(uint32_t *task_keys, int m, int num_segments) {
  TaskBuffers t;
  t.blocks = plan_upper_bound(m, num_segments, kWave / 2);
  t.slots = task_slots(t.blocks);
  t.groups = (t.blocks + kBlock - 1) / kBlock;
  t.extra_used = reinterpret_cast<int *>(task_keys);
  t.desc = reinterpret_cast<int2 *>(task_keys + 64);
  t.cls = task_keys + 64 + 2 * (size_t)t.slots;
  t.order = t.cls + t.slots;
  t.hist = reinterpret_cast<int *>(t.order + t.slots);
  return t;
}

// Workgroups per segment of seg_box_kernel: enough to fill the device when
// segments are few (more of them were no quicker: their atomic updates of the
// same few words take turns).
int seg_box_parts(int n, int num_segments) {
  return std::max(1, std::min((n / num_segments + 16 * kBlock - 1) /
                                  (16 * kBlock),
                              std::max(1, 1024 / num_segments)));
}

// Orders rows and queries along the curve, copies the rows, builds the boxes;
// with `with_tasks` also the tasks of 32 queries and their starting order.
hipError_t prepare_bins(const SearchInput &in, void *scratch, bool with_tasks,
                        bool plain_rows, Bins &bins, hipStream_t stream) {
  const BinnedLayout lay = binned_layout(in.n, in.m, in.num_segments);
  char *cursor = static_cast<char *>(scratch);
  auto take = [&cursor](size_t bytes) {
    char *piece = cursor;
    cursor += bytes;
    return static_cast<void *>(piece);
  };
  int *seg_box = static_cast<int *>(take(lay.seg_box));
  uint32_t *keys_x = static_cast<uint32_t *>(take(lay.keys_x));
  uint32_t *keys_y = static_cast<uint32_t *>(take(lay.keys_y));
  uint32_t *perm_x = static_cast<uint32_t *>(take(lay.perm_x));
  uint32_t *perm_y = static_cast<uint32_t *>(take(lay.perm_y));
  float4 *rows = static_cast<float4 *>(take(lay.rows));
  uint4 *packed = static_cast<uint4 *>(take(lay.packed));
  Box *box = static_cast<Box *>(take(lay.box));
  Box *group_box = static_cast<Box *>(take(lay.group_box));
  int *tile_start = static_cast<int *>(take(lay.tile_start));
  int *group_start = static_cast<int *>(take(lay.group_start));
  int *wave_start = static_cast<int *>(take(lay.wave_start));
  int *half_start = static_cast<int *>(take(lay.half_start));
  uint32_t *task_keys = static_cast<uint32_t *>(take(lay.task_keys));
  void *sort_x = take(lay.sort_x);
  void *sort_y = take(lay.sort_y);

  const float *x = static_cast<const float *>(in.x);
  const float *y = static_cast<const float *>(in.y);
  const int nseg = in.num_segments;
  // the rows searching for themselves (the graph entry points): one order
  // serves both sides
  const bool self_search = in.y == in.x && in.m == in.n &&
                           (in.ptr_y == in.ptr_x || in.ptr_x == nullptr);
  if (self_search) {
    keys_y = keys_x;
    perm_y = perm_x;
  }
  bins.tile_start = tile_start;
  bins.group_start = group_start;
  bins.wave_start = wave_start;
  bins.half_start = half_start;
  bins.keys_x = keys_x;
  bins.keys_y = keys_y;
  bins.perm_y = perm_y;
  bins.rows = rows;
  bins.packed = packed;
  bins.box = box;
  bins.group_box = group_box;
  bins.task_desc = nullptr;
  bins.task_order = nullptr;
  bins.task_slots = 0;
  bins.task_grid = 0;
  bins.code_bits = 0;

  hipError_t err;
  {
    BinsSetup setup = {};
    setup.num_segments = nseg;
    setup.add(in.ptr_x, in.n, kBinTile, tile_start);
    setup.add(in.ptr_x, in.n, kBinTile * kBinGroup, group_start);
    setup.add(in.ptr_y, in.m, kWave, wave_start);
    setup.add(in.ptr_y, in.m, kWave / 2, half_start);
    setup.add_sort(0, in.ptr_x, in.n, sort_x);
    if (!self_search)
      setup.add_sort(1, in.ptr_y, in.m, sort_y);
    setup.seg_box = seg_box;
    const TaskBuffers t = task_buffers(task_keys, in.m, nseg);
    setup.task_blocks = t.blocks;
    setup.task_extra = with_tasks ? t.slots - t.blocks : 0;
    setup.extra_used = with_tasks ? t.extra_used : nullptr;
    setup.task_desc = t.desc;
    if ((err = launch_bins_setup(setup, stream)) != hipSuccess)
      return err;
  }
  {
    hipLaunchKernelGGL(seg_box_kernel,
                       dim3(seg_box_parts(in.n, nseg), std::min(nseg, 65535)),
                       dim3(kBlock), 0, stream, x, in.ptr_x, in.n, in.d, nseg,
                       seg_box);
  }
  if ((err = hipGetLastError()) != hipSuccess)
    return err;

  const CurveSortSide sides[2] = {{x, in.ptr_x, in.n, sort_x, keys_x, perm_x},
                                  {y, in.ptr_y, in.m, sort_y, keys_y, perm_y}};
  if ((err = launch_curve_sort(sides, self_search ? 1 : 2, in.d, nseg,
                               axis_bits(nseg), seg_box, stream)) != hipSuccess)
    return err;
  // the rows' tiles; the tasks (blocks of 32 queries, long spans split) and their
  // starting order, from the sorted keys of the queries (the extra slots were
  // cleared by bins_setup_kernel)
  const TaskBuffers t = task_buffers(task_keys, in.m, nseg);
  const BinsTasks tasks = {t.groups, t.blocks, t.slots - t.blocks,
                           t.extra_used, t.desc, t.cls, t.order, t.hist};
  const int per_block = kBlock / kBinTile, groups_per_block = kBlock / kWave;
  const BinsRows r = {
      x,        in.ptr_x,   in.n,
      in.d,     nseg,       (lay.tiles_bound + per_block - 1) / per_block,
      (lay.groups_bound + groups_per_block - 1) / groups_per_block,
      tile_start, group_start, perm_x, plain_rows ? rows : nullptr, packed,
      box,      group_box};
  BinnedParams p; // (what task_spans reads)
  memset(&p, 0, sizeof(p));
  p.ptr_y = in.ptr_y;
  p.m = in.m;
  p.num_segments = nseg;
  p.wave_start = half_start;
  p.keys_y = keys_y;
  p.code_bits = 3 * axis_bits(nseg);
  const int task_blocks = with_tasks ? t.groups : 0;
  hipLaunchKernelGGL(tiles_and_tasks_kernel, dim3(r.tile_blocks + task_blocks),
                     dim3(kBlock), 0, stream, r, p, tasks);
  hipLaunchKernelGGL(groups_and_tasks_kernel,
                     dim3(r.group_blocks + task_blocks), dim3(kBlock), 0,
                     stream, r, tasks);
  if (with_tasks) {
    bins.task_desc = t.desc;
    bins.task_order = t.order;
    bins.task_slots = t.slots;
    bins.task_grid = xcd_run_grid(t.slots);
    bins.code_bits = p.code_bits;
  }
  return hipGetLastError();
}

void fill_params(BinnedParams &p, const SearchInput &in, const Bins &bins,
                 const DenseResult &out) {
  p.y = static_cast<const float *>(in.y);
  p.ptr_x = in.ptr_x;
  p.ptr_y = in.ptr_y;
  p.n = in.n;
  p.m = in.m;
  p.d = in.d;
  p.num_segments = in.num_segments;
  p.tile_start = bins.tile_start;
  p.wave_start = bins.wave_start;
  p.keys_x = bins.keys_x;
  p.keys_y = bins.keys_y;
  p.perm_y = bins.perm_y;
  p.rows = bins.rows;
  p.packed = bins.packed;
  p.box = bins.box;
  p.group_start = bins.group_start;
  p.group_box = bins.group_box;
  p.out_idx = out.idx;
  p.out_dist = out.dist;
  p.out_count = out.count;
  p.out_nearest = nullptr;
  p.task_order = bins.task_order;
  p.task_desc = bins.task_desc;
  p.task_slots = bins.task_slots;
  p.xcd_run_log2 = xcd_run_log2(bins.task_slots);
  p.code_bits = bins.code_bits;
}

} // namespace

// The rows of every segment in curve order, for kernels that look at them in
// that order only (fps): boxes, keys and the sort of prepare_bins.
namespace {
struct CurveLayout {
  size_t seg_box, keys, perm, sort;
  size_t total() const { return seg_box + keys + perm + sort; }
};
CurveLayout curve_layout(int n, int num_segments) {
  CurveLayout w;
  w.seg_box = align256(sizeof(int) * 6 * (size_t)num_segments);
  w.keys = w.perm = align256(sizeof(uint32_t) * (size_t)n);
  w.sort = curve_sort_bytes(n, num_segments);
  return w;
}
} // namespace

size_t curve_order_bytes(int n, int num_segments) {
  return curve_layout(n, num_segments).total();
}

hipError_t launch_curve_order(const float *x, const int64_t *ptr, int n, int d,
                              int num_segments, void *scratch,
                              const uint32_t **perm, hipStream_t stream) {
  const CurveLayout lay = curve_layout(n, num_segments);
  char *cursor = static_cast<char *>(scratch);
  auto take = [&cursor](size_t bytes) {
    char *piece = cursor;
    cursor += bytes;
    return static_cast<void *>(piece);
  };
  int *seg_box = static_cast<int *>(take(lay.seg_box));
  uint32_t *keys = static_cast<uint32_t *>(take(lay.keys));
  uint32_t *order = static_cast<uint32_t *>(take(lay.perm));
  void *sort = take(lay.sort);
  *perm = order;
  BinsSetup setup = {};
  setup.num_segments = num_segments;
  setup.seg_box = seg_box;
  setup.add_sort(0, ptr, n, sort);
  hipError_t err = launch_bins_setup(setup, stream);
  if (err != hipSuccess)
    return err;
  hipLaunchKernelGGL(seg_box_kernel,
                     dim3(seg_box_parts(n, num_segments),
                          std::min(num_segments, 65535)),
                     dim3(kBlock), 0, stream, x, ptr, n, d, num_segments,
                     seg_box);
  if ((err = hipGetLastError()) != hipSuccess)
    return err;
  const CurveSortSide side = {x, ptr, n, sort, keys, order};
  return launch_curve_sort(&side, 1, d, num_segments, axis_bits(num_segments),
                           seg_box, stream);
}

bool knn_binned_supported(int d, int k, bool cosine) {
  return !cosine && d >= 1 && d <= 3 && k >= 1 && k <= 64;
}

size_t knn_binned_scratch_bytes(int n, int m, int num_segments) {
  return binned_layout(n, m, num_segments).total();
}

hipError_t launch_knn_binned(const SearchInput &in, int k, void *scratch,
                             const DenseResult &out, hipEvent_t time_start,
                             hipEvent_t time_stop, hipStream_t stream) {
  if (time_start)
    (void)hipEventRecord(time_start, stream);
  // (diagnostic switch: the vector-ALU scan instead of the matrix-core one)
  // (lists of more than 32 entries exist for the matrix-core scan only)
  const char *env = getenv("PCA_KNN_BINNED_MATRIX_CORES");
  const bool matrix_cores = k > 32 || !(env != nullptr && env[0] == '0');
  Bins bins;
  const hipError_t err =
      prepare_bins(in, scratch, matrix_cores, !matrix_cores, bins, stream);
  if (err != hipSuccess)
    return err;
  BinnedParams p;
  fill_params(p, in, bins, out);
  p.k = k;
  if (matrix_cores)
    p.wave_start = bins.half_start;
  const int waves = plan_upper_bound(in.m, in.num_segments, kWave);
  const int grid = (waves + kBlock / kWave - 1) / (kBlock / kWave);
  const int slots = bins.task_grid;
#define PCA_BINNED_LAUNCH(K_)                                                  \
  do {                                                                         \
    if (matrix_cores)                                                          \
      hipLaunchKernelGGL((knn_binned_mc_kernel<K_>), dim3(slots),              \
                         dim3(kBinMcBlock), 0, stream, p);                     \
    else                                                                       \
      hipLaunchKernelGGL((knn_binned_kernel<K_>), dim3(grid), dim3(kBlock), 0, \
                         stream, p);                                           \
  } while (0)
#define PCA_BINNED_LAUNCH_WIDE(K_)                                             \
  hipLaunchKernelGGL((knn_binned_mc_kernel<K_>), dim3(slots),                  \
                     dim3(kBinMcBlock), 0, stream, p)
  // (list widths in steps of 8: the bound shared by the two lanes of a query
  // reads one of the five middle entries of a list)
  if (k <= 8)
    PCA_BINNED_LAUNCH(8);
  else if (k <= 16)
    PCA_BINNED_LAUNCH(16);
  else if (k <= 24)
    PCA_BINNED_LAUNCH(24);
  else if (k <= 32)
    PCA_BINNED_LAUNCH(32);
  else if (k <= 40)
    PCA_BINNED_LAUNCH_WIDE(40);
  else if (k <= 48)
    PCA_BINNED_LAUNCH_WIDE(48);
  else if (k <= 56)
    PCA_BINNED_LAUNCH_WIDE(56);
  else
    PCA_BINNED_LAUNCH_WIDE(64);
#undef PCA_BINNED_LAUNCH_WIDE
#undef PCA_BINNED_LAUNCH
  if (time_stop)
    (void)hipEventRecord(time_stop, stream);
  return hipGetLastError();
}

hipError_t launch_nearest_binned(const SearchInput &in, void *scratch,
                                 int64_t *out, hipEvent_t time_start,
                                 hipEvent_t time_stop, hipStream_t stream) {
  if (time_start)
    (void)hipEventRecord(time_start, stream);
  Bins bins;
  const hipError_t err = prepare_bins(in, scratch, true, false, bins, stream);
  if (err != hipSuccess)
    return err;
  BinnedParams p;
  const DenseResult none{nullptr, nullptr, nullptr, 1};
  fill_params(p, in, bins, none);
  p.k = 1;
  p.out_nearest = out;
  p.wave_start = bins.half_start;
  hipLaunchKernelGGL((knn_binned_mc_kernel<1, true>), dim3(bins.task_grid),
                     dim3(kBinMcBlock), 0, stream, p);
  if (time_stop)
    (void)hipEventRecord(time_stop, stream);
  return hipGetLastError();
}

bool radius_binned_supported(int d, int slots) {
  return d >= 1 && d <= 3 && slots >= 1 && slots <= 64;
}

hipError_t launch_radius_binned(const SearchInput &in, float r2,
                                bool ignore_same_index, void *scratch,
                                const DenseResult &out, hipStream_t stream) {
  // (diagnostic switch: the vector-ALU scan instead of the matrix-core one)
  // (lists of more than 32 entries exist for the matrix-core scan only)
  const char *env = getenv("PCA_RADIUS_BINNED_MATRIX_CORES");
  const bool matrix_cores =
      out.slots > 32 || !(env != nullptr && env[0] == '0');
  Bins bins;
  const hipError_t err =
      prepare_bins(in, scratch, false, !matrix_cores, bins, stream);
  if (err != hipSuccess)
    return err;
  BinnedParams p;
  fill_params(p, in, bins, out);
  p.k = out.slots;
  const int same = ignore_same_index ? 1 : 0;
  const int per_task = matrix_cores ? kWave / 2 : kWave;
  if (matrix_cores)
    p.wave_start = bins.half_start;
  const int waves = plan_upper_bound(in.m, in.num_segments, per_task);
  const int grid = (waves + kBlock / kWave - 1) / (kBlock / kWave);
  p.xcd_run_log2 = xcd_run_log2(waves); // (tasks in curve order, no slots)
#define PCA_BINNED_LAUNCH(K_)                                                  \
  do {                                                                         \
    if (matrix_cores)                                                          \
      hipLaunchKernelGGL((radius_binned_mc_kernel<K_>),                        \
                         dim3(xcd_run_grid(waves)), dim3(kBinMcBlock), 0,   \
                         stream, p, r2, same);                                 \
    else                                                                       \
      hipLaunchKernelGGL((radius_binned_kernel<K_>), dim3(grid), dim3(kBlock), \
                         0, stream, p, r2, same);                              \
  } while (0)
#define PCA_BINNED_LAUNCH_WIDE(K_)                                             \
  hipLaunchKernelGGL((radius_binned_mc_kernel<K_>),                            \
                     dim3(xcd_run_grid(waves)), dim3(kBinMcBlock), 0,       \
                     stream, p, r2, same)
  if (out.slots <= 8)
    PCA_BINNED_LAUNCH(8);
  else if (out.slots <= 16)
    PCA_BINNED_LAUNCH(16);
  else if (out.slots <= 24)
    PCA_BINNED_LAUNCH(24);
  else if (out.slots <= 32)
    PCA_BINNED_LAUNCH(32);
  else if (out.slots <= 40)
    PCA_BINNED_LAUNCH_WIDE(40);
  else if (out.slots <= 48)
    PCA_BINNED_LAUNCH_WIDE(48);
  else if (out.slots <= 56)
    PCA_BINNED_LAUNCH_WIDE(56);
  else
    PCA_BINNED_LAUNCH_WIDE(64);
#undef PCA_BINNED_LAUNCH_WIDE
#undef PCA_BINNED_LAUNCH
  return hipGetLastError();
}

} // namespace pca
