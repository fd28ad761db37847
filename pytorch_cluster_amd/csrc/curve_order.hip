// Rows in the order of a space-filling curve, segment by segment: the sort in
// front of the binned searches and of fps over large examples.
//
// Up to four million rows it is a sample sort in four launches, both sides of a
// search in each of them.  The keys (the segment above the 30-bit place on the Hilbert
// curve through its box) are made unique by the row number below them, so that buckets cut between
// sampled keys are of similar size whatever the points are -- half of a LiDAR
// scan's rows share a few cells, and equal places part by their row numbers --
// and the result is that of a stable sort:
//   sample   every segment's samples (eight to a bucket, one per stratum of rows,
//            at a hashed place in it) are ranked by counting; every eighth one is
//            a splitter;
//   count    a workgroup per tile of rows: keys, buckets (a search among the
//            splitters in LDS), the rows' ranks in the tile's share of their
//            bucket, the shares' places in the buckets;
//   scatter  rows to their buckets;
//   buckets  a workgroup per bucket of 768 rows on average, a bitonic network in
//            registers; segments of a single bucket come straight from the points.
//            A bucket of more than 4,096 rows (eight samples to a bucket leave one
//            with a probability of about 1e-10 where buckets have 768 rows, 1 %
//            where they have 2,000) is merged in memory.
// Larger calls and long segments are sorted by the keys' digits of eight bits, the
// lowest first, three launches each: the tiles' rows by digit are counted, the counts
// summed over the tiles, the rows put in their places (DigitPass).
// No workgroup waits for another one and nothing is cleared by memset.
//
// 952,000 LiDAR-like rows in eight segments and 119,000 of them as the other side:
// 13 + 20 + 11 + 24 us (rocPRIM's one-sweep radix sort, which was here before, of
// both sides on two streams: 22 launches, 171 us of kernels and clears); nearest of
// the 952,000 among the 119,000 334 -> 262 us a call, kNN of every fourth row of
// them 696 -> 621.  Bound by latency: hash places and their keys in `sample`, the
// Hilbert steps and the search among splitters in `count`, the network's exchanges
// in `buckets` (LDS instead of registers 65 us; 256 threads of up to 16 rows 25).
//
// The digits' kernels pass over the rows twice per digit, 100 bytes a row; samples cost
// more per row the more of them a segment has (every workgroup looks at all of them) and
// larger buckets take more steps of the network.  Calls, us, radix sort as above /
// samples / digits, nearest of uniform rows to every 16th of them: 1 x 500,000 244 /
// 195 / 203, 1 x 1 M 324 / 308 / 288, 1 x 2 M 499 / 523 / 434, 20 x 100,000 470 / 390 /
// 406, 40 x 100,000 756 / 683 / 674, 200 x 100,000 3,537 / 3,652 / 3,085, 1 x 8 M
// 1,615 / 1,786 / 1,473, 1 x 20 M 4,567 / 5,367 / 4,191; LiDAR-like 1 x 1 M 354 / 343 /
// 331, 40 x 100,000 904 / 837 / 849, 1 x 8 M 2,069 / 2,248 / 1,973.
#include "device_utils.hpp"
#include "launchers.hpp"

#include <algorithm>

namespace pca {

namespace {

constexpr int kSortThreads = 512;   // of a workgroup that counts
constexpr int kSortTile = 2048;     // rows of a tile
constexpr int kBucketThreads = 512; // of a workgroup that sorts a bucket
constexpr int kSortCap = 8 * kBucketThreads; // rows it sorts on the chip
constexpr int kSortPer = 8;         // samples per bucket
constexpr int kSortRanked = 64;     // samples a workgroup ranks
constexpr int kMaxBuckets = 2048;   // of a segment

// The most rows of a side, and of its segments on average, that are sorted by samples
// (calls on both sides of the lines: above).
constexpr int kSampledRows = 4000000, kSampledSegment = 750000;
bool sorted_by_digits(int n, int num_segments) {
  return n > kSampledRows || n / num_segments > kSampledSegment;
}
constexpr int kDigitBits = 8, kDigits = 1 << kDigitBits;
constexpr int kDigitPer = 8;                         // rows of a thread
constexpr int kDigitTile = kDigitPer * kSortThreads; // ... of a workgroup

// Rows of a bucket on average (one segment may have almost all rows) and of the
// buckets whose samples a workgroup ranks, by the number of all rows.
int bucket_rows(int n) {
  return std::max(768, (int)(((int64_t)n + kMaxBuckets - 1) / kMaxBuckets));
}
int chunk_rows(int n) { return bucket_rows(n) * (kSortRanked / kSortPer); }

size_t sort_align(size_t v) { return (v + 255) & ~(size_t)255; }

// One side as the kernels see it.
struct SortSide {
  const float *pts;
  const int64_t *ptr;
  int n;
  CurveSortPlan plan;
  uint64_t *splitters;  // [buckets]
  uint32_t *base;       // [buckets]
  union {
    uint32_t *tile_off; // [tiles][stride]
    uint32_t *digits;   // [kDigits][stride], then [kDigits] totals
  };
  int stride;           // largest number of buckets of a segment; digits: tiles
  uint64_t *pairs;      // [n] (key, row), by bucket
  uint64_t *spare;      // [n]; until the scatter: keys, then places
  uint32_t *keys, *perm;
};
struct SortSides {
  SortSide side[2];
  int blocks; // workgroups of side 0
  int d, num_segments, axis_bits;
  const int *seg_box;
};

struct SortSegment {
  int begin, rows, buckets;
};
__device__ __forceinline__ SortSegment sort_segment(const SortSide &s, int seg) {
  const int64_t lo = s.ptr ? s.ptr[seg] : 0;
  const int64_t hi = s.ptr ? s.ptr[seg + 1] : s.n;
  SortSegment r;
  r.begin = (int)min(max(lo, (int64_t)0), (int64_t)s.n);
  r.rows = (int)max(min(hi, (int64_t)s.n) - r.begin, (int64_t)0);
  const int first = s.plan.bucket_start[seg];
  r.buckets = min(s.plan.bucket_start[seg + 1], s.plan.buckets) - first;
  return r;
}

struct SortBox {
  float lo[3], hi[3];
};
__device__ __forceinline__ SortBox sort_box(const SortSides &p, int seg) {
  SortBox b;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    b.lo[c] = from_ordered_int(p.seg_box[seg * 6 + c]);
    b.hi[c] = from_ordered_int(p.seg_box[seg * 6 + 3 + c]);
  }
  return b;
}
__device__ __forceinline__ uint32_t sort_key(const SortSides &p,
                                             const SortSide &s,
                                             const SortBox &box, int seg,
                                             int row) {
  float v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    v[c] = c < p.d ? s.pts[(size_t)row * p.d + c] : 0.0f;
  return ((uint32_t)seg << (3 * p.axis_bits)) |
         curve_place(v, box.lo, box.hi, p.d, p.axis_bits);
}

// Which side and which of its workgroups.
__device__ __forceinline__ int sort_block(const SortSides &p, int &block) {
  block = (int)blockIdx.x;
  if (block < p.blocks)
    return 0;
  block -= p.blocks;
  return 1;
}

__global__ __launch_bounds__(1024) void curve_sample_kernel(SortSides p) {
  __shared__ __align__(16) uint64_t sample[kMaxBuckets * kSortPer];
  int block;
  const SortSide &s = p.side[sort_block(p, block)];
  const int *chunk_start = s.plan.chunk_start;
  if (block >= chunk_start[p.num_segments])
    return;
  const int seg = find_segment(chunk_start, p.num_segments, block);
  const SortSegment r = sort_segment(s, seg);
  const int buckets = min(r.buckets, kMaxBuckets);
  if (buckets <= 1 || r.rows < buckets * kSortPer)
    return; // (the whole workgroup)
  const int samples = buckets * kSortPer;
  const SortBox box = sort_box(p, seg);
  for (int i = threadIdx.x; i < samples; i += 1024) {
    const int from = (int)((int64_t)i * r.rows / samples);
    const int to = (int)((int64_t)(i + 1) * r.rows / samples);
    const uint32_t h = ((uint32_t)i * 2654435761u) ^ (uint32_t)seg * 40503u;
    const int row = r.begin + from +
                    (int)((uint64_t)(h ^ h >> 15) * (uint32_t)(to - from) >> 32);
    sample[i] = (uint64_t)sort_key(p, s, box, seg, row) << 32 | (uint32_t)row;
  }
  __syncthreads();
  // sixteen threads to a sample, two samples a read
  constexpr int PARTS = 1024 / kSortRanked;
  const int part = (int)threadIdx.x % PARTS;
  const int mine =
      (block - chunk_start[seg]) * kSortRanked + (int)threadIdx.x / PARTS;
  const uint64_t v = sample[min(mine, samples - 1)];
  const ulonglong2 *pairs = reinterpret_cast<const ulonglong2 *>(sample);
  int rank = 0;
#pragma unroll 8
  for (int i = part; i < samples / 2; i += PARTS) {
    const ulonglong2 o = pairs[i];
    rank += (o.x < v ? 1 : 0) + (o.y < v ? 1 : 0);
  }
#pragma unroll
  for (int sh = 1; sh < PARTS; sh <<= 1)
    rank += __shfl_xor(rank, sh);
  if (mine < samples && part == 0 && rank > 0 && rank % kSortPer == 0)
    s.splitters[s.plan.bucket_start[seg] + rank / kSortPer - 1] = v;
}

__global__ __launch_bounds__(kSortThreads) void curve_count_kernel(SortSides p) {
  __shared__ uint64_t splitter[kMaxBuckets];
  __shared__ uint32_t count[kMaxBuckets];
  int block;
  const SortSide &s = p.side[sort_block(p, block)];
  const int *tile_start = s.plan.tile_start;
  if (block >= tile_start[p.num_segments])
    return;
  const int seg = find_segment(tile_start, p.num_segments, block);
  const SortSegment r = sort_segment(s, seg);
  const SortBox box = sort_box(p, seg);
  const int first = (block - tile_start[seg]) * kSortTile;
  const int some = min(kSortTile, r.rows - first);
  const int begin = r.begin + first;
  const int bucket0 = s.plan.bucket_start[seg];
  const int buckets = min(r.buckets, kMaxBuckets);
  int top = 1; // power of two above every bucket number
  while (top < buckets)
    top <<= 1;
  for (int i = threadIdx.x; i < buckets; i += kSortThreads) {
    if (i < buckets - 1)
      splitter[i] = s.splitters[bucket0 + i];
    count[i] = 0u;
  }
  __syncthreads();
  uint32_t *keys = reinterpret_cast<uint32_t *>(s.spare);
  uint32_t *places = keys + s.n;
  // (a thread's rows together: their reads and searches overlap)
  constexpr int PER = kSortTile / kSortThreads;
  uint64_t v[PER];
  int at[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = begin + min(i * kSortThreads + (int)threadIdx.x, some - 1);
    v[i] = (uint64_t)sort_key(p, s, box, seg, row) << 32 | (uint32_t)row;
    at[i] = 0;
  }
  // number of splitters that are not above a row
  for (int step = top >> 1; step > 0; step >>= 1) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int probe = at[i] + step;
      const bool is = probe <= buckets - 1;
      at[i] = splitter[is ? probe - 1 : 0] <= v[i] && is ? probe : at[i];
    }
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = i * kSortThreads + (int)threadIdx.x;
    if (row < some) {
      const uint32_t rank = atomicAdd(&count[at[i]], 1u);
      keys[begin + row] = (uint32_t)(v[i] >> 32);
      places[begin + row] = (uint32_t)at[i] << 16 | rank;
    }
  }
  __syncthreads();
  uint32_t *off = s.tile_off + (size_t)block * s.stride;
  for (int i = threadIdx.x; i < buckets; i += kSortThreads)
    off[i] = count[i] != 0u ? atomicAdd(&s.plan.total[bucket0 + i], count[i])
                            : 0u;
}

__global__ __launch_bounds__(kSortThreads) void
curve_scatter_kernel(SortSides p) {
  constexpr int PER = kMaxBuckets / kSortThreads;
  __shared__ uint32_t start[kMaxBuckets];
  __shared__ uint32_t part[kSortThreads / kWave];
  int block;
  const SortSide &s = p.side[sort_block(p, block)];
  const int *tile_start = s.plan.tile_start;
  if (block >= tile_start[p.num_segments])
    return;
  const int seg = find_segment(tile_start, p.num_segments, block);
  const SortSegment r = sort_segment(s, seg);
  const int buckets = min(r.buckets, kMaxBuckets);
  const int tile = block - tile_start[seg];
  const int first = tile * kSortTile;
  const int some = min(kSortTile, r.rows - first);
  const int begin = r.begin + first;
  const int bucket0 = s.plan.bucket_start[seg];
  // rows of the buckets before each
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  uint32_t v[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = tid * PER + i;
    v[i] = at < buckets ? s.plan.total[bucket0 + at] : 0u;
    sum += v[i];
  }
  uint32_t before = sum;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)before, sh);
    before += lane >= sh ? o : 0u;
  }
  if (lane == kWave - 1)
    part[wave] = before;
  __syncthreads();
  before -= sum;
  for (int w = 0; w < wave; ++w)
    before += part[w];
  const uint32_t *off = s.tile_off + (size_t)block * s.stride;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = tid * PER + i;
    if (at < buckets) {
      start[at] = before + off[at];
      if (tile == 0)
        s.base[bucket0 + at] = before;
    }
    before += v[i];
  }
  __syncthreads();
  const uint32_t *keys = reinterpret_cast<const uint32_t *>(s.spare);
  const uint32_t *places = keys + s.n;
  for (int i = tid; i < some; i += kSortThreads) {
    const uint32_t place = places[begin + i];
    const uint32_t to = start[place >> 16] + (place & 0xffffu);
    if (to < (uint32_t)r.rows)
      s.pairs[r.begin + to] =
          (uint64_t)keys[begin + i] << 32 | (uint32_t)(begin + i);
  }
}

// Value of lane (lane ^ X).
template <int X> __device__ __forceinline__ uint32_t xor_lane(uint32_t v) {
  if (X == 1) // quad_perm 1, 0, 3, 2
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf,
                                                 false);
  if (X == 2) // quad_perm 2, 3, 0, 1
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf,
                                                 false);
  if (X == 8) // row_ror:8
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf,
                                                 false);
  if (X < 32)
    return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, X << 10 | 0x1f);
  return (uint32_t)__shfl_xor((int)v, X);
}

// E pairs per thread of a workgroup of kBucketThreads threads, thread t's from place E t
// on, in ascending order: a bitonic network whose exchanges over fewer than E
// places stay in a thread, over fewer than 64 E in a wave (LDS holds E kBucketThreads).
template <int E, int J>
__device__ __forceinline__ void sort_step(uint64_t (&v)[E], int k,
                                          uint64_t *lds) {
  const int tid = threadIdx.x;
  if constexpr (J < E) {
#pragma unroll
    for (int r = 0; r < E; ++r)
      if ((r & J) == 0) {
        const bool up = ((tid * E + r) & k) == 0;
        const uint64_t a = v[r], b = v[r | J];
        const bool swap = (a > b) == up;
        v[r] = swap ? b : a;
        v[r | J] = swap ? a : b;
      }
  } else if constexpr (J < kWave * E) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const uint32_t lo = xor_lane<J / E>((uint32_t)v[r]);
      const uint32_t hi = xor_lane<J / E>((uint32_t)(v[r] >> 32));
      const uint64_t o = (uint64_t)hi << 32 | lo;
      const bool least = (((tid * E + r) & k) == 0) == ((tid * E & J) == 0);
      v[r] = (o < v[r]) == least ? o : v[r];
    }
  } else {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r)
      lds[r * kBucketThreads + tid] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const uint64_t o = lds[r * kBucketThreads + (tid ^ (J / E))];
      const bool least = (((tid * E + r) & k) == 0) == ((tid * E & J) == 0);
      v[r] = (o < v[r]) == least ? o : v[r];
    }
  }
}
template <int E, int J>
__device__ __forceinline__ void sort_steps(uint64_t (&v)[E], int k,
                                           uint64_t *lds) {
  sort_step<E, J>(v, k, lds);
  if constexpr (J > 1)
    sort_steps<E, J / 2>(v, k, lds);
}
template <int E, int K>
__device__ __forceinline__ void sort_levels(uint64_t (&v)[E], uint64_t *lds) {
  if constexpr (K > 2)
    sort_levels<E, K / 2>(v, lds);
  sort_steps<E, K / 2>(v, K, lds);
}
template <int E, typename Get, typename Put>
__device__ __forceinline__ void sort_bucket(Get get, int count, uint64_t *lds,
                                            Put put) {
  uint64_t v[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int at = r * kBucketThreads + (int)threadIdx.x;
    v[r] = at < count ? get(at) : ~(uint64_t)0;
  }
  sort_levels<E, E * kBucketThreads>(v, lds);
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int at = (int)threadIdx.x * E + r;
    if (at < count)
      put(at, v[r]);
  }
}

__global__ __launch_bounds__(kBucketThreads) void curve_bucket_kernel(SortSides p) {
  __shared__ uint64_t lds[kSortCap];
  int block;
  const SortSide &s = p.side[sort_block(p, block)];
  const int *bucket_start = s.plan.bucket_start;
  if (block >= bucket_start[p.num_segments])
    return;
  const int seg = find_segment(bucket_start, p.num_segments, block);
  const SortSegment r = sort_segment(s, seg);
  auto sorted = [&](int count, auto get, auto put) {
    if (count <= kBucketThreads)
      sort_bucket<1>(get, count, lds, put);
    else if (count <= 2 * kBucketThreads)
      sort_bucket<2>(get, count, lds, put);
    else if (count <= 4 * kBucketThreads)
      sort_bucket<4>(get, count, lds, put);
    else
      sort_bucket<8>(get, count, lds, put);
  };
  const bool whole = r.buckets == 1; // (a segment: from the points themselves)
  const int64_t base = whole ? 0 : s.base[block];
  const int begin = r.begin + (int)min(base, (int64_t)r.rows);
  const int count =
      (int)min(whole ? (int64_t)r.rows : (int64_t)s.plan.total[block],
               (int64_t)(r.begin + r.rows - begin));
  const SortBox box = sort_box(p, seg);
  uint64_t *from = s.pairs + begin, *to = s.spare + begin;
  auto get = [&](int at) -> uint64_t {
    if (!whole)
      return from[at];
    return (uint64_t)sort_key(p, s, box, seg, begin + at) << 32 |
           (uint32_t)(begin + at);
  };
  auto put = [&](int at, uint64_t pair) {
    s.keys[begin + at] = (uint32_t)(pair >> 32);
    s.perm[begin + at] = (uint32_t)pair;
  };
  if (count <= kSortCap)
    return sorted(count, get, put);
  for (int first = 0; first < count; first += kSortCap) {
    sort_bucket<kSortCap / kBucketThreads>(
        [&](int at) { return get(first + at); },
        min(kSortCap, count - first), lds,
        [&](int at, uint64_t pair) { from[first + at] = pair; });
    __syncthreads();
  }
  for (int64_t run = kSortCap; run < count; run *= 2) {
    for (int i = threadIdx.x; i < count; i += kBucketThreads) {
      const uint64_t mine = from[i];
      const int64_t first = i / (2 * run) * (2 * run);
      const int64_t middle = min(first + run, (int64_t)count);
      const int64_t end = min(first + 2 * run, (int64_t)count);
      // its place: the pairs before it in its own run and in the other one
      const bool left = i < middle;
      int64_t lo = left ? middle : first, hi = left ? end : middle;
      const int64_t other = lo;
      while (lo < hi) {
        const int64_t probe = (lo + hi) / 2;
        if (from[probe] < mine)
          lo = probe + 1;
        else
          hi = probe;
      }
      to[first + (i - (left ? first : middle)) + (lo - other)] = mine;
    }
    __syncthreads();
    uint64_t *t = from;
    from = to;
    to = t;
  }
  for (int i = threadIdx.x; i < count; i += kBucketThreads)
    put(i, from[i]);
}

// A pass of the sort by digits, the one from bit `shift` on.  The first one reads the
// points and leaves their keys in `spare`, then the rows go from one buffer of pairs to
// the other; the last pass writes keys and rows.  Rows of equal digits stay in their
// order, so the result is a stable sort's whatever the points are.
struct DigitPass {
  int shift, number;
  bool last;
};
struct DigitRows {
  int begin, rows, first, some; // of all segments; of the tile
};
__device__ __forceinline__ DigitRows digit_rows(const SortSides &p,
                                                const SortSide &s, int tile) {
  const int64_t lo = s.ptr ? s.ptr[0] : 0;
  const int64_t hi = s.ptr ? s.ptr[p.num_segments] : s.n;
  DigitRows r;
  r.begin = (int)min(max(lo, (int64_t)0), (int64_t)s.n);
  r.rows = (int)max(min(hi, (int64_t)s.n) - r.begin, (int64_t)0);
  r.first = tile * kDigitTile;
  r.some = min(kDigitTile, r.rows - r.first);
  return r;
}

// Rows of a tile by digit.  Bound by its reads: 8.5 M rows 16 us a pass (4.3 TB/s), 72
// with the Hilbert steps of the first one.
__global__ __launch_bounds__(kSortThreads) void
digit_count_kernel(SortSides p, DigitPass pass) {
  __shared__ uint32_t count[kDigits];
  int tile;
  const SortSide &s = p.side[sort_block(p, tile)];
  const DigitRows r = digit_rows(p, s, tile);
  if (r.some <= 0)
    return; // (the whole workgroup)
  const int tid = threadIdx.x;
  if (tid < kDigits)
    count[tid] = 0u;
  __syncthreads();
  const int begin = r.begin + r.first;
  uint32_t key[kDigitPer];
  if (pass.number == 0) {
    uint32_t *keys = reinterpret_cast<uint32_t *>(s.spare);
    const int seg0 = find_segment64(s.ptr, p.num_segments, begin);
    const int64_t end0 = s.ptr ? s.ptr[seg0 + 1] : s.n;
    const SortBox box0 = sort_box(p, seg0);
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i) {
      const int row = begin + min(i * kSortThreads + tid, r.some - 1);
      if (row < end0) {
        key[i] = sort_key(p, s, box0, seg0, row);
      } else {
        const int seg = find_segment64(s.ptr, p.num_segments, row);
        key[i] = sort_key(p, s, sort_box(p, seg), seg, row);
      }
      if (i * kSortThreads + tid < r.some)
        keys[row] = key[i];
    }
  } else {
    const uint64_t *from = (pass.number & 1 ? s.pairs : s.spare) + begin;
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i)
      key[i] =
          (uint32_t)(from[min(i * kSortThreads + tid, r.some - 1)] >> 32);
  }
#pragma unroll
  for (int i = 0; i < kDigitPer; ++i)
    if (i * kSortThreads + tid < r.some)
      atomicAdd(&count[key[i] >> pass.shift & (kDigits - 1)], 1u);
  __syncthreads();
  if (tid < kDigits)
    s.digits[(size_t)tid * s.stride + tile] = count[tid];
}

// Exclusive prefix of one value per thread of a workgroup; part: a word per wave.
__device__ __forceinline__ uint32_t digit_prefix(uint32_t v, uint32_t *part,
                                                 uint32_t &total) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t up = v;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)up, sh);
    up += lane >= sh ? o : 0u;
  }
  __syncthreads(); // (part may be in use)
  if (lane == kWave - 1)
    part[wave] = up;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kSortThreads / kWave; ++w) {
    before += w < wave ? part[w] : 0u;
    total += part[w];
  }
  return before + up - v;
}

// A workgroup per digit: rows of the digit in the tiles before each.
__global__ __launch_bounds__(kSortThreads) void digit_scan_kernel(SortSides p) {
  __shared__ uint32_t part[kSortThreads / kWave];
  const int digit = (int)blockIdx.x % kDigits;
  const SortSide &s = p.side[(int)blockIdx.x / kDigits];
  const int rows = digit_rows(p, s, 0).rows;
  const int tiles = (rows + kDigitTile - 1) / kDigitTile;
  uint32_t *column = s.digits + (size_t)digit * s.stride;
  uint32_t before = 0;
  for (int first = 0; first < tiles; first += kSortThreads * kDigitPer) {
    const int at = first + (int)threadIdx.x * kDigitPer;
    uint32_t v[kDigitPer], sum = 0, total;
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i) {
      v[i] = at + i < tiles ? column[at + i] : 0u;
      sum += v[i];
    }
    uint32_t run = before + digit_prefix(sum, part, total);
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i) {
      if (at + i < tiles)
        column[at + i] = run;
      run += v[i];
    }
    before += total;
  }
  if (threadIdx.x == 0)
    s.digits[(size_t)kDigits * s.stride + digit] = before;
}

// A tile's rows by digit, rows of a digit in the order they came in: a wave ranks its
// rows among their like by ballots, sixty-four at a time; in LDS the rows are put
// together digit by digit, so that neighbouring threads write neighbouring places.
// 8.5 M rows 40 us a pass (3.4 TB/s).
__global__ __launch_bounds__(kSortThreads) void
digit_scatter_kernel(SortSides p, DigitPass pass) {
  constexpr int WAVES = kSortThreads / kWave;
  __shared__ uint64_t lds[kDigitTile];
  __shared__ uint32_t place[WAVES][kDigits]; // 40 KB in all: four to a CU
  int tile;
  const SortSide &s = p.side[sort_block(p, tile)];
  const DigitRows r = digit_rows(p, s, tile);
  if (r.some <= 0)
    return; // (the whole workgroup)
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int begin = r.begin + r.first;
  const int mine = wave * (kDigitTile / WAVES) + lane;
  uint64_t v[kDigitPer];
  if (pass.number == 0) {
    const uint32_t *keys = reinterpret_cast<const uint32_t *>(s.spare);
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i) {
      const int row = begin + min(mine + i * kWave, r.some - 1);
      v[i] = (uint64_t)keys[row] << 32 | (uint32_t)row;
    }
  } else {
    const uint64_t *from = (pass.number & 1 ? s.pairs : s.spare) + begin;
#pragma unroll
    for (int i = 0; i < kDigitPer; ++i)
      v[i] = from[min(mine + i * kWave, r.some - 1)];
  }
  // what is before the digit's rows: of smaller digits, in the tiles before
  uint32_t offset = 0, all = 0;
  if (tid < kDigits) {
    offset = s.digits[(size_t)tid * s.stride + tile];
    all = s.digits[(size_t)kDigits * s.stride + tid];
  }
  for (int i = tid; i < WAVES * kDigits; i += kSortThreads)
    (&place[0][0])[i] = 0u;
  __syncthreads();
  const int shift = 32 + pass.shift;
  uint32_t rank[kDigitPer];
#pragma unroll
  for (int i = 0; i < kDigitPer; ++i) {
    const uint32_t digit = (uint32_t)(v[i] >> shift) & (kDigits - 1);
    const bool is = mine + i * kWave < r.some;
    uint64_t same = __ballot(is);
#pragma unroll
    for (int b = 0; b < kDigitBits; ++b) {
      const bool set = (digit >> b & 1u) != 0u;
      const uint64_t lanes = __ballot(set);
      same &= set ? lanes : ~lanes;
    }
    // (the first of them counts for all; a wave's atomics come in order)
    const int leader = same != 0 ? __ffsll((unsigned long long)same) - 1 : lane;
    uint32_t before = 0;
    if (is && lane == leader)
      before = atomicAdd(&place[wave][digit], (uint32_t)__popcll(same));
    before = (uint32_t)__shfl((int)before, leader);
    rank[i] =
        before + (uint32_t)__popcll(same & (((uint64_t)1 << lane) - 1));
  }
  __syncthreads();
  uint32_t *part = reinterpret_cast<uint32_t *>(lds);
  uint32_t count = 0, total;
  if (tid < kDigits)
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      count += place[w][tid];
  offset += digit_prefix(all, part, total);
  const uint32_t local = digit_prefix(count, part, total);
  if (tid < kDigits) {
    uint32_t run = local;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const uint32_t c = place[w][tid];
      place[w][tid] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kDigitPer; ++i) {
    const uint32_t digit = (uint32_t)(v[i] >> shift) & (kDigits - 1);
    if (mine + i * kWave < r.some)
      lds[place[wave][digit] + rank[i]] = v[i];
  }
  __syncthreads();
  if (tid < kDigits)
    place[0][tid] = offset - local; // (modulo 2^32)
  __syncthreads();
  uint64_t *out = (pass.number & 1 ? s.spare : s.pairs) + r.begin;
#pragma unroll
  for (int i = 0; i < kDigitPer; ++i) {
    const int at = i * kSortThreads + tid;
    if (at < r.some) {
      const uint64_t pair = lds[at];
      const uint32_t to =
          place[0][(uint32_t)(pair >> shift) & (kDigits - 1)] + (uint32_t)at;
      if (to < (uint32_t)r.rows) {
        if (pass.last) {
          s.keys[r.begin + to] = (uint32_t)(pair >> 32);
          s.perm[r.begin + to] = (uint32_t)pair;
        } else {
          out[to] = pair;
        }
      }
    }
  }
}

int digit_tiles(int n, int) { return n / kDigitTile + 1; }

// Segments of more than one bucket, at most; their items of so many rows.
int sort_items(int n, int num_segments, int rows) {
  return n / rows + std::min(num_segments, n / bucket_rows(n)) + 1;
}
int sort_tiles(int n, int num_segments) {
  return sort_items(n, num_segments, kSortTile);
}
int sort_chunks(int n, int num_segments) {
  return sort_items(n, num_segments, chunk_rows(n));
}
int sort_buckets(int n, int num_segments) {
  return plan_upper_bound(n, num_segments, bucket_rows(n));
}

struct SortCarve {
  char *cursor;
  template <typename T> T *take(size_t count) {
    T *piece = reinterpret_cast<T *>(cursor);
    cursor += sort_align(sizeof(T) * count);
    return piece;
  }
};
SortSide carve_side(char *&cursor, int n, int num_segments) {
  SortSide s = {};
  SortCarve c{cursor};
  s.n = n;
  const size_t digits = (size_t)kDigits * (digit_tiles(n, num_segments) + 1);
  if (sorted_by_digits(n, num_segments)) {
    s.digits = c.take<uint32_t>(digits);
    s.pairs = c.take<uint64_t>((size_t)n);
    s.spare = c.take<uint64_t>((size_t)n);
    cursor = c.cursor;
    return s;
  }
  const size_t segs = (size_t)num_segments + 1;
  s.stride = (n + bucket_rows(n) - 1) / bucket_rows(n);
  const size_t buckets = (size_t)sort_buckets(n, num_segments);
  s.plan.bucket_rows = bucket_rows(n);
  s.plan.tile_rows = kSortTile;
  s.plan.chunk_rows = chunk_rows(n);
  s.plan.buckets = (int)buckets;
  s.plan.bucket_start = c.take<int>(segs);
  s.plan.tile_start = c.take<int>(segs);
  s.plan.chunk_start = c.take<int>(segs);
  s.plan.total = c.take<uint32_t>(buckets);
  s.base = c.take<uint32_t>(buckets);
  s.splitters = c.take<uint64_t>(buckets);
  // (by digits beside a larger side)
  s.tile_off = c.take<uint32_t>(std::max(
      (size_t)sort_tiles(n, num_segments) * s.stride, digits));
  s.pairs = c.take<uint64_t>((size_t)n);
  s.spare = c.take<uint64_t>((size_t)n);
  cursor = c.cursor;
  return s;
}

} // namespace

size_t curve_sort_bytes(int n, int num_segments) {
  char *cursor = nullptr;
  (void)carve_side(cursor, n, num_segments);
  return (size_t)(cursor - (char *)nullptr);
}

CurveSortPlan curve_sort_plan(void *scratch, int n, int num_segments) {
  char *cursor = static_cast<char *>(scratch);
  return carve_side(cursor, n, num_segments).plan;
}

hipError_t launch_curve_sort(const CurveSortSide *sides, int num_sides, int d,
                             int num_segments, int axis_bits,
                             const int *seg_box, hipStream_t stream) {
  SortSides p = {};
  for (int i = 0; i < num_sides; ++i) {
    char *cursor = static_cast<char *>(sides[i].scratch);
    p.side[i] = carve_side(cursor, sides[i].n, num_segments);
    p.side[i].pts = sides[i].pts;
    p.side[i].ptr = sides[i].ptr;
    p.side[i].keys = sides[i].keys;
    p.side[i].perm = sides[i].perm;
  }
  p.d = d;
  p.num_segments = num_segments;
  p.axis_bits = axis_bits;
  p.seg_box = seg_box;
  auto grid = [&](int (*bound)(int, int)) {
    int all = 0;
    for (int i = 0; i < num_sides; ++i) {
      p.blocks = i == 0 ? bound(p.side[0].n, num_segments) : p.blocks;
      all += bound(p.side[i].n, num_segments);
    }
    return dim3(all);
  };
  bool by_digits = false; // (both sides, if one of them is better off)
  for (int i = 0; i < num_sides; ++i)
    by_digits = by_digits || sorted_by_digits(sides[i].n, num_segments);
  if (by_digits) {
    for (int i = 0; i < num_sides; ++i)
      p.side[i].stride = digit_tiles(p.side[i].n, num_segments);
    int bits = 3 * axis_bits; // of the keys
    while (((int64_t)1 << (bits - 3 * axis_bits)) < num_segments)
      ++bits;
    const dim3 tiles = grid(digit_tiles);
    for (DigitPass pass = {0, 0, false}; !pass.last; ++pass.number) {
      pass.shift = pass.number * kDigitBits;
      pass.last = pass.shift + kDigitBits >= bits;
      hipLaunchKernelGGL(digit_count_kernel, tiles, dim3(kSortThreads), 0,
                         stream, p, pass);
      hipLaunchKernelGGL(digit_scan_kernel, dim3(num_sides * kDigits),
                         dim3(kSortThreads), 0, stream, p);
      hipLaunchKernelGGL(digit_scatter_kernel, tiles, dim3(kSortThreads), 0,
                         stream, p, pass);
    }
    return hipGetLastError();
  }
  dim3 blocks = grid(sort_chunks);
  hipLaunchKernelGGL(curve_sample_kernel, blocks, dim3(1024), 0, stream, p);
  blocks = grid(sort_tiles);
  hipLaunchKernelGGL(curve_count_kernel, blocks, dim3(kSortThreads), 0, stream,
                     p);
  hipLaunchKernelGGL(curve_scatter_kernel, blocks, dim3(kSortThreads), 0,
                     stream, p);
  blocks = grid(sort_buckets);
  hipLaunchKernelGGL(curve_bucket_kernel, blocks, dim3(kBucketThreads), 0,
                     stream, p);
  return hipGetLastError();
}

} // namespace pca
