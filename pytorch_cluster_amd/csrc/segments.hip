// Segment planning and output compaction kernels.
//
// Replaces, on the device and without host synchronisation:
//   * get_example_idx (csrc/cuda/utils.cuh:11-19 in the reference): instead of
//     every thread scanning ptr linearly, one tiny kernel turns ptr_y into a
//     table "first work item of each segment" that workgroups binary-search;
//   * the reference's post-kernel epilogue `mask = col != -1`,
//     2x masked_select, stack (csrc/cuda/knn_cuda.cu:133-134,
//     csrc/cuda/radius_cuda.cu:94-95): per-query counts -> exclusive scan ->
//     scatter into a contiguous [2, E] matrix, E left in device memory;
//   * on request the epilogue of the graph entry points as well
//     (torch_cluster/knn.py:135-144, torch_cluster/radius.py:143-148): pairs
//     of a row with itself are left out and the x row is written first, in
//     the same pass.
#include "device_utils.hpp"
#include "launchers.hpp"

#include <algorithm>

namespace pca {

namespace {

// Single workgroup: exclusive scan of ceil(m_b / per_item) over segments;
// before that, when the caller passed sorted example ids instead of pointers,
// the pointers of both sides (ptr_y is then src.ptr_y).
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(
    const int64_t *__restrict__ ptr_y, int m, int num_segments, int per_item,
    int *__restrict__ work_start, SegmentSource src) {
  __shared__ int partial[kPlanThreads];
  if (src.ids_x != nullptr) {
    pointers_from_ids(src, num_segments);
    __syncthreads();
  }
  plan_segments(ptr_y, m, num_segments, per_item, work_start, partial);
}

// One search per wave, whatever the number of examples: the searches are
// chains of dependent reads, so they take as long as one of them as long as
// each has a wave of its own (1,000 examples: 3 us; by the 16 waves of one
// workgroup, 125 searches each, 150 us).
__global__ __launch_bounds__(kBlock) void segment_pointers_kernel(
    SegmentSource src, int num_segments) {
  pointers_from_ids(src, num_segments, (int)blockIdx.x, (int)gridDim.x);
}

// What `nearest` needs to know of its example ids before it may answer: the
// pointers of both sides, whether a vector is not sorted (report[0] for x,
// [1] for y), whether an example has rows on one side only ([2]), and the
// number of examples the ids speak of ([3]).  report: four numbers set to 0
// by the host, in memory it reads.  A wave per example, and all threads look
// for a decrease; pointers of unsorted ids ascend too (a larger bound never
// takes a search further to the left).
__global__ __launch_bounds__(kBlock) void two_sides_kernel(
    const int64_t *__restrict__ ids_x, int n,
    const int64_t *__restrict__ ids_y, int m, int num_segments,
    int64_t *__restrict__ ptr_x, int64_t *__restrict__ ptr_y,
    int64_t *__restrict__ report) {
  const int thread = blockIdx.x * kBlock + threadIdx.x;
  const int threads = gridDim.x * kBlock;
  const int lane = threadIdx.x & (kWave - 1);
  if (thread == 0)
    report[3] = max(max(ids_x[n - 1], ids_y[m - 1]), (int64_t)-1) + 1;
  for (int b = thread / kWave; b <= num_segments; b += threads / kWave) {
    const int64_t ends[2] = {(int64_t)b, (int64_t)b + 1};
    int in_x[2], in_y[2];
    wave_rows_below(ids_x, n, ends, lane, in_x);
    wave_rows_below(ids_y, m, ends, lane, in_y);
    if (lane == 0) {
      // (searching rows beyond the last example: the last one's, as above)
      ptr_x[b] = b == num_segments ? n : in_x[0];
      ptr_y[b] = in_y[0];
      if (b < num_segments && (in_x[1] > in_x[0]) != (in_y[1] > in_y[0]))
        report[2] = 1;
    }
  }
  bool falls = false;
  for (int64_t i = thread; i < n - 1; i += threads)
    falls = falls || ids_x[i + 1] < ids_x[i];
  if (falls)
    report[0] = 1;
  falls = false;
  for (int64_t i = thread; i < m - 1; i += threads)
    falls = falls || ids_y[i + 1] < ids_y[i];
  if (falls)
    report[1] = 1;
}

// The samples of `fps`, ceil(rows * ratio) of every example in fp32 as the
// host wrapper of the reference forms them (csrc/cuda/fps_cuda.cu:68-109):
// out_ptr, and in report[0] their number, [1] the largest example, [2] the
// examples the ids speak of.  One workgroup; ids NULL: one example of n rows,
// whose pointers are written here too.
__global__ __launch_bounds__(kPlanThreads) void fps_sizes_kernel(
    const int64_t *__restrict__ ids, int n, int num_segments, float ratio,
    int64_t *__restrict__ ptr, int64_t *__restrict__ out_ptr,
    int64_t *__restrict__ report) {
  __shared__ int64_t partial[kPlanThreads];
  __shared__ int longest;
  const int tid = threadIdx.x;
  const int per_thread = (num_segments + kPlanThreads - 1) / kPlanThreads;
  const int b0 = min(tid * per_thread, num_segments);
  const int b1 = min(b0 + per_thread, num_segments);
  auto rows_of = [&](int b) -> int64_t {
    return ids != nullptr ? ptr[b + 1] - ptr[b] : (int64_t)n;
  };
  auto samples_of = [&](int64_t rows) {
    return (int64_t)__builtin_ceilf((float)rows * ratio);
  };
  if (tid == 0)
    longest = 0;
  int64_t sum = 0;
  int most = 0;
  for (int b = b0; b < b1; ++b) {
    const int64_t rows = rows_of(b);
    sum += samples_of(rows);
    most = max(most, (int)rows);
  }
  partial[tid] = sum;
  __syncthreads();
  atomicMax(&longest, most);
  for (int off = 1; off < kPlanThreads; off <<= 1) {
    const int64_t v = tid >= off ? partial[tid - off] : 0;
    __syncthreads();
    partial[tid] += v;
    __syncthreads();
  }
  int64_t run = partial[tid] - sum;
  for (int b = b0; b < b1; ++b) {
    out_ptr[b] = run;
    run += samples_of(rows_of(b));
  }
  if (tid == kPlanThreads - 1) {
    out_ptr[num_segments] = partial[tid];
    if (ids == nullptr) {
      ptr[0] = 0;
      ptr[1] = n;
    }
    if (report != nullptr) {
      report[0] = partial[tid];
      report[1] = longest;
      report[2] = ids != nullptr ? max(ids[n - 1], (int64_t)-1) + 1 : 1;
    }
  }
}

// ---- compaction -----------------------------------------------------------

constexpr int kCompactQueries = kBlock; // queries per workgroup

// Block-wide exclusive scan of one int per thread; returns the exclusive
// prefix, *total receives the block sum.
__device__ __forceinline__ int block_exclusive_scan(int v, int *lds,
                                                    int *total) {
  const int tid = threadIdx.x;
  lds[tid] = v;
  __syncthreads();
  for (int off = 1; off < kBlock; off <<= 1) {
    int t = tid >= off ? lds[tid - off] : 0;
    __syncthreads();
    lds[tid] += t;
    __syncthreads();
  }
  *total = lds[kBlock - 1];
  return lds[tid] - v;
}

__global__ __launch_bounds__(kBlock) void block_sum_kernel(
    const int *__restrict__ count, int m, int64_t *__restrict__ block_sums) {
  __shared__ int lds[kBlock];
  const int q = blockIdx.x * kCompactQueries + threadIdx.x;
  int total;
  block_exclusive_scan(q < m ? count[q] : 0, lds, &total);
  if (threadIdx.x == 0)
    block_sums[blockIdx.x] = total;
}

// Single workgroup: in-place exclusive scan of the block sums, total -> E.
__global__ __launch_bounds__(kPlanThreads) void scan_block_sums_kernel(
    int64_t *__restrict__ block_sums, int num_blocks,
    int64_t *__restrict__ num_edges) {
  __shared__ int64_t partial[kPlanThreads];
  const int tid = threadIdx.x;
  const int per_thread = (num_blocks + kPlanThreads - 1) / kPlanThreads;
  const int i0 = min(tid * per_thread, num_blocks);
  const int i1 = min(i0 + per_thread, num_blocks);
  int64_t sum = 0;
  for (int i = i0; i < i1; ++i)
    sum += block_sums[i];
  partial[tid] = sum;
  __syncthreads();
  for (int off = 1; off < kPlanThreads; off <<= 1) {
    int64_t v = tid >= off ? partial[tid - off] : 0;
    __syncthreads();
    partial[tid] += v;
    __syncthreads();
  }
  int64_t run = partial[tid] - sum;
  for (int i = i0; i < i1; ++i) {
    int64_t v = block_sums[i];
    block_sums[i] = run;
    run += v;
  }
  // (the total also behind the offsets: the scatter reads it from there, so
  // that num_edges is only ever written -- it may be host memory)
  if (tid == kPlanThreads - 1) {
    *num_edges = partial[tid];
    block_sums[num_blocks] = partial[tid];
  }
}

// e / slots without a division, for the entries e < kCompactQueries * slots
// of a block: with magic = ceil(2^32 / slots) the product's high word is the
// quotient as long as e (slots - 1) < 2^32, which holds up to 4,000 slots; 0
// (one slot, or more than that) stands for "divide".
inline uint32_t slots_magic(int slots) {
  if (slots < 2 || slots > 4000)
    return 0;
  return (uint32_t)((((uint64_t)1 << 32) + (uint64_t)slots - 1) /
                    (uint64_t)slots);
}
__device__ __forceinline__ int quotient_by_slots(int e, int slots,
                                                 uint32_t magic) {
  return magic != 0 ? (int)__umulhi((uint32_t)e, magic) : e / slots;
}

// Both kernels below walk the slot rows of a block of queries as ONE flat
// range (element e = slot e % slots of query e / slots): reads are contiguous
// and independent of each other, so many are in flight per thread.
//
// find_self_kernel: position of the slot that holds the query's own row
// number (at most one: the rows of a query are distinct), or -1, and the
// number of slots without it.
__global__ __launch_bounds__(kBlock) void find_self_kernel(
    const int *__restrict__ idx, const int *__restrict__ count, int m,
    int slots, uint32_t magic, int *__restrict__ self_pos,
    int *__restrict__ kept) {
  __shared__ int s_self[kCompactQueries];
  __shared__ int s_count[kCompactQueries];
  const int tid = threadIdx.x;
  const int q0 = blockIdx.x * kCompactQueries;
  const int nq = min(kCompactQueries, m - q0);
  s_self[tid] = -1;
  s_count[tid] = tid < nq ? count[q0 + tid] : 0;
  __syncthreads();
  const int *rows = idx + (size_t)q0 * slots;
  const int total = nq * slots;
#pragma unroll 4
  for (int e = tid; e < total; e += kBlock) {
    const int ql = quotient_by_slots(e, slots, magic);
    const int sl = e - ql * slots;
    const int v = rows[e];
    if (sl < s_count[ql] && v == q0 + ql)
      s_self[ql] = sl;
  }
  __syncthreads();
  if (tid < nq) {
    self_pos[q0 + tid] = s_self[tid];
    kept[q0 + tid] = s_count[tid] - (s_self[tid] >= 0 ? 1 : 0);
  }
}

// The two kernels of the short path (up to kInlineScanBlocks blocks of
// queries): count_block_kernel = find_self_kernel + block_sum_kernel in one
// pass (self_pos == nullptr: nothing is left out, only the sums), and a
// scatter that adds up the sums of the blocks before it on its own.
constexpr int kInlineScanBlocks = 2048;

__global__ __launch_bounds__(kBlock) void count_block_kernel(
    const int *__restrict__ idx, const int *__restrict__ count, int m,
    int slots, uint32_t magic, int *__restrict__ self_pos,
    int *__restrict__ kept, int64_t *__restrict__ block_sums) {
  __shared__ int s_self[kCompactQueries];
  __shared__ int s_count[kCompactQueries];
  __shared__ int lds[kBlock];
  const int tid = threadIdx.x;
  const int q0 = blockIdx.x * kCompactQueries;
  const int nq = min(kCompactQueries, m - q0);
  int c = tid < nq ? count[q0 + tid] : 0;
  if (self_pos != nullptr) {
    s_self[tid] = -1;
    s_count[tid] = c;
    __syncthreads();
    const int *rows = idx + (size_t)q0 * slots;
    const int total = nq * slots;
#pragma unroll 4
    for (int e = tid; e < total; e += kBlock) {
      const int ql = quotient_by_slots(e, slots, magic);
      const int sl = e - ql * slots;
      const int v = rows[e];
      if (sl < s_count[ql] && v == q0 + ql)
        s_self[ql] = sl;
    }
    __syncthreads();
    if (tid < nq) {
      c -= s_self[tid] >= 0 ? 1 : 0;
      self_pos[q0 + tid] = s_self[tid];
      kept[q0 + tid] = c;
    }
  }
  int total;
  block_exclusive_scan(c, lds, &total);
  if (tid == 0)
    block_sums[blockIdx.x] = total;
}

// Inclusive prefix sum over the lanes of a wave.
__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int t = __shfl_up(v, off);
    v += lane >= off ? t : 0;
  }
  return v;
}

// count: slots to write per query (without the self slot when self_pos is
// given).  x_first: the x row goes to the first half of `edges`.
// inline_scan 1: block_offsets holds the blocks' SUMS; this block adds up the
// ones before it and all of them (block 0 also stores the total).  2: it adds
// up the counts themselves.
//
// Bound by the latency of its reads -- counts and sums, then slots -- as long
// as the device is not full: 1 << parts_log2 workgroups share a block of
// queries (every one scans the block's counts and writes its part of the
// rows), and the scans stay inside the waves, with one barrier for everything.
__global__ __launch_bounds__(kBlock) void scatter_kernel(
    const int *__restrict__ idx, const float *__restrict__ dist,
    const int *__restrict__ count, const int *__restrict__ self_pos, int m,
    int slots, uint32_t magic, int x_first, int parts_log2, int num_blocks,
    const int64_t *__restrict__ block_offsets,
    int64_t *__restrict__ num_edges, int64_t *__restrict__ edges,
    float *__restrict__ dist_out, int inline_scan) {
  constexpr int W = kBlock / kWave;
  __shared__ int64_t s_before[W], s_all[W];
  __shared__ int s_sum[W];
  __shared__ int s_count[kCompactQueries];
  __shared__ int s_offset[kCompactQueries]; // within the wave's queries
  __shared__ int s_self[kCompactQueries];
  static_assert(kBlock == kCompactQueries, "one thread per query");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int block = blockIdx.x >> parts_log2;
  const int part = blockIdx.x - (block << parts_log2);
  const int q0 = block * kCompactQueries;
  const int q = q0 + tid;
  const int c = q < m ? count[q] : 0;
  const int self = self_pos && q < m ? self_pos[q] : -1;
  int64_t before = 0, all = 0;
  if (inline_scan == 1)
    for (int b = tid; b < num_blocks; b += kBlock) {
      const int64_t v = block_offsets[b];
      all += v;
      before += b < block ? v : 0;
    }
  else if (inline_scan == 2)
#pragma unroll 4
    for (int i = tid; i < m; i += kBlock) {
      const int v = count[i];
      all += v;
      before += i < q0 ? v : 0;
    }
  const int inclusive = wave_inclusive_scan(c, lane);
  s_count[tid] = c;
  s_offset[tid] = inclusive - c;
  // (a position no slot has when nothing is left out)
  s_self[tid] = self >= 0 ? self : slots;
  if (lane == kWave - 1)
    s_sum[wave] = inclusive;
  if (inline_scan) {
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      before += __shfl_xor(before, sh);
      all += __shfl_xor(all, sh);
    }
    if (lane == 0) {
      s_before[wave] = before;
      s_all[wave] = all;
    }
  }
  __syncthreads();
  int wave_base[W];
  int64_t E = 0, base = 0;
  {
    int run = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      wave_base[w] = run;
      run += s_sum[w];
    }
  }
  if (inline_scan) {
#pragma unroll
    for (int w = 0; w < W; ++w) {
      E += s_all[w];
      base += s_before[w];
    }
    if (blockIdx.x == 0 && tid == 0)
      *num_edges = E;
  } else {
    E = block_offsets[num_blocks];
    base = block_offsets[block];
  }

  const int per_part = kCompactQueries >> parts_log2;
  const int first_q = part * per_part;
  const int nq = min(per_part, m - q0 - first_q);
  int64_t *first = x_first ? edges + E : edges;  // receives the query rows
  int64_t *second = x_first ? edges : edges + E; // receives the x rows
  const size_t row0 = (size_t)(q0 + first_q) * slots;
  const int *rows = idx + row0;
  const float *row_dist = dist ? dist + row0 : nullptr;
  const int span = nq * slots; // (nothing to do for nq <= 0)
#pragma unroll 4
  for (int e = tid; e < span; e += kBlock) {
    const int el = quotient_by_slots(e, slots, magic);
    const int ql = first_q + el;
    const int sl = e - el * slots;
    const int skip = s_self[ql];
    // slot sl goes to position sl, or sl - 1 behind the left-out slot
    const int pos = sl - (sl > skip ? 1 : 0);
    if (sl != skip && pos < s_count[ql]) {
      int in_block = s_offset[ql] + pos;
#pragma unroll
      for (int w = 1; w < W; ++w)
        in_block += ql / kWave == w ? wave_base[w] : 0;
      const int64_t o = base + in_block;
      first[o] = q0 + ql;
      second[o] = rows[e];
      if (dist_out)
        dist_out[o] = row_dist[e];
    }
  }
}

// workgroups of 4 waves that fill 256 CUs
constexpr int kScatterGroups = 2048;

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

} // namespace

hipError_t launch_plan(const int64_t *ptr_y, int m, int num_segments,
                       int per_item, int *work_start, hipStream_t stream,
                       const SegmentSource *src) {
  hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(kPlanThreads), 0, stream, ptr_y,
                     m, num_segments, per_item, work_start,
                     src ? *src : SegmentSource{});
  return hipGetLastError();
}

hipError_t launch_segment_pointers(const SegmentSource &src, int num_segments,
                                   hipStream_t stream) {
  const int waves = kBlock / kWave;
  const int searches = 2 * (num_segments + 1);
  const int blocks = std::min((searches + waves - 1) / waves, 4096);
  hipLaunchKernelGGL(segment_pointers_kernel, dim3(blocks), dim3(kBlock), 0,
                     stream, src, num_segments);
  return hipGetLastError();
}

hipError_t launch_two_sides(const SegmentSource &src, int num_segments,
                            int64_t *report, hipStream_t stream) {
  // (a wave per example, some rows per thread)
  const int waves = kBlock / kWave;
  const int by_rows = (int)std::min<int64_t>(
      ((int64_t)src.n + src.m) / (kBlock * 4), 2048);
  const int blocks =
      std::max(std::min((num_segments + waves) / waves, 4096), by_rows);
  hipLaunchKernelGGL(two_sides_kernel, dim3(blocks), dim3(kBlock), 0, stream,
                     src.ids_x, src.n, src.ids_y, src.m, num_segments,
                     src.ptr_x, src.ptr_y, report);
  return hipGetLastError();
}

hipError_t launch_fps_sizes(const int64_t *ids, int n, int num_segments,
                            float ratio, int64_t *ptr, int64_t *out_ptr,
                            int64_t *report, hipStream_t stream) {
  hipLaunchKernelGGL(fps_sizes_kernel, dim3(1), dim3(kPlanThreads), 0, stream,
                     ids, n, num_segments, ratio, ptr, out_ptr, report);
  return hipGetLastError();
}

size_t compact_workspace_bytes(int m) {
  const int blocks = (m + kCompactQueries - 1) / kCompactQueries;
  // block sums, then the two per-query arrays of find_self_kernel
  return align256(sizeof(int64_t) * (size_t)(blocks + 1)) +
         2 * align256(sizeof(int) * (size_t)m);
}

void compact_hints(DenseResult &dense, int m, void *workspace, bool drop_self) {
  static_assert(kCompactBlockQueries == kCompactQueries, "one block, one sum");
  const int blocks = (m + kCompactQueries - 1) / kCompactQueries;
  if (blocks > kInlineScanBlocks)
    return;
  char *ws = static_cast<char *>(workspace);
  dense.edge_sums = reinterpret_cast<unsigned long long *>(ws);
  ws += align256(sizeof(int64_t) * (size_t)(blocks + 1));
  if (drop_self) {
    dense.self_pos = reinterpret_cast<int *>(ws);
    dense.kept = reinterpret_cast<int *>(ws + align256(sizeof(int) * (size_t)m));
  }
}

void compact_counted(DenseResult &dense, int m, void *workspace,
                     bool drop_self) {
  if (m > kCompactCountedQueries)
    return;
  dense.counted = true;
  if (drop_self) {
    dense.self_pos = static_cast<int *>(workspace);
    dense.kept = reinterpret_cast<int *>(static_cast<char *>(workspace) +
                                         align256(sizeof(int) * (size_t)m));
  }
}

hipError_t launch_compact(const DenseResult &dense, int m, int64_t *edges,
                          int64_t *num_edges, float *dist_out, void *workspace,
                          hipStream_t stream, bool drop_self, bool x_first) {
  const int blocks = (m + kCompactQueries - 1) / kCompactQueries;
  char *ws = static_cast<char *>(workspace);
  int64_t *block_sums = reinterpret_cast<int64_t *>(ws);
  ws += align256(sizeof(int64_t) * (size_t)(blocks + 1));
  int *self_pos = reinterpret_cast<int *>(ws);
  int *kept = reinterpret_cast<int *>(ws + align256(sizeof(int) * (size_t)m));
  const int *count = dense.count;
  const uint32_t magic = slots_magic(dense.slots);
  // as many workgroups as bring the device to eight waves per SIMD, at least
  // 32 queries each
  int parts_log2 = 0;
  while (parts_log2 < 3 && (blocks << (parts_log2 + 1)) <= kScatterGroups)
    ++parts_log2;
  const dim3 scatter_grid((unsigned)blocks << parts_log2);
  if (dense.edge_sums != nullptr && blocks <= kInlineScanBlocks &&
      (!drop_self || dense.self_pos != nullptr)) {
    // the search left the block sums (and the self slots) behind
    hipLaunchKernelGGL(scatter_kernel, scatter_grid, dim3(kBlock), 0, stream,
                       dense.idx, dense.dist, drop_self ? dense.kept : count,
                       drop_self ? dense.self_pos : (const int *)nullptr, m,
                       dense.slots, magic, x_first ? 1 : 0, parts_log2, blocks,
                       reinterpret_cast<const int64_t *>(dense.edge_sums),
                       num_edges, edges, dist_out, 1);
    return hipGetLastError();
  }
  if (dense.counted) {
    hipLaunchKernelGGL(scatter_kernel, scatter_grid, dim3(kBlock), 0, stream,
                       dense.idx, dense.dist, drop_self ? dense.kept : count,
                       drop_self ? dense.self_pos : (const int *)nullptr, m,
                       dense.slots, magic, x_first ? 1 : 0, parts_log2, blocks,
                       (const int64_t *)nullptr, num_edges, edges, dist_out,
                       2);
    return hipGetLastError();
  }
  if (blocks <= kInlineScanBlocks) {
    hipLaunchKernelGGL(count_block_kernel, dim3(blocks), dim3(kBlock), 0,
                       stream, dense.idx, dense.count, m, dense.slots, magic,
                       drop_self ? self_pos : (int *)nullptr, kept,
                       block_sums);
    hipLaunchKernelGGL(scatter_kernel, scatter_grid, dim3(kBlock), 0, stream,
                       dense.idx, dense.dist, drop_self ? kept : count,
                       drop_self ? self_pos : (const int *)nullptr, m,
                       dense.slots, magic, x_first ? 1 : 0, parts_log2, blocks, block_sums,
                       num_edges, edges, dist_out, 1);
    return hipGetLastError();
  }
  if (drop_self) {
    hipLaunchKernelGGL(find_self_kernel, dim3(blocks), dim3(kBlock), 0, stream,
                       dense.idx, dense.count, m, dense.slots, magic, self_pos,
                       kept);
    count = kept;
  }
  hipLaunchKernelGGL(block_sum_kernel, dim3(blocks), dim3(kBlock), 0, stream,
                     count, m, block_sums);
  hipLaunchKernelGGL(scan_block_sums_kernel, dim3(1), dim3(kPlanThreads), 0,
                     stream, block_sums, blocks, num_edges);
  hipLaunchKernelGGL(scatter_kernel, scatter_grid, dim3(kBlock), 0, stream,
                     dense.idx, dense.dist, count,
                     drop_self ? self_pos : (const int *)nullptr, m,
                     dense.slots, magic, x_first ? 1 : 0, parts_log2, blocks, block_sums, num_edges,
                     edges, dist_out, 0);
  return hipGetLastError();
}

} // namespace pca
