// Fixed-radius neighbour search for low-dimensional fp32 points (d <= 8) with
// the candidate filter on the gfx950 matrix cores.
//
// Computes what radius_kernel of the reference computes
// (csrc/cuda/radius_cuda.cu:9-42: one thread per query scans its segment of x
// in ascending row order, keeps the first max_num_neighbors rows with
// dist < r^2, stops as soon as it has them) -- same rows, same order.
//
// The machinery is that of knn_lowd_mc_impl.hpp with a threshold that never
// moves: t - cut = w - 2 x.y - cut, cut = r^2 (1 + eps) - fl(|y|^2) (1 - eps),
// comes out of one v_mfma_f32_32x32x16_bf16 per 32 rows x 32 queries
// (split-bf16 operands, -cut in the two spare accumulation slots), the sign
// bits of a lane's 16 results are gathered with funnel shifts, and a pair of
// lanes with a row that passed parks (step, mask) in its LDS queue.  A candidate with an
// exact distance below r^2 always has its sign bit set (error budget in
// knn_lowd_mc_impl.hpp); whether a row with the bit set IS a neighbour is
// decided by the exact distance (direct differences, one FMA per component in
// ascending order) taken from the fp32 coordinates in the LDS tile.
//
// Lanes l and l + 32 share a query and see interleaved groups of four rows.
// When a queue fills up or the tile ends, the lower lane of each pair walks
// the parked rows in ascending order and appends the
// neighbours to the query's slot row until it holds max_num_neighbors.  A
// query that is full stops parking; a wave whose queries are all full skips
// the matrix-core work, a workgroup whose waves are all done leaves the scan.
//
// A few queries far from everything would keep the whole workgroup scanning
// (clustered points: after an eighth of the rows 85 % of the queries are
// full, but hardly a wave is).  So from the first tile on at whose start at
// most kRadiusFew queries are open, these are dealt to the four waves, and a
// wave goes through the rows on its own, straight from memory, 256 at a time,
// once for all its open queries: hits are found and numbered by ballots, in
// row order as they are.  No barriers, no tiles, and a wave whose queries are
// full leaves.
//
// 8 clouds of 16,384 clustered points, r = 0.05, 32 neighbours: kernel 228 ->
// 132 us (the walk of parked rows without nested branches 20 us of that; 64
// open queries instead of 32: 4 us more); two thirds of what is left are the
// first three tiles, in which every query meets its neighbours one by one.
//
// A workgroup owns 128 queries of one segment and scans the whole segment
// (rows must be reported in order, so the segment is not sliced).
#pragma once

#include "knn_lowd_mc_impl.hpp"

namespace pca {

constexpr int kRadiusFew = 32; // open queries a workgroup deals to its waves

struct RadiusMcParams {
  const float *x;
  const float *y;
  const int64_t *ptr_x;
  const int64_t *ptr_y;
  const uint4 *x_split; // packed rows of x (mc_pack_rows_kernel)
  int n, m, d_in, num_segments;
  float r2;
  int slots;
  int ignore_same_index;
  const int *work_start; // [num_segments + 1] first 128-query tile per segment
  int *out_idx;          // [m, slots]
  int *out_count;        // [m]
  // for the compaction (DenseResult::edge_sums; NULL: not asked for):
  // neighbours found per kCompactBlockQueries queries
  unsigned long long *edge_sums = nullptr;
};

template <int DIM>
__global__ __launch_bounds__(kBlock) void radius_mc_kernel(RadiusMcParams p) {
  constexpr int NI = McShape<DIM>::NI;
  constexpr int XF = McShape<DIM>::XF;
  constexpr int REC = McShape<DIM>::REC;
  constexpr int TX = McShape<DIM>::TX;
  constexpr int TQ = kMcQueries;
  constexpr int QCAP = kMcQueueCap;
  constexpr int PT = TX / kBlock; // rows staged per thread

  // (every 16-byte unit of a row in a plane of its own, as in
  // knn_lowd_mc_impl.hpp: conflict-free reads)
  __shared__ __attribute__((aligned(16))) uint4 rows_lds[REC][TX];
  // parked steps of the pairs of lanes: in the lower lane's column the mask of
  // the 32 rows, in the upper lane's the step
  // (also carries, between the two barriers at the top of a tile, the four
  // waves' numbers of open queries, and the last few open queries: one more
  // variable would take the workgroup past 40,960 bytes, the most that lets
  // four of them share a CU)
  __shared__ uint32_t queue[QCAP][kBlock];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int half = lane >> 5;
  const int col = lane & 31;

  const int total_tiles = p.work_start[p.num_segments];
  const int tile = blockIdx.x;
  if (tile >= total_tiles)
    return;
  const int seg = find_segment(p.work_start, p.num_segments, tile);
  const int x_begin = p.ptr_x ? (int)p.ptr_x[seg] : 0;
  const int x_end = p.ptr_x ? (int)p.ptr_x[seg + 1] : p.n;
  const int y_begin = p.ptr_y ? (int)p.ptr_y[seg] : 0;
  const int y_end = p.ptr_y ? (int)p.ptr_y[seg + 1] : p.m;
  const int q = y_begin + (tile - p.work_start[seg]) * TQ + wave * 32 + col;
  const bool valid = q < y_end;
  const int d_in = p.d_in;
  const int slots = p.slots;
  const float r2 = p.r2;
  const int c_count = x_end - x_begin;
  const int num_tiles = (c_count + TX - 1) / TX;

  // ---- per-lane query state ---------------------------------------------
  float yq[DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c)
    yq[c] = (valid && c < d_in) ? p.y[(size_t)q * d_in + c] : 0.0f;
  float ysq = yq[0] * yq[0];
#pragma unroll
  for (int c = 1; c < DIM; ++c)
    ysq = __builtin_fmaf(yq[c], yq[c], ysq);
  const bool y_moderate = ysq <= kFilterNormLimit;
  // B operands as in knn_lowd_mc_kernel: the hi (lanes 0-31) or lo (lanes
  // 32-63) parts of (-2 y, 1, 0 ...), the upper lanes with the parts of -cut'
  // where the lo part of the 1 would be
  constexpr int WI = DIM / 4;
  constexpr int WE = DIM % 4;
  mc_bf16x8_t yb[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    uint32_t part[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = 4 * i + e;
      float v = 0.0f;
      if (c < DIM)
        v = (valid && y_moderate) ? -2.0f * yq[c] : 0.0f;
      else if (c == DIM)
        v = valid ? 1.0f : 0.0f;
      uint32_t hi, lo;
      mc_split(v, hi, lo);
      part[e] = half ? lo : hi;
    }
    uint32_t w0 = part[0] | (part[1] << 16);
    uint32_t w1 = part[2] | (part[3] << 16);
    uint32_t w2 = w0, w3 = w1;
    if (i == WI && half) {
      // a lane without a query never passes: start from +1e38
      const float cut =
          valid ? mc_filter_cut(r2, mc_damped_norm(ysq)) : -1e38f;
      float neg = -__builtin_fmaf(__builtin_fabsf(cut), 3.0517578125e-05f, cut);
      uint32_t hi, lo;
      if (__builtin_fabsf(neg) < 1e38f) {
        mc_split(neg, hi, lo);
      } else {
        hi = neg < 0.0f ? 0xff7fu : 0x7f7fu;
        lo = 0;
      }
      const uint32_t keep = ~(0xffffu << (16 * (WE & 1)));
      const uint32_t sh = 16 * (WE & 1);
      if (WE < 2) {
        w0 = (w0 & keep) | (hi << sh);
        w2 = (w2 & keep) | (lo << sh);
      } else {
        w1 = (w1 & keep) | (hi << sh);
        w3 = (w3 & keep) | (lo << sh);
      }
    }
    yb[i] = __builtin_bit_cast(mc_bf16x8_t, make_uint4(w0, w1, w2, w3));
  }
  const uint32_t one_keep =
      half ? ~(0xffffu << (16 * (WE & 1))) : 0xffffffffu;
  const uint32_t one_bits = half ? (0x3f80u << (16 * (WE & 1))) : 0u;

  // neighbours found so far (kept by the lower lane of a pair, mirrored to
  // the upper one after every drain); a query without a slot left is done
  int count = 0;
  bool done = !valid || slots <= 0;
  int qn = 0; // parked steps of this pair: queue[0 .. qn)[lower, upper lane]
  const bool ignore_same = p.ignore_same_index != 0;
  int *const slot_row = p.out_idx + (size_t)(valid ? q : y_begin) * slots;

  // ---- tile staging -------------------------------------------------------
  uint4 stage[PT][REC];
  auto pad_quad = [](int i) {
    uint4 o = make_uint4(0u, 0u, 0u, 0u);
    if (i == DIM / 4) {
      const uint32_t nan_bits = 0x7fc0u << (16 * (DIM % 2));
      if (DIM % 4 < 2)
        o.x = nan_bits;
      else
        o.y = nan_bits;
    }
    return o;
  };
  auto load_tile = [&](int t) {
#pragma unroll
    for (int r = 0; r < PT; ++r) {
      const int pos = t * TX + r * kBlock + tid;
      const size_t g = (size_t)x_begin + pos;
      const bool ok = pos < c_count;
#pragma unroll
      for (int i = 0; i < REC; ++i)
        stage[r][i] = ok ? p.x_split[g * REC + i] : pad_quad(i);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int r = 0; r < PT; ++r)
#pragma unroll
      for (int i = 0; i < REC; ++i)
        rows_lds[i][r * kBlock + tid] = stage[r][i];
  };

  // Resolves the parked rows of the tile: the lower lane of every pair takes
  // them in ascending order.  (No nested loops or branches but the refill: all
  // lanes of a wave pass through every branch some lane takes.)
  auto drain = [&](int g_base, int rows) {
    uint32_t pending = 0;
    int base = 0, taken = 0;
    const int entries = half == 0 && !done ? qn : 0;
    for (;;) {
      const bool refill = pending == 0 && taken < entries;
      if (__any(refill)) {
        const int at = min(taken, QCAP - 1);
        const uint32_t mask = queue[at][tid];
        const int step = (int)queue[at][min(tid + 32, kBlock - 1)];
        pending = refill ? mask : pending;
        base = refill ? step * 32 : base;
        taken += refill ? 1 : 0;
      }
      const bool has = pending != 0;
      if (!__any(has))
        break;
      const int v = __builtin_clz(pending | 1u);
      const int j = base + v;
      pending &= ~(0x80000000u >> v);
      float row[XF];
#pragma unroll
      for (int e = 0; e < XF; e += 4) {
        const uint4 q4 = rows_lds[NI + e / 4][min(j, TX - 1)];
        row[e] = __uint_as_float(q4.x);
        row[e + 1] = __uint_as_float(q4.y);
        row[e + 2] = __uint_as_float(q4.z);
        row[e + 3] = __uint_as_float(q4.w);
      }
      const float d0 = row[0] - yq[0];
      float dist = d0 * d0;
#pragma unroll
      for (int c = 1; c < DIM; ++c) {
        const float dc = row[c] - yq[c];
        dist = __builtin_fmaf(dc, dc, dist);
      }
      const int g = g_base + j;
      // (j < rows: no padding rows)
      if (has && dist < r2 && j < rows && !(ignore_same && g == q)) {
        slot_row[count] = g;
        ++count;
        if (count >= slots) {
          pending = 0;
          taken = entries;
        }
      }
    }
    qn = 0;
    // the upper lane learns whether the query still has room
    const bool full = count >= slots;
    const auto f = __builtin_amdgcn_permlane32_swap((unsigned)full,
                                                    (unsigned)full, false,
                                                    false);
    if (f[0]) // the lower lane's verdict, for both lanes
      done = true;
  };

  if (num_tiles > 0)
    load_tile(0);
  bool wave_done = false;
  int few = 0, few_before = 0; // open queries, those of the waves before
  int t = 0;

  for (; t < num_tiles; ++t) {
    // one LDS buffer: the next tile waits in registers while this one is
    // scanned
    // (no lane has anything parked here)
    const uint32_t open_queries = (uint32_t)__ballot(!done);
    if (lane == 0)
      queue[0][wave * kWave] = (uint32_t)__builtin_popcount(open_queries);
    __syncthreads();
    int open = 0;
    few_before = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
      few_before = w == wave ? open : few_before;
      open += (int)queue[0][w * kWave];
    }
    // (read between two barriers: the same for every thread)
    if (open <= kRadiusFew) {
      few = open;
      break;
    }
    store_tile();
    __syncthreads();
    if (t + 1 < num_tiles)
      load_tile(t + 1);
    if (wave_done)
      continue;
    const int g_base = x_begin + t * TX;
    const int rows = min(TX, c_count - t * TX);
    const int steps32 = (rows + 31) / 32;

    uint4 a_next[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
      a_next[i] = rows_lds[i][col];
    for (int rt = 0; rt < steps32; ++rt) {
      mfma_acc_t acc = {0};
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        uint4 a = a_next[i];
        if (i == WI) {
          // upper lanes: 1 in place of w_hi and w_lo (times -cut' parts)
          if (WE < 2) {
            a.x = (a.x & one_keep) | one_bits;
            a.z = (a.z & one_keep) | one_bits;
          } else {
            a.y = (a.y & one_keep) | one_bits;
            a.w = (a.w & one_keep) | one_bits;
          }
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(mc_bf16x8_t, a), yb[i], acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < NI; ++i)
        a_next[i] = rows_lds[i][min(rt + 1, TX / 32 - 1) * 32 + col];

      uint32_t mask = 0;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(acc[v]), 31);
      if (done)
        mask = 0;
      if (__any(mask != 0)) {
        // the rows of both lanes of a pair in order: nibbles of the lower and
        // of the upper lane in turn, the first row in the highest bit
        uint32_t rows_of = (mask | (mask << 8)) & 0x00ff00ffu;
        rows_of = (rows_of | (rows_of << 4)) & 0x0f0f0f0fu;
        rows_of <<= half == 0 ? 4 : 0;
        const auto both = __builtin_amdgcn_permlane32_swap(rows_of, rows_of,
                                                           false, false);
        rows_of = both[0] | both[1];
        if (rows_of != 0) {
          queue[qn][tid] = half == 0 ? rows_of : (uint32_t)rt;
          ++qn;
        }
        if (__any(qn >= QCAP)) {
          drain(g_base, rows);
          if (!__any(!done))
            break;
        }
      }
    }
    drain(g_base, rows);
    if (!__any(!done))
      wave_done = true;
  }

  if (few > 0) {
    // entry e: query, slots filled, coordinates
    constexpr int W = kBlock / kWave;
    constexpr int MINE = (kRadiusFew + W - 1) / W;
    static_assert(DIM * kRadiusFew <= kBlock && QCAP >= 4, "the queue's rows");
    const uint32_t open_queries = (uint32_t)__ballot(!done);
    const int entry =
        few_before + __builtin_popcount(open_queries & ((1u << col) - 1u));
    const bool mine = half == 0 && !done;
    if (mine) {
      queue[1][entry] = (uint32_t)q;
      queue[2][entry] = (uint32_t)count;
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        queue[3][c * kRadiusFew + entry] = __float_as_uint(yq[c]);
    }
    __syncthreads();
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    auto uniform = [](uint32_t v) {
      return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    };
    int of[MINE], filled[MINE];
    float at[MINE][DIM];
    uint32_t open = 0; // the wave's queries that are not full
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      const int e = min(wave_u + W * i, few - 1);
      of[i] = (int)uniform(queue[1][e]);
      filled[i] = (int)uniform(queue[2][e]);
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        at[i][c] = __uint_as_float(uniform(queue[3][c * kRadiusFew + e]));
      open |= wave_u + W * i < few ? 1u << i : 0u;
    }
    // the rows from the tile that waits in registers on, straight from memory,
    // one round of G x 64 ahead of the one that is looked at
    constexpr int G = DIM <= 4 ? 4 : 2;
    float next[G][DIM];
    auto load_rows = [&](int pos) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int row = x_begin + min(pos + g * kWave + lane, c_count - 1);
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          next[g][c] = c < d_in ? p.x[(size_t)row * d_in + c] : 0.0f;
      }
    };
    if (open != 0)
      load_rows(t * TX);
    for (int pos = t * TX; pos < c_count && open != 0; pos += G * kWave) {
      float row[G][DIM];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          row[g][c] = next[g][c];
      if (pos + G * kWave < c_count)
        load_rows(pos + G * kWave);
#pragma unroll
      for (int i = 0; i < MINE; ++i) {
        if ((open & (1u << i)) == 0)
          continue;
        bool hit[G];
        bool any = false;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float d0 = row[g][0] - at[i][0];
          float dist = d0 * d0;
#pragma unroll
          for (int c = 1; c < DIM; ++c) {
            const float dc = row[g][c] - at[i][c];
            dist = __builtin_fmaf(dc, dc, dist);
          }
          hit[g] = dist < r2;
          any = any || hit[g];
        }
        if (!__any(any))
          continue;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int j = pos + g * kWave + lane;
          const bool take = hit[g] && j < c_count &&
                            !(p.ignore_same_index && x_begin + j == of[i]);
          const uint64_t hits = __ballot(take);
          const int slot =
              filled[i] + (int)__builtin_amdgcn_mbcnt_hi(
                              (uint32_t)(hits >> 32),
                              __builtin_amdgcn_mbcnt_lo((uint32_t)hits, 0u));
          if (take && slot < slots)
            p.out_idx[(size_t)of[i] * slots + slot] = x_begin + j;
          filled[i] += __builtin_popcountll(hits);
        }
        if (filled[i] >= slots) {
          filled[i] = slots;
          open &= ~(1u << i);
        }
      }
    }
    // the lanes that own the queries take the counts back
#pragma unroll
    for (int i = 0; i < MINE; ++i)
      if (lane == 0 && wave_u + W * i < few)
        queue[2][wave_u + W * i] = (uint32_t)filled[i];
    __syncthreads();
    if (mine)
      count = (int)queue[2][entry];
  }

  if (valid && half == 0) {
    p.out_count[q] = count;
    if (p.edge_sums != nullptr) // (count <= slots; wide lists: one by one)
      if (p.slots < 128)
        add_to_block_sum(p.edge_sums, q / kCompactBlockQueries, count);
      else
        atomicAdd(&p.edge_sums[q / kCompactBlockQueries],
                  (unsigned long long)count);
  }
}

} // namespace pca
