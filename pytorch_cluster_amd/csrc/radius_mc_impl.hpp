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
// lanes puts the masks of its 32 rows into an LDS queue, 16 steps of 32 rows
// at a time (8 for d > 4).  A candidate with an exact distance below r^2
// always has its sign bit set (error budget in knn_lowd_mc_impl.hpp); whether
// a row with the bit set IS a neighbour is decided by the exact distance
// (direct differences, one FMA per component in ascending order) taken from
// the fp32 coordinates in the LDS tile.
//
// Lanes l and l + 32 share a query and see interleaved groups of four rows.
// After the 16 steps the lower lane of each pair walks the rows that passed
// in ascending order and appends the neighbours to the query's slot row until
// it holds max_num_neighbors.  (No branch in a step, and a walk is as long as
// that of its longest lane: the longer the steps gather, the fewer rounds.
// Steps parked one by one in a queue of eight that is walked when some lane's
// is full: 580 cycles a step and 83 rounds per wave instead of 180 and 64.)
// A wave whose queries are all full skips the matrix-core work, a workgroup
// whose waves are all done leaves the scan.
//
// A few queries far from everything would keep the whole workgroup scanning
// (clustered points: after an eighth of the rows 85 % of the queries are
// full, but hardly a wave is).  So from the first tile on at whose start at
// most kRadiusFew queries are open, these become the 32 columns of every wave,
// and the waves share the rows: 16 steps each, operands straight from memory,
// the exact distances of even and odd steps by the two lanes of a pair; the
// waves tell each other how many hits they have and each writes its own behind
// those of the waves before it.  One barrier per 2,048 rows (1,024 for d > 4), no
// tiles.  An exact scan per query costs a wave 8 instructions per 64 rows whatever
// they hold, the filter 30 per 32 rows x 32 queries and then some 60 for a row that
// passes: where more than few + 8 of a lane's 256 rows (128) pass, or up to four
// queries are open, the rest is scanned query by query.  (32 queries each in
// 64 clouds of 16,384 points, by neighbours per query: 20 / 70 / 230 / 1,000 /
// 4,400: 72 / 77 / 118 / 182 / 239 us, all by query 116 / 156 / 234 / 270 /
// 249 us; a threshold without the 8: 234 us for the fourth, with 2 few: 253 us
// for the last.)  So are the rows of less than a wave at the end, which would leave
// three waves idle (32 queries each in 128 clouds of 2,500 rows, 0.05 / 0.5 / 4 % in
// reach: 56 / 62 / 59 -> 48 / 53 / 50 us), and all of them where no tile was scanned
// yet and after four steps most lists look full soon (64 clouds of 4,096 rows, lists
// of 32, 20 / 40 % in reach: 8 queries each 41 / 40 -> 39 / 38 us, 16 42 / 41 -> 41 /
// 39, 32 45 / 42 -> 44 / 40; all by query 40 / 39, 42 / 40, 44 / 41).  Between that and the
// few hits that the filter is for, at 4 - 12 % in reach, short lists take up to 10 %
// more time than all by query (32 queries, 12 %: 58 us instead of 48): four steps
// cannot tell, and asking 256 rows query by query first costs the others 4 us.
//
// 8 clouds of 16,384 clustered points, r = 0.05, 32 neighbours: kernel 132 ->
// 100 us (the shared rows alone 117 us), r = 0.02: the call 277 -> 225 us.
// It is bound by instruction issue: about half of them in the walks, a fifth
// in the last queries.
//
// A workgroup owns 128 queries of one segment and scans the whole segment
// (rows must be reported in order, so the segment is not sliced).
#pragma once

#include "knn_lowd_mc_impl.hpp"

namespace pca {

constexpr int kRadiusFew = 32; // open queries a workgroup deals to its waves
// Rows times open queries that take as long query by query as a round of the filter
// and its walks.
constexpr float kRadiusSoon = 8192.0f;

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
  constexpr int STEPS = DIM <= 4 ? 16 : 8; // of 32 rows, filtered at a time
  constexpr int PT = TX / kBlock; // rows staged per thread

  // (every 16-byte unit of a row in a plane of its own, as in
  // knn_lowd_mc_impl.hpp: conflict-free reads)
  __shared__ __attribute__((aligned(16))) uint4 rows_lds[REC][TX];
  // the rows that passed, per step and query, the first row in the highest bit
  // (also carries, between the two barriers at the top of a tile, the four
  // waves' numbers of open queries: one more variable would take the
  // workgroup past 40,960 bytes, the most that lets four of them share a CU)
  __shared__ uint32_t queue[STEPS][kBlock / 2];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int half = lane >> 5;
  const int col = lane & 31;
  const int pair = wave * 32 + col;

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
  // B operands as in knn_lowd_mc_kernel: the hi (lanes 0-31) or lo (lanes
  // 32-63) parts of (-2 y, 1, 0 ...), the upper lanes with the parts of -cut'
  // where the lo part of the 1 would be
  constexpr int WI = DIM / 4;
  constexpr int WE = DIM % 4;
  auto operands = [&](bool is, const float(&y)[DIM], mc_bf16x8_t(&out)[NI]) {
    float ysq = y[0] * y[0];
#pragma unroll
    for (int c = 1; c < DIM; ++c)
      ysq = __builtin_fmaf(y[c], y[c], ysq);
    const bool moderate = ysq <= kFilterNormLimit;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t part[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = 4 * i + e;
        float v = 0.0f;
        if (c < DIM)
          v = (is && moderate) ? -2.0f * y[c] : 0.0f;
        else if (c == DIM)
          v = is ? 1.0f : 0.0f;
        uint32_t hi, lo;
        mc_split(v, hi, lo);
        part[e] = half ? lo : hi;
      }
      uint32_t w0 = part[0] | (part[1] << 16);
      uint32_t w1 = part[2] | (part[3] << 16);
      uint32_t w2 = w0, w3 = w1;
      if (i == WI && half) {
        // a lane without a query never passes: start from +1e38
        const float cut = is ? mc_filter_cut(r2, mc_damped_norm(ysq)) : -1e38f;
        float neg =
            -__builtin_fmaf(__builtin_fabsf(cut), 3.0517578125e-05f, cut);
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
      out[i] = __builtin_bit_cast(mc_bf16x8_t, make_uint4(w0, w1, w2, w3));
    }
  };
  mc_bf16x8_t yb[NI];
  operands(valid, yq, yb);
  const uint32_t one_keep =
      half ? ~(0xffffu << (16 * (WE & 1))) : 0xffffffffu;
  const uint32_t one_bits = half ? (0x3f80u << (16 * (WE & 1))) : 0u;
  // the filter of 32 rows x 32 queries: the sign bits of a lane's 16 results,
  // the first row's in bit 15
  auto passing = [&](const uint4(&rows)[NI], const mc_bf16x8_t(&qb)[NI]) {
    mfma_acc_t acc = {0};
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint4 a = rows[i];
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
          __builtin_bit_cast(mc_bf16x8_t, a), qb[i], acc, 0, 0, 0);
    }
    uint32_t mask = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v)
      mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(acc[v]), 31);
    return mask;
  };
  // Steps [from, to) of the filter into the queue: those with a row that passed
  // as a set, the rows of the lane's steps that passed added to `ones`.  A swap gives the
  // lower lane of a pair both masks of the first of two steps, the upper lane
  // those of the second; their nibbles alternate in the rows' order.
  auto filter = [&](auto from, auto to, auto rows_of_step,
                    const mc_bf16x8_t(&qb)[NI], int &ones) {
    uint32_t some = 0;
#pragma unroll
    for (int s = from; s < to; s += 2) {
      uint4 rows[NI];
      rows_of_step(s, rows);
      const uint32_t first = passing(rows, qb);
      rows_of_step(s + 1, rows);
      const uint32_t second = passing(rows, qb);
      const auto m =
          __builtin_amdgcn_permlane32_swap(first, second, false, false);
      // bytes: lower lane's, upper lane's, lower lane's, upper lane's
      const uint32_t u = __builtin_amdgcn_perm(m[0], m[1], 0x05010400u);
      const uint32_t word = (u & 0xf00ff00fu) | ((u & 0x0f000f00u) >> 4) |
                            ((u & 0x00f000f0u) << 4);
      queue[s + half][pair] = word;
      some |= word != 0 ? 1u << s : 0u;
      ones += __builtin_popcount(word);
    }
    const auto f = __builtin_amdgcn_permlane32_swap(some, some, false, false);
    return f[0] | (f[1] << 1);
  };

  // neighbours found so far (kept by the lower lane of a pair, mirrored to
  // the upper one after every drain); a query without a slot left is done
  int count = 0;
  // (nor has one with a component that is no finite number any neighbour)
  bool done = !valid || slots <= 0;
#pragma unroll
  for (int c = 0; c < DIM; ++c)
    done = done || !(__builtin_fabsf(yq[c]) <= 3.402823466e+38f);
  const bool ignore_same = p.ignore_same_index != 0;
  const int self = ignore_same ? q : -1; // the row that is left out
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

  // Resolves STEPS steps of the tile from row `start` on: the lower lane of
  // every pair takes the rows that passed in ascending order.  (No nested loops
  // or branches but the refill: all lanes of a wave pass through every branch
  // some lane takes.)
  auto drain = [&](uint32_t left, int start, int g_base, int rows) {
    uint32_t pending = 0;
    int base = 0;
    left = half == 0 && !done ? left : 0u;
    for (;;) {
      const bool refill = pending == 0 && left != 0;
      if (__any(refill)) {
        const int next = __builtin_ctz(left | (1u << (STEPS - 1)));
        const uint32_t mask = queue[next][pair];
        pending = refill ? mask : pending;
        base = refill ? start + next * 32 : base;
        left = refill ? left & (left - 1u) : left;
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
        const uint4 q4 = rows_lds[NI + e / 4][j];
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
      if (has && dist < r2 && j < rows && g != self) {
        slot_row[count] = g;
        ++count;
        if (count >= slots) {
          pending = 0;
          left = 0;
        }
      }
    }
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
  constexpr std::integral_constant<int, 0> no_steps{};
  constexpr std::integral_constant<int, STEPS> all_steps{};
  bool wave_done = false;
  int few = 0, few_before = 0; // open queries, those of the waves before
  int t = 0;

  for (; t < num_tiles; ++t) {
    // one LDS buffer: the next tile waits in registers while this one is
    // scanned
    const uint32_t open_queries = (uint32_t)__ballot(!done);
    if (lane == 0)
      queue[0][wave * 32] = (uint32_t)__builtin_popcount(open_queries);
    __syncthreads();
    int open = 0;
    few_before = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
      few_before = w == wave ? open : few_before;
      open += (int)queue[0][w * 32];
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
    for (int start = 0; start < rows; start += STEPS * 32) {
      int ones = 0;
      const uint32_t some = filter(
          no_steps, all_steps,
          [&](int s, uint4(&a)[NI]) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
              a[i] = rows_lds[i][start + s * 32 + col];
          },
          yb, ones);
      drain(some, start, g_base, rows);
      if (!__any(!done))
        break;
    }
    if (!__any(!done))
      wave_done = true;
  }

  if (few > 0) {
    // The open queries, in the tile's LDS: query, slots filled, coordinates;
    // behind them the hits per wave and query of two rounds.
    constexpr int W = kBlock / kWave;
    constexpr int ROUND = W * STEPS * 32;
    constexpr int AHEAD = NI == 1 ? 8 : NI == 2 ? 4 : 2;
    constexpr uint32_t kMany = 0xffffffffu;
    constexpr int LOOK = 4; // steps after which a wave may know better
    static_assert((2 + DIM + 2 * W) * kRadiusFew <= 4 * TX, "the tile's LDS");
    uint32_t *const table = reinterpret_cast<uint32_t *>(&rows_lds[0][0]);
    uint32_t *const hits_of = table + (2 + DIM) * kRadiusFew;
    const uint32_t open_queries = (uint32_t)__ballot(!done);
    const int entry =
        few_before + __builtin_popcount(open_queries & ((1u << col) - 1u));
    const bool handed = half == 0 && !done;
    if (handed) {
      table[entry] = (uint32_t)q;
      table[kRadiusFew + entry] = (uint32_t)count;
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        table[(2 + c) * kRadiusFew + entry] = __float_as_uint(yq[c]);
    }
    __syncthreads();
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int e = min(col, few - 1);
    const int qe = (int)table[e];
    const int self_e = ignore_same ? qe : -1;
    int filled = (int)table[kRadiusFew + e];
    float at[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      at[c] = __uint_as_float(table[(2 + c) * kRadiusFew + e]);
    bool full = col >= few;
    operands(!full, at, yb);
    int *const row_of = p.out_idx + (size_t)qe * slots;

    // packed rows straight from memory, AHEAD steps ahead of the filter
    const uint4 *const packed = p.x_split + (size_t)x_begin * REC;
    uint4 ahead[AHEAD][NI];
    auto load_step = [&](int pos, uint4(&a)[NI]) {
      const size_t row = (size_t)min(pos + col, c_count - 1);
#pragma unroll
      for (int i = 0; i < NI; ++i)
        a[i] = packed[row * REC + i];
    };
    int first = t * TX + wave_u * (STEPS * 32); // the wave's rows of a round
    // (up to a query a wave: query by query at once, which takes no more time)
    const bool filtered = few > W;
    if (filtered) {
#pragma unroll
      for (int s = 0; s < AHEAD; ++s)
        load_step(first + s * 32, ahead[s]);
    }
    int rest = t * TX; // the first row that no query was compared to
    // (the rows of less than a wave would leave the others idle)
    for (int round = 0; filtered && c_count - rest > STEPS * 32; ++round) {
      auto rows_ahead = [&](int s, uint4(&a)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
          a[i] = ahead[s % AHEAD][i];
        const int next = s + AHEAD;
        load_step(first + (next < STEPS ? next * 32
                                        : ROUND + (next - STEPS) * 32),
                  ahead[s % AHEAD]);
      };
      constexpr std::integral_constant<int, LOOK> look{};
      const int there = c_count - first; // rows of the wave
      int ones = 0;
      uint32_t some = 0;
      bool many = false; // too many pass, or most lists are full soon
      if (there > 0) {
        some = filter(no_steps, look, rows_ahead, yb, ones);
        if (t == 0 && round == 0 && there >= STEPS * 32) {
          const auto both = __builtin_amdgcn_permlane32_swap(
              (unsigned)ones, (unsigned)ones, false, false);
          const float met = (float)(both[0] + both[1]); // of LOOK x 32 rows
          const uint64_t soon =
              __ballot(!full && met * (kRadiusSoon / (LOOK * 32)) >=
                                    (float)(slots - filled) * (float)few);
          many = 4 * __builtin_popcountll(soon) >=
                 3 * __builtin_popcountll(__ballot(!full));
        }
      }
      if (there > 0 && !many) {
        some |= filter(look, all_steps, rows_ahead, yb, ones);
        if (there < STEPS * 32) {
          // (beyond the last row it was that row again)
          const int last = there / 32; // the first step that is not whole
          some &= (2u << last) - 1u;
          const uint32_t rest_of = ~(uint32_t)(0xffffffffull >> (there & 31));
          if ((last & 1) == half)
            queue[last][pair] &= rest_of;
          ones = 0;
          for (int s = half; s <= last; s += 2)
            ones += __builtin_popcount(queue[s][pair]);
        }
        many = __any(!full && ones > few + 8);
      }
      some = full ? 0u : some;
      // the lower lane of a pair takes the even steps, the upper lane the odd
      // ones; what is left of a mask are the hits
      uint32_t left = many ? 0u : some & (half ? 0xaaaaaaaau : 0x55555555u);
      uint32_t pending = 0;
      int mine = 0, step = 0;
      for (;;) {
        const bool refill = pending == 0 && left != 0;
        if (__any(refill)) {
          const int next = __builtin_ctz(left | (1u << (STEPS - 1)));
          const uint32_t mask = queue[next][pair];
          pending = refill ? mask : pending;
          step = refill ? next : step;
          left = refill ? left & (left - 1u) : left;
        }
        const bool has = pending != 0;
        if (!__any(has))
          break;
        const int v = __builtin_clz(pending | 1u);
        const uint32_t bit = 0x80000000u >> v;
        pending &= ~bit;
        const int j = first + step * 32 + v;
        float row[XF];
#pragma unroll
        for (int i = 0; i < XF; i += 4) {
          const uint4 q4 =
              packed[(size_t)min(j, c_count - 1) * REC + NI + i / 4];
          row[i] = __uint_as_float(q4.x);
          row[i + 1] = __uint_as_float(q4.y);
          row[i + 2] = __uint_as_float(q4.z);
          row[i + 3] = __uint_as_float(q4.w);
        }
        const float d0 = row[0] - at[0];
        float dist = d0 * d0;
#pragma unroll
        for (int c = 1; c < DIM; ++c) {
          const float dc = row[c] - at[c];
          dist = __builtin_fmaf(dc, dc, dist);
        }
        const bool hit = dist < r2 && x_begin + j != self_e;
        mine += has && hit ? 1 : 0;
        if (has && !hit)
          queue[step][pair] &= ~bit;
      }

      // slots before the wave's own hits: those of the waves before it
      const auto both = __builtin_amdgcn_permlane32_swap(
          (unsigned)mine, (unsigned)mine, false, false);
      uint32_t *const hits = hits_of + (round & 1) * (W * kRadiusFew);
      if (half == 0)
        hits[wave_u * kRadiusFew + col] = many ? kMany : both[0] + both[1];
      __syncthreads();
      int slot = filled, after = filled;
      bool stop = false;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const uint32_t h = hits[w * kRadiusFew + col];
        stop = stop || h == kMany;
        slot += w < wave_u ? (int)h : 0;
        after += (int)h;
      }
      // (the same in every wave)
      if (__any(stop))
        break;
      rest += ROUND;
      left = half == 0 && slot < slots ? some : 0u;
      for (;;) {
        const bool refill = pending == 0 && left != 0;
        if (__any(refill)) {
          const int next = __builtin_ctz(left | (1u << (STEPS - 1)));
          const uint32_t mask = queue[next][pair];
          pending = refill ? mask : pending;
          step = refill ? next : step;
          left = refill ? left & (left - 1u) : left;
        }
        const bool has = pending != 0;
        if (!__any(has || left != 0))
          break;
        const int v = __builtin_clz(pending | 1u);
        pending &= ~(0x80000000u >> v);
        if (has) {
          row_of[slot] = x_begin + first + step * 32 + v;
          ++slot;
          if (slot >= slots) {
            pending = 0;
            left = 0;
          }
        }
      }
      filled = min(after, slots);
      full = full || filled >= slots;
      // (the same in every wave)
      if (!__any(!full))
        break;
      first += ROUND;
    }

    // Query by query: a wave takes every fourth one, and all rows from `rest`
    // on, straight from memory, G x 64 at a time, once for all its queries:
    // hits are found and numbered by ballots.  No barriers; a wave whose
    // queries are full leaves.
    constexpr int G = DIM <= 4 ? 4 : 2;
    constexpr int MINE = (kRadiusFew + W - 1) / W;
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
    const uint32_t still = (uint32_t)__ballot(!full);
    uint32_t open = 0; // the wave's queries that are not full
#pragma unroll
    for (int i = 0; i < MINE; ++i)
      open |= ((still >> (wave_u + W * i)) & 1u) << i;
    if (rest < c_count && open != 0)
      load_rows(rest);
    for (int pos = rest; pos < c_count && open != 0; pos += G * kWave) {
      float row[G][DIM];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          row[g][c] = next[g][c];
      if (pos + G * kWave < c_count)
        load_rows(pos + G * kWave);
      for (uint32_t left = open; left != 0; left &= left - 1u) {
        const int i = __builtin_ctz(left);
        const int of = wave_u + W * i;
        float to[DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          to[c] = __uint_as_float(
              __builtin_amdgcn_readlane(__float_as_uint(at[c]), of));
        bool hit[G];
        bool any = false;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float d0 = row[g][0] - to[0];
          float dist = d0 * d0;
#pragma unroll
          for (int c = 1; c < DIM; ++c) {
            const float dc = row[g][c] - to[c];
            dist = __builtin_fmaf(dc, dc, dist);
          }
          hit[g] = dist < r2;
          any = any || hit[g];
        }
        if (!__any(any))
          continue;
        const int self = __builtin_amdgcn_readlane(qe, of);
        int have = __builtin_amdgcn_readlane(filled, of);
        int *const list = p.out_idx + (size_t)self * slots;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int j = pos + g * kWave + lane;
          const bool take =
              hit[g] && j < c_count && !(ignore_same && x_begin + j == self);
          const uint64_t hits = __ballot(take);
          const int slot =
              have + (int)__builtin_amdgcn_mbcnt_hi(
                         (uint32_t)(hits >> 32),
                         __builtin_amdgcn_mbcnt_lo((uint32_t)hits, 0u));
          if (take && slot < slots)
            list[slot] = x_begin + j;
          have += __builtin_popcountll(hits);
        }
        if (have >= slots) {
          have = slots;
          open &= ~(1u << i);
        }
        filled = lane == of ? have : filled;
      }
    }
    // the lanes that own the queries take the counts back
    if ((col % W) == wave_u && half == 0 && col < few)
      table[kRadiusFew + col] = (uint32_t)filled;
    __syncthreads();
    if (handed)
      count = (int)table[kRadiusFew + entry];
  }

  if (valid && half == 0) {
    p.out_count[q] = count;
    if (p.edge_sums != nullptr) { // (count <= slots; wide lists: one by one)
      if (p.slots < 128)
        add_to_block_sum(p.edge_sums, q / kCompactBlockQueries, count);
      else
        atomicAdd(&p.edge_sums[q / kCompactBlockQueries],
                  (unsigned long long)count);
    }
  }
}

} // namespace pca
