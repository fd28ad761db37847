// `nearest` in feature space (fp32, 8 < d <= 128): every row of y gets the
// nearest row of x, the entries of a code book as a rule, with the results of
// the reference's loop (csrc/cuda/nearest_cuda.cu:10-66) bit for bit.
//
// ONE fp16 product per pair and component on the matrix cores ranks a query's
// candidates, and a few of them are evaluated exactly afterwards.  With
// a = s_c x, b = s_q y (s_c, s_q powers of two, of the call and of the
// workgroup's queries, that bring the largest component near the end of the fp16
// range) and
// r = s_q / s_c, a chain of v_mfma_f32_32x32x16_f16 that starts from
// kappa |a|^2 gives
//     s = kappa |a|^2 + sum_c h(a_c) h(-2 b_c),    h: fp16, |h| < 2^-14 flushed,
// and  s + |b|^2 / r - C  is a LOWER bound of s_c s_q |x - y|^2 for
//   * |a_c b_c' - h(a_c) h(b_c')| summed over the components (b' = 2 b): at
//     most (2^-10 + 2^-22) |a| |b'| + 2^-14 (1 + 2^-11) sqrt(d) (|a| + |b'|)
//     + d 2^-28;
//   * the accumulation: d + 16 terms, each within 2^-22 of a running magnitude
//     below |kappa| |a|^2 + 1.01 |a| |b'|;
//   * |a| |b'| <= l |a|^2 + |b|^2 / l with l = B / A, B the largest |b| of the
//     workgroup and A a typical |a|, and |a| <= (|a|^2 / A + A) / 2,
// (any A > 0 will do; it is the root mean square of the |a|, or twice their
// geometric mean where large rows bring the mean square above that) so that
//     kappa = r (1 - delta) - eps l - 2^-15 sqrt(d) / A  and
//     C = eps |b|^2 / l + 2^-15 sqrt(d) A + 2^-13 sqrt(d) |b| + d 2^-27
// (each sqrt term times 1.01), eps = 2^-10 + (d + 20) 2^-21,
// delta = (d + 20) 2^-21.
//
// A scan keeps, per query and half of the rows (lanes l and l + 32 share a
// query and see rows 8 v + 4 (l / 32) + 0..3 of 32), the three smallest
// MINIMA OF FOUR consecutive rows, the number of the four in the low nine bits
// of the value (2^-14 of it, which the cut allows for).  That is 24 vector
// instructions for 16 values; the matrix cores need 32 cycles per 16
// components for them, and the vector ALU 4 cycles each: alike from 48
// components on, more for the vector ALU below.  After 4,096 rows the four rows of a query's
// smallest minimum are evaluated exactly; their distance D gives the cut
// below which s has to lie for a row to come before them; of the other
// minima kept, those below the cut are evaluated too.  Only if at the end of
// the example a third minimum lies below the final cut (four fours of rows
// within the rounding margin of the nearest one: duplicates, rows far from the
// origin) there may be candidates that were not kept: the workgroup then goes
// through such 4,096 rows again and evaluates whatever lies below the cut.
//
// One row or query far larger than the others must not set the scale, A or l for
// all.  Rows of a norm beyond 4,096 times the geometric mean take part with
// zeros for operands and s = r |a|^2 / 4 - B^2 / r, a lower bound as long as
// |b| <= r |a| / 2 (otherwise they are left to a second pass).  Queries with a
// component of 2^12 times the workgroup's mean are searched exactly, and where
// the largest of the others is far beyond an ordinary one, l lies between the
// two.  Calls of 100,000 queries x 4,096 rows x 64, 135 us: with one row a
// million times the others 18,050 us without the limit, 162 with it; with every
// thousandth query ten thousand times the others 4,660, now 162.  50,000 x
// 8,192 x 128: the candidates of all scans but the one with the nearest row were
// searched for again before its distance was known; 300 -> 240 us, 10 standard
// deviations from the origin 1,004 -> 254.  What is left: an entry that occurs
// 16 times or more brings the second pass to every query (640 us; the
// kernel of knn_mfma_impl.hpp 407).
//
// Rows of x with a component that is not finite never qualify (their distance
// is not below 1e38); finite ones of |x|^2 > 1e30 enter with s = -1e37, always
// looked at.  Queries likewise: not finite, no candidate; |y|^2 > 1e30, searched
// exactly.
//
// Mapping: a workgroup owns 4 waves x S x 32 queries of one segment; the query
// operands stay in registers, packed rows of x (2 NB units of 16 bytes, an odd
// stride against bank conflicts) go through two LDS tiles of 128 rows filled
// by LDS-direct loads.  S sets of queries per wave share the reads of a row:
// with one set the LDS would have to deliver 128 bytes per cycle and CU, all
// it can.
//
// Measured figures: nearest_feat.hip.
#pragma once

#include "device_utils.hpp"
#include "knn_lowd_impl.hpp"
#include "launchers.hpp"

namespace pca {

typedef _Float16 nf_f16x8_t __attribute__((ext_vector_type(8)));
typedef float nf_acc_t __attribute__((ext_vector_type(16)));
// four floats at any float's address
typedef float nf_float4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kNfTileRows = 128;
constexpr int kNfEpochRows = 4096; // nine bits: 128 steps of 32 rows, 8 fours
constexpr uint32_t kNfIndexMask = 511u;
constexpr float kNfNothing = 1.7e38f;  // s of a row that is none
constexpr float kNfAlways = -1e37f;    // s of a row that is always looked at
constexpr float kNfCutLimit = 1e38f;

// What the rows' operands are made with.
struct NfRows {
  float typical;  // the A of the bound, unscaled
  float limit_sq; // rows of a larger squared norm have no operands
  float scale;
};
struct NearestFeatGlobals {
  unsigned max_bits; // largest |component| of the moderate rows of x
  unsigned rows;     // moderate rows of x that are not zero
  double sum_sq;     // of their squared norms
  double sum_log;    // of log2 of those
  NfRows rows_of_x;  // what follows from these (by the pack kernel)
};

struct NearestFeatParams {
  const float *x; // [n, d] candidates
  const float *y; // [m, d] rows that search
  const int64_t *ptr_x;
  const int64_t *ptr_y;
  int n, m, d, num_segments;
  const int *work_start;
  const uint4 *pack;   // [n + kNfTileRows][2 NB + 1] fp16 rows
  const float *weight; // [n] |x|^2, -1: always looked at, -2: never
  const NearestFeatGlobals *globals;
  int64_t *out;
};

__device__ __forceinline__ float nf_uniform(float v) {
  return __uint_as_float(
      (uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v)));
}
__device__ __forceinline__ double nf_uniform(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Largest components after scaling: rows in [2^14, 2^15), queries in [2^13,
// 2^14), as -2 b has to be an fp16 number too.  What is flushed below 2^-14 is
// that much less of a small row or query than with feat_inv_sigma alone ([2^10,
// 2^11)).  Norms of both log-normal with sigma 2, us a call, with the second
// term of per_sq (below) taken for r_inv + 1 / as it is, scaled so: 100,000 x
// 4,096 x 64 342 / 221, 50,000 x 4,096 x 128 489 / 305; of the rows with sigma 3
// 476 / 192 and 7,469 / 247.
constexpr float kNfRowScale = 16.0f;
constexpr float kNfQueryScale = 8.0f;

constexpr float kNfLargeRow = 4096.0f;
constexpr int kNfLargeExponents = 12;
__device__ __forceinline__ float nf_mean_norm(double sum_log, unsigned rows) {
  return rows != 0 ? __builtin_exp2f((float)(0.5 * sum_log / (double)rows))
                   : 1.0f;
}
__device__ __forceinline__ NfRows nf_rows(const NearestFeatGlobals *g) {
  NfRows r;
  const float mean = nf_mean_norm(g->sum_log, g->rows);
  const float rms =
      g->rows != 0 ? (float)__builtin_sqrt(g->sum_sq / (double)g->rows) : 1.0f;
  r.typical = __builtin_fminf(rms, 2.0f * mean);
  const float limit = __builtin_fminf(mean * kNfLargeRow, 1e18f);
  r.limit_sq = limit * limit;
  r.scale = kNfRowScale *
            feat_inv_sigma(min(g->max_bits, __float_as_uint(limit)));
  return r;
}

__device__ __forceinline__ uint4 nf_pack8(const float (&v)[8]) {
  uint32_t h[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    h[e] = feat_h(v[e]);
  return make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16),
                    h[4] | (h[5] << 16), h[6] | (h[7] << 16));
}

// Components c0 .. c0 + 7 of a row (zeros from d on).
__device__ __forceinline__ void nf_load8(const float *row, int c0, int d,
                                         float (&v)[8]) {
  if (c0 + 8 <= d) {
    const nf_float4 a = *reinterpret_cast<const nf_float4 *>(row + c0);
    const nf_float4 b = *reinterpret_cast<const nf_float4 *>(row + c0 + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = c0 + e < d ? row[c0 + e] : 0.0f;
  }
}

// The reference's distance: direct differences, one fused multiply-add per
// component in ascending order.  R rows at a time.
template <int R>
__device__ __forceinline__ void nf_exact(const float *y, const float *x,
                                         const int (&row)[R], int d,
                                         float (&dist)[R]) {
#pragma unroll
  for (int i = 0; i < R; ++i)
    dist[i] = 0.0f;
  int c = 0;
#pragma unroll 2
  for (; c + 4 <= d; c += 4) {
    const nf_float4 q = *reinterpret_cast<const nf_float4 *>(y + c);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const nf_float4 p = *reinterpret_cast<const nf_float4 *>(
          x + (size_t)row[i] * d + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float t = p[e] - q[e];
        dist[i] = __builtin_fmaf(t, t, dist[i]);
      }
    }
  }
#pragma unroll 1
  for (; c < d; ++c) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float t = x[(size_t)row[i] * d + c] - y[c];
      dist[i] = __builtin_fmaf(t, t, dist[i]);
    }
  }
}

// (distance, order among equal ones) as one number; kNfNoKey: none below 1e38
constexpr unsigned long long kNfNoKey = ~0ull;
__device__ __forceinline__ unsigned long long nf_key(float dist, int rel) {
  return dist < kNearestLimit
             ? ((unsigned long long)__float_as_uint(dist) << 32) |
                   nearest_tie((uint32_t)rel)
             : kNfNoKey;
}

// NB blocks of 16 components (16 (NB - 1) < d <= 16 NB), S sets of 32 queries
// per wave.
template <int NB, int S>
__global__ __launch_bounds__(kBlock, 2) void
nearest_feat_kernel(NearestFeatParams p) {
  constexpr int RSU = 2 * NB + 1;
  constexpr int TR = kNfTileRows;
  constexpr int UNITS = TR * RSU;
  constexpr int PIECES = (UNITS + kWave - 1) / kWave;
  constexpr int WAVES = kBlock / kWave;
  constexpr int WAVE_PIECES = (PIECES + WAVES - 1) / WAVES;
  constexpr int TQ = WAVES * S * 32;
  static_assert(UNITS % kWave == 0, "whole pieces");
  __shared__ __attribute__((aligned(16))) uint4 tile_rows[2][UNITS];
  __shared__ __attribute__((aligned(16))) float tile_weight[2][TR];
  __shared__ unsigned wave_top[WAVES];
  __shared__ unsigned wave_queries[WAVES];
  __shared__ float wave_norm[WAVES];
  __shared__ unsigned long long wave_scans[WAVES];
  __shared__ unsigned long long wave_best[2][WAVES];
  __shared__ uint32_t alone[WAVES][S]; // queries searched exactly

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int half = lane >> 5;
  const int col = lane & 31;

  const int tile = blockIdx.x;
  if (tile >= p.work_start[p.num_segments])
    return;
  const int seg = find_segment(p.work_start, p.num_segments, tile);
  const int x_begin = p.ptr_x ? (int)p.ptr_x[seg] : 0;
  const int x_end = p.ptr_x ? (int)p.ptr_x[seg + 1] : p.n;
  const int y_begin = p.ptr_y ? (int)p.ptr_y[seg] : 0;
  const int y_end = p.ptr_y ? (int)p.ptr_y[seg + 1] : p.m;
  const int q0 = y_begin + (tile - p.work_start[seg]) * TQ + wave * (S * 32) +
                 col;
  const int d = p.d;

  // ---- queries ------------------------------------------------------------
  // 0: no query, or one no candidate is close enough to; 1: through the
  // filter; 2: searched exactly
  int kind[S];
  uint32_t top_bits[S]; // largest component
  unsigned bits = 0;
  // exponents of the queries that are not zero, added up, from bit 16 on their
  // number, from bit 24 on that of the queries of the last kind (of a wave)
  unsigned queries = 0;
  static_assert(S <= 4, "sums over 128 queries");
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int q = q0 + s * 32;
    kind[s] = 0;
    top_bits[s] = 0;
    if (q < y_end) {
      const float *row = p.y + (size_t)q * d;
      float sq = 0.0f;
      unsigned top = 0;
#pragma unroll 1
      for (int b = 0; b < NB; ++b) {
        float v[8];
        nf_load8(row, 16 * b + 8 * half, d, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          sq = __builtin_fmaf(v[e], v[e], sq);
          top = max(top, __float_as_uint(v[e]) & 0x7fffffffu);
        }
      }
      sq += __shfl_xor(sq, 32);
      top = max(top, (unsigned)__shfl_xor((int)top, 32));
      kind[s] = top >= 0x7f800000u ? 0 : sq <= kFilterNormLimit ? 1 : 2;
      top_bits[s] = top;
      if (kind[s] == 1) {
        bits = max(bits, top);
        queries += top != 0 ? (top >> 23) + 0x10000u : 0u;
      } else if (kind[s] == 2) {
        queries += 0x1000000u;
      }
    }
  }
#pragma unroll
  for (int sh = 1; sh < 32; sh <<= 1) {
    bits = max(bits, (unsigned)__shfl_xor((int)bits, sh));
    queries += (unsigned)__shfl_xor((int)queries, sh);
  }
  if (lane == 0) {
    wave_top[wave] = bits;
    wave_queries[wave] = queries;
  }
  __syncthreads();
  unsigned exponents = 0, counted = 0;
  bool any_alone = false;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    bits = max(bits, wave_top[w]);
    exponents += wave_queries[w] & 0xffffu;
    counted += (wave_queries[w] >> 16) & 0xffu;
    any_alone = any_alone || (wave_queries[w] >> 24) != 0;
  }
  // the mean exponent of the largest components
  const int mean_exponent =
      counted != 0 ? (int)((float)exponents / (float)counted) : 127;
  if ((int)(bits >> 23) > mean_exponent + kNfLargeExponents) {
    // a few queries far beyond the others' range (the same in all threads)
    any_alone = true;
    __syncthreads();
    bits = 0;
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (kind[s] == 1) {
        if ((int)(top_bits[s] >> 23) > mean_exponent + kNfLargeExponents)
          kind[s] = 2;
        else
          bits = max(bits, top_bits[s]);
      }
#pragma unroll
    for (int sh = 1; sh < 32; sh <<= 1)
      bits = max(bits, (unsigned)__shfl_xor((int)bits, sh));
    if (lane == 0)
      wave_top[wave] = bits;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      bits = max(bits, wave_top[w]);
  }
  const float s_q = kNfQueryScale * feat_inv_sigma(bits);

  nf_f16x8_t yb[S][NB];
  float ysq[S]; // |b|^2
  float top_sq = 0.0f;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int q = q0 + s * 32;
    ysq[s] = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (kind[s] == 1)
        nf_load8(p.y + (size_t)q * d, 16 * b + 8 * half, d, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[e] *= s_q;
        ysq[s] = __builtin_fmaf(v[e], v[e], ysq[s]);
        v[e] *= -2.0f;
      }
      yb[s][b] = __builtin_bit_cast(nf_f16x8_t, nf_pack8(v));
    }
    ysq[s] += __shfl_xor(ysq[s], 32);
    top_sq = __builtin_fmaxf(top_sq, ysq[s]);
  }
#pragma unroll
  for (int sh = 1; sh < 32; sh <<= 1)
    top_sq = __builtin_fmaxf(top_sq, __shfl_xor(top_sq, sh));
  if (lane == 0)
    wave_norm[wave] = top_sq;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w)
    top_sq = __builtin_fmaxf(top_sq, wave_norm[w]);

  // ---- constants of the bound ------------------------------------------------
  // (the same in every lane: kept in scalar registers)
  const NfRows rows_of_x = p.globals->rows_of_x;
  const float s_c = nf_uniform(rows_of_x.scale);
  const float limit_sq = nf_uniform(rows_of_x.limit_sq);
  const double scale2 = nf_uniform((double)s_c * (double)s_q);
  const double r = (double)s_q / (double)s_c;
  double typical = (double)rows_of_x.typical * (double)s_c;
  if (!(typical > 9.765625e-4 && typical < 1e7))
    typical = 1.0;
  // l: of the largest query, or of the geometric mean of it and of an ordinary
  // one where it is much larger (2^e of the largest component and less times
  // the root of d)
  float largest = __builtin_sqrtf(top_sq) + 1e-3f;
  {
    const float ordinary =
        2.0f * __builtin_sqrtf((float)d) *
        __uint_as_float((uint32_t)max(mean_exponent, 1) << 23) * s_q;
    if (largest > ordinary)
      largest = __builtin_sqrtf(largest) * __builtin_sqrtf(ordinary);
    // (of queries whose components are all flushed: any number will do)
    largest = __builtin_fmaxf(largest, 1e-3f);
  }
  const double lambda = (double)largest / typical;
  const double eps = 1.0 / 1024.0 + (double)(d + 20) / 2097152.0;
  const double delta = (double)(d + 20) / 2097152.0;
  const double root_d = nf_uniform(__builtin_sqrt((double)d) * 1.01);
  float kappa;
  {
    const double k = r * (1.0 - delta) - eps * lambda -
                     root_d / (32768.0 * typical);
    kappa = nf_uniform((float)(k < 1e30 ? k : 1e30));
  }
  const double r_inv = (double)s_c / (double)s_q;
  const double per_sq = nf_uniform(
      eps / lambda - r_inv +
      // (|b|^2 is a sum in fp32)
      (double)(d + 6) * (r_inv + eps / lambda) / 16777216.0);
  const double constant = nf_uniform(root_d * typical / 32768.0 +
                                     (double)d / 134217728.0);
  // (a factor beyond the fp32 range leaves no bound or the largest one)
  const float large_gain = nf_uniform((float)(0.24 * r * s_c * s_c));
  const float large_loss = nf_uniform((float)(1.01 * top_sq * r_inv));
  // the largest s a row can have whose distance is not above `dist`
  auto cut_of = [&](float dist, float sq) {
    const double norm = (double)__builtin_sqrtf(sq) * 1.000001;
    double c = scale2 * ((double)dist + (double)d * 5.7e-45) *
                   (1.0 + (double)(d + 6) / 16777216.0) +
               (double)sq * per_sq + root_d * norm / 8192.0 + constant;
    c += __builtin_fabs(c) * 2.4e-7; // (the conversion rounds)
    return c < (double)kNfCutLimit ? (float)c : kNfCutLimit;
  };
  // ... and the largest value its minimum of four can be kept as
  auto kept_cut = [](float cut) {
    return __builtin_fmaf(__builtin_fabsf(cut), 1.220703125e-4f, cut);
  };

  // the cut of a query whose best row so far is `best`
  auto query_cut = [&](unsigned long long best_row, float sq) {
    return cut_of(best_row != kNfNoKey
                      ? __uint_as_float((uint32_t)(best_row >> 32))
                      : kNearestLimit,
                  sq);
  };

  unsigned long long best[S];
  float cut[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    best[s] = kNfNoKey;
    cut[s] = kNfCutLimit;
  }

  // ---- one scan over rows c0 .. c1 of x ------------------------------------
  auto request = [&](int c0, int t, int buf) {
    const uint4 *src = p.pack + ((size_t)c0 + (size_t)t * TR) * RSU;
    const uint32_t dst = (uint32_t)(uintptr_t)&tile_rows[buf][0];
#pragma unroll
    for (int e = 0; e < WAVE_PIECES; ++e) {
      const int piece = wave + WAVES * e;
      if (piece < PIECES) {
        const uint4 *g = src + piece * kWave + lane;
        const uint32_t base = dst + (uint32_t)piece * (kWave * 16);
        // (M0 is written and used inside one statement)
        asm volatile("s_mov_b32 m0, %1\n\t"
                     "s_nop 0\n\t"
                     "global_load_lds_dwordx4 %0, off"
                     :
                     : "v"(g), "s"(base)
                     : "memory");
      }
    }
  };
  // a row's weight, and the start value of its chains (apart: the load is on
  // its way while a tile is searched)
  auto weight_of = [&](int c0, int c1, int t) {
    const int row = c0 + t * TR + tid;
    return tid < TR && row < c1 ? p.weight[row] : -2.0f;
  };
  // (in the first pass a large row that every query would have to look at is left
  // out: with a dozen of them the three minima that a query keeps were all
  // theirs, their distances gave the cut, and the second pass looked at every
  // row.  Norms of rows and queries log-normal with sigma 3, us a call: 100,000
  // x 4,096 x 64 2,778 / 723, 50,000 x 4,096 x 128 4,146 / 1,058, 100,000 x
  // 4,096 x 16 942 / 214)
  bool left_out = false;
  auto start_of = [&](float v, bool first) {
    float w = __builtin_fminf(v * s_c * s_c * kappa, 1e37f);
    // (negative ones compare as large ones; all waves wait for this)
    const bool special = __float_as_uint(v) > __float_as_uint(limit_sq);
    if (__any(special)) {
      // a large row: 0.24 r |a|^2 is at least B^2 / r, or a bound of none
      const float own = __builtin_fminf(v * large_gain, 1e37f);
      const float large = __builtin_fmaxf(
          (own >= large_loss ? own : 0.0f) - large_loss, -1e37f);
      const bool later =
          first && special && v >= 0.0f && own < large_loss;
      left_out = left_out || later;
      if (special)
        w = v >= 0.0f    ? (later ? kNfNothing : large)
            : v == -1.0f ? kNfAlways
                         : kNfNothing;
    }
    return w;
  };
  // `visit(step, s, v, acc)` for every 32 rows, set of queries and four rows
  auto scan = [&](int c0, int c1, bool first, auto &&visit)
                  __attribute__((always_inline)) {
    const int tiles = (c1 - c0 + TR - 1) / TR;
    __syncthreads(); // (nobody reads an earlier scan's tiles any more)
    request(c0, 0, 0);
    float w = weight_of(c0, c1, 0);
    if (tid < TR)
      tile_weight[0][tid] = start_of(w, first);
    for (int t = 0; t < tiles; ++t) {
      const int buf = t & 1;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (t + 1 < tiles) {
        w = weight_of(c0, c1, t + 1);
        request(c0, t + 1, buf ^ 1);
      }
#pragma unroll 1
      for (int i = 0; i < TR / 32; ++i) {
        const uint4 *arow = &tile_rows[buf][(i * 32 + col) * RSU + half];
        nf_f16x8_t a[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
          a[b] = __builtin_bit_cast(nf_f16x8_t, arow[2 * b]);
        nf_acc_t start;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float4 w4 = *reinterpret_cast<const float4 *>(
              &tile_weight[buf][i * 32 + 8 * v + 4 * half]);
          start[4 * v] = w4.x;
          start[4 * v + 1] = w4.y;
          start[4 * v + 2] = w4.z;
          start[4 * v + 3] = w4.w;
        }
        // the results of a set are looked at while the matrix cores work on
        // the next one, four values per matrix instruction or so
        nf_acc_t done = start;
#pragma unroll
        for (int s = 0; s <= S; ++s) {
          nf_acc_t acc = start;
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            if (s < S)
              acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                  a[b], yb[s < S ? s : 0][b], acc, 0, 0, 0);
            if (s > 0) {
#pragma unroll
              for (int v = 0; v < 4; ++v)
                if (v * NB / 4 == b)
                  visit(t * (TR / 32) + i, s - 1, v, done);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          done = acc;
        }
      }
      if (t + 1 < tiles && tid < TR)
        tile_weight[buf ^ 1][tid] = start_of(w, first);
    }
  };

  uint32_t keep_bits = ~kNfIndexMask; // (in a register)
  asm volatile("" : "+v"(keep_bits));
  float lowest = -__builtin_inff(); // (the compiler must not know)
  asm volatile("" : "+s"(lowest));
  unsigned long long scans = 0; // those with a third minimum below its cut
  float third[S];               // smallest third minimum of the scans
  bool any_left_out = false;
#pragma unroll
  for (int s = 0; s < S; ++s)
    third[s] = kNfNothing;
  for (int c0 = x_begin; c0 < x_end; c0 += kNfEpochRows) {
    const int c1 = min(x_end, c0 + kNfEpochRows);
    float top[S][3];
#pragma unroll
    for (int s = 0; s < S; ++s)
      top[s][0] = top[s][1] = top[s][2] = kNfNothing;
    scan(c0, c1, true, [&](int step, int s, int v, const nf_acc_t &acc)
                           __attribute__((always_inline)) {
      // (fmed3 with -inf is a minimum without the quieting of NaNs that fminf
      // comes with; it is also the instruction that waits for the matrix
      // cores, which the compiler sees to only for instructions of its own)
      float m = __builtin_amdgcn_fmed3f(acc[4 * v], acc[4 * v + 1], lowest);
      float t;
      asm("v_min3_f32 %0, %1, %2, %3"
          : "=v"(m)
          : "v"(m), "v"(acc[4 * v + 2]), "v"(acc[4 * v + 3]));
      asm("v_and_or_b32 %0, %1, %2, %3"
          : "=v"(t)
          : "v"(m), "v"(keep_bits), "s"(step * 4 + v));
      top[s][2] = __builtin_amdgcn_fmed3f(top[s][1], top[s][2], t);
      top[s][1] = __builtin_amdgcn_fmed3f(top[s][0], top[s][1], t);
      asm("v_min_f32 %0, %1, %2" : "=v"(top[s][0]) : "v"(top[s][0]), "v"(t));
    });

#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int q = q0 + s * 32;
      const float *row_y = p.y + (size_t)q * d;
      // first row of the four behind a kept value
      auto four_of = [&](float v, int h) {
        const int index = (int)(__float_as_uint(v) & kNfIndexMask);
        return c0 + (index >> 2) * 32 + (index & 3) * 8 + 4 * h;
      };
      const float other = __shfl_xor(top[s][0], 32);
      const int owner =
          half ? (other <= top[s][0] ? 0 : 1) : (top[s][0] <= other ? 0 : 1);
      const float least = owner == half ? top[s][0] : other;
      if (kind[s] == 1 && least <= cut[s]) {
        // two of the four rows per lane
        const int first = four_of(least, owner) + 2 * half;
        const int rows[2] = {min(first, c1 - 1), min(first + 1, c1 - 1)};
        float dist[2];
        nf_exact<2>(row_y, p.x, rows, d, dist);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          best[s] = min(best[s], nf_key(dist[i], rows[i] - x_begin));
      }
      best[s] = min(best[s], (unsigned long long)__shfl_xor(best[s], 32));
      if (kind[s] == 1) {
        const float kept = kept_cut(query_cut(best[s], ysq[s]));
        unsigned long long own = best[s];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          if (top[s][e] <= kept && !(e == 0 && owner == half)) {
#pragma unroll 1
            for (int i = 0; i < 4; ++i) {
              const int rows[1] = {four_of(top[s][e], half) + i};
              if (rows[0] < c1) {
                float dist[1];
                nf_exact<1>(row_y, p.x, rows, d, dist);
                own = min(own, nf_key(dist[0], rows[0] - x_begin));
              }
            }
          }
        }
        best[s] = own;
        if (top[s][2] <= kept)
          scans |= 1ull << min((c0 - x_begin) / kNfEpochRows, 63);
        third[s] = __builtin_fminf(third[s], top[s][2]);
      }
      // both lanes go on with the query's best row and a cut that follows it
      best[s] = min(best[s], (unsigned long long)__shfl_xor(best[s], 32));
      cut[s] = kind[s] == 1 ? kept_cut(query_cut(best[s], ysq[s])) : kNfCutLimit;
    }
    if (left_out)
      scans |= 1ull << min((c0 - x_begin) / kNfEpochRows, 63);
    any_left_out = any_left_out || left_out;
    left_out = false;
  }

  // ---- queries that may have rows that were not kept ------------------------
  // (a lane that doubts goes through its rows again, in scans some query of the
  // workgroup has doubted in; all of them where a row was left out)
  bool doubt = false;
  const bool everyone = __syncthreads_or(any_left_out) != 0;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const bool own = kind[s] == 1 && (everyone || third[s] <= cut[s]);
    cut[s] = own ? query_cut(best[s], ysq[s]) : -kNfCutLimit;
    doubt = doubt || own;
  }
  if (__syncthreads_or(doubt)) {
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1)
      scans |= (unsigned long long)__shfl_xor(scans, sh);
    if (lane == 0)
      wave_scans[wave] = scans;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      scans |= wave_scans[w];
    for (int c0 = x_begin; c0 < x_end; c0 += kNfEpochRows) {
      if (((scans >> min((c0 - x_begin) / kNfEpochRows, 63)) & 1) == 0)
        continue;
      const int c1 = min(x_end, c0 + kNfEpochRows);
      unsigned long long hits = 0; // 16 bits per set
      scan(c0, c1, false, [&](int step, int s, int v, const nf_acc_t &acc)
                              __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          hits |= acc[4 * v + i] <= cut[s] ? 1ull << (16 * s + 4 * v + i) : 0;
        if (s < S - 1 || v < 3)
          return;
        while (hits != 0) {
          const int at = __builtin_ctzll(hits);
          hits &= hits - 1;
          const int hit_s = at >> 4, hit_v = (at >> 2) & 3;
          const int rows[1] = {c0 + step * 32 + 8 * hit_v + 4 * half +
                               (at & 3)};
          if (rows[0] < c1) {
            float dist[1];
            nf_exact<1>(p.y + (size_t)(q0 + hit_s * 32) * d, p.x, rows, d,
                        dist);
            const unsigned long long key = nf_key(dist[0], rows[0] - x_begin);
#pragma unroll
            for (int u = 0; u < S; ++u)
              best[u] = u == hit_s ? min(best[u], key) : best[u];
          }
        }
      });
    }
  }
  // ---- queries searched exactly: all threads share out the rows --------------
  if (any_alone) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const uint32_t queries = (uint32_t)__ballot(kind[s] == 2);
      if (lane == 0)
        alone[wave][s] = queries;
    }
    __syncthreads();
    int turn = 0;
#pragma unroll 1
    for (int i = 0; i < WAVES * S; ++i) {
      const int w = i / S, s = i % S;
      uint32_t queries = alone[w][s];
      while (queries != 0) {
        const int at = __builtin_ctz(queries);
        queries &= queries - 1;
        const int q =
            q0 - (wave * (S * 32) + col) + w * (S * 32) + s * 32 + at;
        const float *row_y = p.y + (size_t)q * d;
        unsigned long long key = kNfNoKey;
#pragma unroll 1
        for (int r0 = x_begin + tid; r0 < x_end; r0 += 2 * kBlock) {
          const int rows[2] = {r0, min(r0 + kBlock, x_end - 1)};
          float dist[2];
          nf_exact<2>(row_y, p.x, rows, d, dist);
#pragma unroll
          for (int e = 0; e < 2; ++e)
            key = min(key, nf_key(dist[e], rows[e] - x_begin));
        }
#pragma unroll
        for (int sh = 1; sh < kWave; sh <<= 1)
          key = min(key, (unsigned long long)__shfl_xor(key, sh));
        if (lane == 0)
          wave_best[turn][wave] = key;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < WAVES; ++u)
          key = min(key, wave_best[turn][u]);
        turn ^= 1;
#pragma unroll
        for (int u = 0; u < S; ++u)
          if (u == s && w == wave && col == at)
            best[u] = min(best[u], key);
      }
    }
  }

#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int q = q0 + s * 32;
    best[s] = min(best[s], (unsigned long long)__shfl_xor(best[s], 32));
    if (half == 0 && q < y_end)
      p.out[q] = best[s] != kNfNoKey
                     ? (int64_t)x_begin +
                           (int64_t)nearest_rel((uint32_t)best[s])
                     : 0;
  }
}

// |x|^2 of every row (or what it is instead, see NearestFeatParams), and the
// largest component and the sum of log2 |x|^2 over the moderate rows.
__global__ __launch_bounds__(kBlock) void nearest_feat_rows_kernel(
    const float *__restrict__ x, int n, int d, float *__restrict__ weight,
    NearestFeatGlobals *__restrict__ globals);

// The fp16 operands of the rows, one thread per unit of 8 components; zeros
// for rows the filter does not represent or that are far larger than the
// others, and for a tile of rows behind the last one.
template <int NB>
__global__ __launch_bounds__(kBlock) void nearest_feat_pack_kernel(
    const float *__restrict__ x, int n, int d,
    const float *__restrict__ weight,
    NearestFeatGlobals *globals, uint4 *__restrict__ pack) {
  constexpr int U = 2 * NB;
  const size_t id = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (id >= (size_t)(n + kNfTileRows) * U)
    return;
  const int row = (int)(id / U);
  const int unit = (int)(id - (size_t)row * U);
  uint4 out = make_uint4(0, 0, 0, 0);
  const NfRows rows = nf_rows(globals);
  if (id == 0)
    globals->rows_of_x = rows;
  if (row < n && weight[row] >= 0.0f && weight[row] <= rows.limit_sq) {
    const float scale = rows.scale;
    float v[8];
    nf_load8(x + (size_t)row * d, 8 * unit, d, v);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] *= scale;
    out = nf_pack8(v);
  }
  pack[(size_t)row * (U + 1) + unit] = out;
}

// One number of component blocks (two per translation unit).
template <int NB>
hipError_t launch_nearest_feat_blocks(const NearestFeatParams &p, int sets,
                                      int grid, hipStream_t stream);
// Sets of 32 queries per wave: as many as the registers hold.
constexpr int nearest_feat_sets(int nb) { return nb <= 4 ? 4 : nb <= 6 ? 3 : 2; }

#define PCA_NEAREST_FEAT_DEFINE(NB_)                                           \
  template <>                                                                  \
  hipError_t launch_nearest_feat_blocks<NB_>(const NearestFeatParams &p,       \
                                             int sets, int grid,               \
                                             hipStream_t stream) {             \
    const size_t units = ((size_t)p.n + kNfTileRows) * (2 * NB_);              \
    hipLaunchKernelGGL((nearest_feat_pack_kernel<NB_>),                        \
                       dim3((unsigned)((units + kBlock - 1) / kBlock)),        \
                       dim3(kBlock), 0, stream, p.x, p.n, p.d, p.weight,       \
                       const_cast<NearestFeatGlobals *>(p.globals),            \
                       const_cast<uint4 *>(p.pack));                           \
    if (sets == 1)                                                             \
      hipLaunchKernelGGL((nearest_feat_kernel<NB_, 1>), dim3(grid),            \
                         dim3(kBlock), 0, stream, p);                          \
    else                                                                       \
      hipLaunchKernelGGL((nearest_feat_kernel<NB_, nearest_feat_sets(NB_)>),   \
                         dim3(grid), dim3(kBlock), 0, stream, p);              \
    return hipGetLastError();                                                  \
  }

} // namespace pca
