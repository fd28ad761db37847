// Farthest point sampling: the `fps` operator of the reference
// (csrc/cuda/fps_cuda.cu:10-66, fps_kernel), an example by one workgroup of up to
// 1,024 threads or by several of 1,024.
//
// What the reference computes, and what is reproduced bit for bit: the first
// sample of an example is its start row; every further sample is the row with
// the largest running minimum distance to the samples so far, where
//   * distances are squared, accumulated with one fused multiply-add per
//     dimension (`dd += tmp * tmp`; every operator rounds to 16 bits for
//     fp16), and the running minimum starts at 5e4 for every row (the `dist`
//     array of the host wrapper, :91) -- larger distances count as 5e4;
//   * among rows of equal value the reference's block of 256 threads returns
//     the one with the smallest (row - start) % 256, then the smallest row:
//     thread t scans rows start + t, start + t + 256, ... and keeps its first
//     strict maximum (:35-47), the reduction keeps the lower thread on ties
//     (:52-59, read as lock-step rounds);
//   * `best` starts at -1 and `best_idx` at 0: when no row has a value above
//     -1 (every distance NaN) the sample is row 0.
//
// The sampling is a chain of dependent steps, each an arg-max over the example's
// rows, so the time per sample is what counts.  Who samples (fp32; the caller's bound
// on the rows of an example decides, which for the operators is that of
// torch_ops.cpp::fps_bound):
//   * fps_reg_kernel, up to 256 rows of up to 4 dimensions and up to 1,024 in calls of
//     more than 256 examples: every row in every step, from registers.  So do all
//     others where few samples are wanted (fps_few, fps_bound).
//   * Beyond that most rows are left alone (see "rows in buckets" below).
//     fps_own_kernel, up to 8,192 rows of up to 4 dimensions: one workgroup, several
//     samples per step ("a wave's own stretch of the curve").
//   * fps_bucket_kernel, up to 16,384 rows of up to 4 dimensions by such a bound: one
//     workgroup, one sample per step.
//   * fps_shared_kernel, up to 524,288 rows of up to 3 dimensions in calls of up to 64
//     examples: several workgroups, several samples per step ("the same, an example by
//     several workgroups").  What they tell each other takes 1.1 us of a step.  Any
//     bound above 16,384 leads here, for the operators also examples of 8,193 - 16,384
//     rows from 170 (220) samples on and of 4,097 - 8,192 from 1,100 (1,600) on.
//   * fps_stream_kernel, any number of rows of up to 3 dimensions: one workgroup,
//     several samples per step ("several samples per step").
//   * fps_any_kernel, any size, dimension and element type: rows and a `dist` array
//     stream from memory.
#include "device_utils.hpp"
#include "launchers.hpp"

#include <algorithm>
#include <type_traits>

#include <hip/hip_fp16.h>

namespace pca {

namespace {

constexpr int kFpsThreads = 1024;
constexpr int kFpsWaves = kFpsThreads / kWave;
constexpr uint32_t kFpsNoTie = 0xffffffffu;

// Order among equal values: (row - start) % 256 first, then the row
__device__ __forceinline__ uint32_t fps_tie(uint32_t rel) {
  return ((rel & 255u) << 24) | (rel >> 8);
}
__device__ __forceinline__ uint32_t fps_rel(uint32_t tie) {
  return ((tie & 0xffffffu) << 8) | (tie >> 24);
}

// (value, tie) a beats b
template <typename T>
__device__ __forceinline__ bool fps_better(T ad, uint32_t at, T bd,
                                           uint32_t bt) {
  return ad > bd || (ad == bd && at < bt);
}

__device__ __forceinline__ float shfl_xor_t(float v, int m) {
  return __shfl_xor(v, m);
}
__device__ __forceinline__ double shfl_xor_t(double v, int m) {
  return __shfl_xor(v, m);
}

// Largest value of a wave / of every row of 16 lanes, by data-parallel
// primitives (one fused shift-and-max instruction per step; lanes without a
// source take 0, the smallest value).  The wave's result is uniform.
#define PCA_DPP_UMAX(v, ctrl, rows)                                            \
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(v), ctrl, rows,    \
                                                   0xf, false))
__device__ __forceinline__ uint32_t row16_umax(uint32_t v) {
  PCA_DPP_UMAX(v, 0x111, 0xf); // row_shr:1
  PCA_DPP_UMAX(v, 0x112, 0xf); // row_shr:2
  PCA_DPP_UMAX(v, 0x114, 0xf); // row_shr:4
  PCA_DPP_UMAX(v, 0x118, 0xf); // row_shr:8
  return v; // lane 15 of every row holds the row's maximum
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
  v = row16_umax(v);
  PCA_DPP_UMAX(v, 0x142, 0xa); // row_bcast:15 into rows 1 and 3
  PCA_DPP_UMAX(v, 0x143, 0xc); // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Every lane gets the largest value of its row of 16 lanes.
__device__ __forceinline__ uint32_t row16_umax_all(uint32_t v) {
  PCA_DPP_UMAX(v, 0x128, 0xf); // row_ror:8
  PCA_DPP_UMAX(v, 0x124, 0xf); // row_ror:4
  PCA_DPP_UMAX(v, 0x122, 0xf); // row_ror:2
  PCA_DPP_UMAX(v, 0x121, 0xf); // row_ror:1
  return v;
}
// Every lane gets the sum of its eight.
__device__ __forceinline__ uint32_t row8_sum(uint32_t v) {
#define PCA_DPP_ADD(ctrl)                                                      \
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xf, 0xf, false)
  PCA_DPP_ADD(0xb1);  // quad_perm 1,0,3,2
  PCA_DPP_ADD(0x4e);  // quad_perm 2,3,0,1
  PCA_DPP_ADD(0x141); // row_half_mirror
#undef PCA_DPP_ADD
  return v;
}
// U waves' worth of values at once: their steps fill each other's wait states.
template <int U> __device__ __forceinline__ void wave_umax_of(uint32_t (&v)[U]) {
#define PCA_DPP_EACH(ctrl, rows)                                               \
  _Pragma("unroll") for (int u = 0; u < U; ++u) PCA_DPP_UMAX(v[u], ctrl, rows)
  PCA_DPP_EACH(0x111, 0xf);
  PCA_DPP_EACH(0x112, 0xf);
  PCA_DPP_EACH(0x114, 0xf);
  PCA_DPP_EACH(0x118, 0xf);
  PCA_DPP_EACH(0x142, 0xa);
  PCA_DPP_EACH(0x143, 0xc);
#undef PCA_DPP_EACH
#pragma unroll
  for (int u = 0; u < U; ++u)
    v[u] = (uint32_t)__builtin_amdgcn_readlane((int)v[u], 63);
}
#undef PCA_DPP_UMAX
// Largest number of a wave, of numbers that are not NaN.
__device__ __forceinline__ float wave_fmax(float v) {
  const uint32_t u = __float_as_uint(v);
  const uint32_t top =
      wave_umax((int)u < 0 ? ~u : u | 0x80000000u); // (ordered like v)
  return __uint_as_float((int)top < 0 ? top & 0x7fffffffu : ~top);
}

// ---- element types ----------------------------------------------------------

struct FpsF32 {
  typedef float store_t;
  typedef float calc_t;
  static __device__ __forceinline__ calc_t load(store_t v) { return v; }
  static __device__ __forceinline__ calc_t step(calc_t a, calc_t b,
                                                calc_t acc) {
    const calc_t t = a - b;
    return __builtin_fmaf(t, t, acc);
  }
  static __device__ __forceinline__ calc_t lower(calc_t a, calc_t b) {
    return __builtin_fminf(a, b);
  }
  static __device__ __forceinline__ calc_t limit() { return 5e4f; }
};

struct FpsF64 {
  typedef double store_t;
  typedef double calc_t;
  static __device__ __forceinline__ calc_t load(store_t v) { return v; }
  static __device__ __forceinline__ calc_t step(calc_t a, calc_t b,
                                                calc_t acc) {
    const calc_t t = a - b;
    return __builtin_fma(t, t, acc);
  }
  static __device__ __forceinline__ calc_t lower(calc_t a, calc_t b) {
    return __builtin_fmin(a, b);
  }
  static __device__ __forceinline__ calc_t limit() { return 5e4; }
};

// c10::Half arithmetic: every operator computes in float and rounds to 16
// bits; values travel as floats that are representable halves
struct FpsF16 {
  typedef uint16_t store_t;
  typedef float calc_t;
  static __device__ __forceinline__ float r16(float v) {
    return __half2float(__float2half_rn(v));
  }
  static __device__ __forceinline__ calc_t load(store_t v) {
    return __half2float(__ushort_as_half(v));
  }
  static __device__ __forceinline__ calc_t step(calc_t a, calc_t b,
                                                calc_t acc) {
    const float t = r16(a - b);
    const float p = r16(t * t);
    return r16(acc + p);
  }
  static __device__ __forceinline__ calc_t lower(calc_t a, calc_t b) {
    return __builtin_fminf(a, b);
  }
  static __device__ __forceinline__ calc_t limit() { return r16(5e4f); }
};

// ---- any size, dimension and element type -------------------------------------

// dist: [n] running minima (initialised here); one workgroup per example.
template <typename Tr>
__global__ __launch_bounds__(kFpsThreads) void fps_any_kernel(
    const typename Tr::store_t *__restrict__ src,
    const int64_t *__restrict__ ptr, const int64_t *__restrict__ out_ptr,
    const int64_t *__restrict__ start, int d,
    typename Tr::calc_t *__restrict__ dist, int64_t *__restrict__ out) {
  typedef typename Tr::calc_t calc_t;
  __shared__ calc_t s_d[2][kFpsWaves];
  __shared__ uint32_t s_t[2][kFpsWaves];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int b = blockIdx.x;
  const int64_t start_idx = ptr[b];
  const int64_t end_idx = ptr[b + 1];
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end)
    return;

  for (int64_t n = start_idx + tid; n < end_idx; n += kFpsThreads)
    dist[n] = Tr::limit();
  int64_t old = start_idx + (start ? start[b] : 0);
  if (tid == 0)
    out[o_begin] = old;

  for (int64_t m = o_begin + 1; m < o_end; ++m) {
    const int par = (int)(m & 1);
    const typename Tr::store_t *cur = src + (size_t)old * d;
    calc_t best = (calc_t)-1;
    uint32_t best_tie = kFpsNoTie;
    // a thread's rows share (row - start) % 256, so its first strict
    // maximum is its best by the tie rule as well
    for (int64_t n = start_idx + tid; n < end_idx; n += kFpsThreads) {
      const typename Tr::store_t *row = src + (size_t)n * d;
      calc_t dd = 0;
      for (int c = 0; c < d; ++c)
        dd = Tr::step(Tr::load(cur[c]), Tr::load(row[c]), dd);
      dd = Tr::lower(dist[n], dd);
      dist[n] = dd;
      if (dd > best) {
        best = dd;
        best_tie = fps_tie((uint32_t)(n - start_idx));
      }
    }
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      const calc_t od = shfl_xor_t(best, sh);
      const uint32_t ot = __shfl_xor(best_tie, sh);
      if (fps_better(od, ot, best, best_tie)) {
        best = od;
        best_tie = ot;
      }
    }
    if (lane == 0) {
      s_d[par][wave] = best;
      s_t[par][wave] = best_tie;
    }
    __syncthreads();
    best = s_d[par][0];
    best_tie = s_t[par][0];
#pragma unroll
    for (int w = 1; w < kFpsWaves; ++w) {
      const calc_t od = s_d[par][w];
      const uint32_t ot = s_t[par][w];
      if (fps_better(od, ot, best, best_tie)) {
        best = od;
        best_tie = ot;
      }
    }
    // nothing above -1: the reference's `best_idx` is still 0
    old = best_tie != kFpsNoTie ? start_idx + (int64_t)fps_rel(best_tie) : 0;
    if (tid == 0)
      out[m] = old;
  }
}

// ---- fp32, up to 4 dimensions: every row in every step -------------------------

// T threads hold P rows each.  With T = 256 S, thread t has the rows
// t / S + 256 * ((t % S) * P + i), i < P, of its example; a single wave
// (T = 64) gives thread t the rows 4 t + i / (P / 4) + 256 * (i % (P / 4)).
// Among equal values the reference's order is "(row - start) % 256, then the
// row", which in these layouts reads "t, then i": the first thread wins, and
// inside it the first slot.  Every "first of the equal ones" is therefore a
// count of trailing zeros of a ballot, and only the values themselves go
// through a reduction.  A step costs every wave the same few dozen
// instructions of reduction and hand-over on top of its 8 P of distances,
// and the waves of a SIMD take turns: the launcher picks the shape that
// measured fastest for the row count.  The single wave needs neither the
// hand-over through shared memory nor a barrier.
template <int DIM, int P, int T>
__device__ __forceinline__ void fps_every_row(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int64_t *__restrict__ out) {
  // per wave and parity: value (as an ordered unsigned number,
  // 0 = none), row (relative to the example) and coordinates of the wave's best
  __shared__ uint32_t s_v[2][kFpsWaves];
  __shared__ uint32_t s_rel[2][kFpsWaves];
  __shared__ float s_x[2][DIM][kFpsWaves];
  static_assert(kFpsWaves == 16 && (T % 256 == 0 || T == kWave) &&
                    T <= kFpsThreads,
                "one row of 16 lanes picks the winner among up to 16 waves");
  static_assert(T != kWave || P % 4 == 0, "four tie classes per lane");

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  constexpr int S = T >= 256 ? T / 256 : 1; // threads per tie class
  constexpr int C = T >= 256 ? 1 : 256 / T; // tie classes per thread
  constexpr int PARTS = P / C;              // slots per tie class
  const int rel0 = (tid / S) * C + 256 * ((tid % S) * P);
  // row of slot i, relative to rel0
  auto slot_row = [](int i) { return i / PARTS + 256 * (i % PARTS); };
  const int b = blockIdx.x;
  const int64_t start_idx = ptr[b];
  const int count = (int)(ptr[b + 1] - start_idx);
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end)
    return;
  if (T < kFpsThreads && T > kWave) {
    // the entries of waves that do not run stay "nothing"
    if (tid < 2 * kFpsWaves)
      s_v[tid / kFpsWaves][tid % kFpsWaves] = 0u;
    __syncthreads();
  }

  float px[P][DIM];
  // A slot's running minimum is the high word of a 64-bit pattern whose low
  // word is 15 - i.  Minima are -1 (no row) or in [0, 5e4]: read as doubles,
  // the patterns of rows order by minimum first and smaller slot second, and
  // none is a NaN or an infinity, so one 64-bit maximum per slot tracks the
  // thread's best (the first of its largest minima) and where it is.
  double slot_key[P];
  static_assert(P <= 16, "low words 15 - i");
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int rel = rel0 + slot_row(i);
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      px[i][c] = (rel < count && c < d)
                     ? src[(size_t)(start_idx + rel) * d + c]
                     : 0.0f;
    slot_key[i] = __hiloint2double(
        __float_as_int(rel < count ? 5e4f : -1.0f), 15 - i);
  }
  const int64_t first = start_idx + (start ? start[b] : 0);
  if (tid == 0)
    out[o_begin] = first;
  float cur[DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c)
    cur[c] = c < d ? src[(size_t)first * d + c] : 0.0f;

  for (int64_t m = o_begin + 1; m < o_end; ++m) {
    const int par = (int)(m & 1);
    // (below every slot's pattern: -1 with the largest low word)
    double best_key = __hiloint2double(__float_as_int(-1.0f), -1);
    // (component by component over all slots: independent instructions
    // follow each other, a slot's own chain is spread out)
    float dd[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const float t0 = cur[0] - px[i][0];
      dd[i] = t0 * t0;
    }
#pragma unroll
    for (int c = 1; c < DIM; ++c) {
#pragma unroll
      for (int i = 0; i < P; ++i) {
        // (zero components beyond d add fma(0, 0, acc) = acc)
        const float tc = cur[c] - px[i][c];
        dd[i] = __builtin_fmaf(tc, tc, dd[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      // fminf without its quieting of signalling NaNs, which neither operand
      // can be (5e4, -1, or the result of arithmetic): a NaN loses to a number
      const float before = __int_as_float(__double2hiint(slot_key[i]));
      asm("v_min_f32 %0, %1, %2" : "=v"(dd[i]) : "v"(before), "v"(dd[i]));
      slot_key[i] = __hiloint2double(__float_as_int(dd[i]),
                                     __double2loint(slot_key[i]));
    }
    double part_key[2] = {best_key, best_key};
#pragma unroll
    for (int i = 0; i < P; ++i)
      asm("v_max_f64 %0, %1, %2"
          : "=v"(part_key[i & 1])
          : "v"(part_key[i & 1]), "v"(slot_key[i]));
    asm("v_max_f64 %0, %1, %2"
        : "=v"(best_key)
        : "v"(part_key[0]), "v"(part_key[1]));
    const uint32_t best_bits = (uint32_t)__double2hiint(best_key);
    const int best_i = best_bits != __float_as_uint(-1.0f)
                           ? 15 - __double2loint(best_key)
                           : -1;
    // values are -1 (nothing) or >= 0: their bit patterns, with the top bit
    // set, order like the values
    const uint32_t key = best_i >= 0 ? (best_bits | 0x80000000u) : 0u;
    const uint32_t wave_key = wave_umax(key);
    const int src_lane = (int)__builtin_ctzll(__ballot(key == wave_key));
    // which of its rows that lane means: a uniform number, so every lane
    // picks that slot of its own registers with scalar branches (no per-row
    // bookkeeping of coordinates in the loop above)
    const int slot = __builtin_amdgcn_readlane(best_i, src_lane);
    float bx[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      bx[c] = 0.0f;
    switch (slot) {
#define PCA_FPS_SLOT(i_)                                                       \
  case i_:                                                                     \
    if (i_ < P) {                                                              \
      _Pragma("unroll") for (int c = 0; c < DIM; ++c) bx[c] =                  \
          px[i_ < P ? i_ : 0][c];                                              \
    }                                                                          \
    break;
      PCA_FPS_SLOT(0) PCA_FPS_SLOT(1) PCA_FPS_SLOT(2) PCA_FPS_SLOT(3)
      PCA_FPS_SLOT(4) PCA_FPS_SLOT(5) PCA_FPS_SLOT(6) PCA_FPS_SLOT(7)
      PCA_FPS_SLOT(8) PCA_FPS_SLOT(9) PCA_FPS_SLOT(10) PCA_FPS_SLOT(11)
      PCA_FPS_SLOT(12) PCA_FPS_SLOT(13) PCA_FPS_SLOT(14) PCA_FPS_SLOT(15)
#undef PCA_FPS_SLOT
    default:
      break;
    }
    static_assert(P <= 16, "slots of the switch above");
    int64_t chosen;
    if (T == kWave) {
      if (wave_key != 0u) {
        chosen = start_idx + __builtin_amdgcn_readlane(rel0, src_lane) +
                 slot_row(slot);
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          cur[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
              (int)__float_as_uint(bx[c]), src_lane));
      } else {
        // nothing above -1: the reference's `best_idx` is still 0
        chosen = 0;
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          cur[c] = c < d ? src[c] : 0.0f;
      }
    } else {
      if (lane == src_lane) {
        s_v[par][wave] = wave_key;
        s_rel[par][wave] = (uint32_t)(rel0 + slot_row(slot));
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          s_x[par][c][wave] = bx[c];
      }
      __syncthreads();
      // every row of 16 lanes looks at the 16 wave results
      const uint32_t ev = s_v[par][lane & 15];
      const uint32_t erel = s_rel[par][lane & 15];
      float ex[DIM];
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        ex[c] = s_x[par][c][lane & 15];
        asm volatile("" : "+v"(ex[c])); // (read now, not after the reduction)
      }
      const uint32_t top_key =
          (uint32_t)__builtin_amdgcn_readlane((int)row16_umax(ev), 15);
      if (top_key != 0u) {
        const int win = (int)__builtin_ctzll(__ballot(ev == top_key));
        chosen =
            start_idx + (int64_t)__builtin_amdgcn_readlane((int)erel, win);
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          cur[c] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
              (int)__float_as_uint(ex[c]), win));
      } else {
        // nothing above -1: the reference's `best_idx` is still 0
        chosen = 0;
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          cur[c] = c < d ? src[c] : 0.0f;
      }
    }
    if (tid == 0)
      out[m] = chosen;
    // (in vector registers: the distance code then interleaves its rows)
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      asm volatile("" : "+v"(cur[c]));
  }
}

template <int DIM, int P, int T>
__global__ __launch_bounds__(T) void fps_reg_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int64_t *__restrict__ out) {
  fps_every_row<DIM, P, T>(src, ptr, out_ptr, start, d, out);
}

// ---- fp32, up to 4 dimensions: rows in buckets, most of them left alone -------
//
// A new sample lowers the running minimum only of rows nearer to it than the
// samples before it, so most rows of an example need no distance at all (a
// published method: M. Han et al., QuickFPS, bucket-based sampling, 2023).  The
// rows are ordered along a space-filling curve and cut into buckets of 64
// (one row per lane); the wave that owns a bucket keeps, in one lane of its
// registers, the bucket's box, its largest running minimum and the row that
// has it.  Per sample a lane tests its bucket: if the distance from the sample
// to the box -- formed with the operations of the exact chain on per-axis gaps
// no larger than any row's difference, hence, rounding being monotone, not
// above the COMPUTED distance of any of its rows -- is not below the bucket's
// largest minimum, no minimum of the bucket changes and it is skipped;
// otherwise the whole wave goes through its 64 rows.  Same values, and so the
// same samples, as looking at every row.
//
// What bounds it: the chain of one step (arg-max over the buckets, box test,
// one bucket, hand-over through LDS, one barrier), not the rows.  Buckets go
// round-robin to the waves, so that the few neighbouring ones a sample
// touches are looked at side by side.

constexpr uint32_t kFpsNoRow = 0xffffffffu; // its tie is the largest one
// Largest minimum of a bucket before the first sample: a NaN, which no distance
// is at or above, so that every bucket with rows is looked at and gets the
// value of its rows (5e4 or less) there.  Against infinity a bucket at an
// infinite distance -- rows without a finite coordinate on some axis, a first
// sample with an infinite one, squared gaps beyond fp32 -- would be left alone
// and keep the infinity.
constexpr uint32_t kFpsUnseen = 0x7fc00000u;

// What a wave hands over: the largest running minimum (bits of a float that
// is not negative), the row that has it, and that row's coordinates.
template <int DIM> struct FpsBest {
  uint32_t val, rel;
  float x[DIM];
};

// Of the lanes in `who` (equal values) the one whose row comes first in the
// reference's order; the lanes of `who` hold it in `rel`.
__device__ __forceinline__ int fps_first(uint64_t who, uint32_t rel) {
  if (__builtin_expect((who & (who - 1)) != 0, 0)) {
    const int lane = threadIdx.x & (kWave - 1);
    // (formed here: outside the loop it would take a register per bucket)
    asm volatile("" : "+v"(rel));
    // (umax of the complement: the smallest tie; lanes outside take 0)
    const uint32_t t = (who >> lane) & 1 ? ~fps_tie(rel) : 0u;
    const uint32_t top = wave_umax(t);
    who &= __ballot(t == top);
  }
  return (int)__builtin_ctzll(who);
}

// A lane's value, uniform.  (In a scalar register right here: moved into a
// branch that only some lanes take, the read would see the registers as those
// lanes left them.)
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int lane) {
  int s = __builtin_amdgcn_readlane((int)v, lane);
  asm volatile("" : "+s"(s));
  return (uint32_t)s;
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float(lane_value(__float_as_uint(v), lane));
}

// Lower bound of the chain's distance from a sample to any row of a box.
template <int DIM>
__device__ __forceinline__ float fps_box_distance(const float (&q)[DIM],
                                                  const float (&lo)[DIM],
                                                  const float (&hi)[DIM]) {
  float dd = 0.0f;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    // (a NaN in the sample leaves a gap of 0: the bucket is looked at)
    const float gap = __builtin_fmaxf(
        __builtin_fmaxf(lo[c] - q[c], q[c] - hi[c]), 0.0f);
    dd = c == 0 ? gap * gap : __builtin_fmaf(gap, gap, dd);
  }
  return dd;
}

// Distance of a row to the sample, and the row's running minimum with it.
template <int DIM>
__device__ __forceinline__ float fps_lower(const float (&q)[DIM],
                                           const float (&x)[DIM], float m) {
  float dd = 0.0f;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    // (zero components beyond d add fma(0, 0, acc) = acc)
    const float t = q[c] - x[c];
    dd = c == 0 ? t * t : __builtin_fmaf(t, t, dd);
  }
  // a NaN loses to a number, as in fminf; `m` is never a NaN
  asm("v_min_f32 %0, %1, %2" : "=v"(dd) : "v"(m), "v"(dd));
  return dd;
}

// ---- several samples per step ---------------------------------------------------
//
// The rows of an example are in 64 groups; of each group an entry of a table in
// LDS has the largest running minimum, the row that has it (its number and
// its coordinates), and `rest`, no smaller than any other minimum of
// the group.  The next sample is the entry that comes first (largest value, equal
// ones in the reference's order).  A sample lowers minima only: while an entry's
// row is at least its value away from all samples of the step before it, it
// still has that value and is still the first of its group; and while it comes
// before the `rest` of those samples' groups, no other row can be before it.
// So the entries are ranked, and the samples of a step are the longest run of
// first ones of which that holds for every pair -- the same samples, in the same
// order, as one by one.  (A sample that does not lower its own minimum -- a row
// without a finite distance to itself, or a minimum of 0 -- is the next sample
// again: the run ends with it.)
constexpr int kFpsRun = 8; // at most; 8 x 8 pairs are a wave's lanes

struct FpsTable {
  float4 head[kWave];      // value, row, first two coordinates
  float4 tail[kWave];      // the other coordinates, rest, its tie
  float4 first[kFpsRun]; // of rank i: value, coordinates
  float4 more[kFpsRun];  // fourth coordinate, rest, row, tie of rest
};
// Among rows of the value `rest` of a group the complement of the smallest tie;
// where nobody looked for it, a number that is before all others.
constexpr uint32_t kFpsAnyTie = 0xffffffffu;
template <int DIM>
__device__ __forceinline__ void
fps_enter(FpsTable &t, int group, uint32_t val, uint32_t row,
          const float (&x)[DIM], uint32_t rest, uint32_t rest_tie) {
  t.head[group] = make_float4(__uint_as_float(val), __uint_as_float(row), x[0],
                              DIM > 1 ? x[DIM > 1 ? 1 : 0] : 0.0f);
  t.tail[group] = make_float4(DIM > 2 ? x[DIM > 2 ? 2 : 0] : 0.0f,
                              DIM > 3 ? x[DIM > 3 ? 3 : 0] : 0.0f,
                              __uint_as_float(rest),
                              __uint_as_float(rest_tie));
}

// Waits for this workgroup's LDS traffic and meets its other waves (global
// stores stay in flight: for them __syncthreads).
__device__ __forceinline__ void fps_meet() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Entries to samples, by a workgroup of 64 / OWN waves, after the entries of
// this step are written; wave w ranks entries OWN w ...  Returns the number of
// samples, the same for all waves; lane i % 8 holds the i-th: coordinates and
// `row`.  `rel`: from an entry's row to its number in the example.
template <int OWN, int DIM, typename Rel>
__device__ __forceinline__ int fps_rank(FpsTable &t, int wave, Rel rel,
                                        float (&sx)[DIM], uint32_t &row) {
  const int lane = threadIdx.x & (kWave - 1);
  fps_meet();
  const uint32_t v = __float_as_uint(t.head[lane].x);
  const int own = wave * OWN + (lane & (OWN - 1));
  const float4 h = t.head[own];
  const float4 g = t.tail[own];
  int before[OWN], equal = 0;
#pragma unroll
  for (int e = 0; e < OWN; ++e) {
    const uint32_t mine = lane_value(v, wave * OWN + e);
    before[e] = __builtin_popcountll(__ballot(v > mine));
    equal += __builtin_popcountll(__ballot(v >= mine)) - before[e];
  }
  if (__builtin_expect(equal != OWN, 0)) {
    const uint32_t tie = fps_tie(rel(__float_as_uint(t.head[lane].y)));
#pragma unroll
    for (int e = 0; e < OWN; ++e) {
      const uint32_t mine = lane_value(v, wave * OWN + e);
      const uint32_t mine_tie = lane_value(tie, wave * OWN + e);
      before[e] += __builtin_popcountll(
          __ballot(v == mine && (tie < mine_tie ||
                                 (tie == mine_tie && lane < wave * OWN + e))));
    }
  }
  int rank = before[0];
#pragma unroll
  for (int e = 1; e < OWN; ++e)
    rank = (lane & (OWN - 1)) == e ? before[e] : rank;
  if (lane < OWN && rank < kFpsRun) {
    t.first[rank] = make_float4(h.x, h.z, h.w, g.x);
    t.more[rank] = make_float4(g.y, g.z, h.y, g.w);
  }
  fps_meet();
  const int a = lane & (kFpsRun - 1), b = lane / kFpsRun;
  const float4 ra = t.first[a], rb = t.first[b];
  const float4 ma = t.more[a];
  const float xa[4] = {ra.y, ra.z, ra.w, ma.x};
  const float xb[4] = {rb.y, rb.z, rb.w, DIM > 3 ? t.more[b].x : 0.0f};
  float dd = 0.0f;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    const float df = xa[c] - xb[c];
    dd = c == 0 ? df * df : __builtin_fmaf(df, df, dd);
    sx[c] = xa[c];
  }
  row = __float_as_uint(ma.z);
  // (infinite: one of the two has no distance to itself; 0: nor is a minimum of 0
  // lowered by its own sample)
  bool apart = dd >= rb.x && dd < __builtin_inff() && ma.y <= rb.x &&
               rb.x > 0.0f;
  const bool equal_rest = a < b && apart && ma.y == rb.x;
  if (__builtin_expect(__ballot(equal_rest) != 0, 0)) {
    // the next row of that group comes after this one
    const uint32_t tie = ~fps_tie(rel(__float_as_uint(t.more[b].z)));
    apart = apart && (!equal_rest || __float_as_uint(ma.w) < tie);
  }
  const uint64_t ends = __ballot(a < b && !apart);
  return ends != 0 ? (int)__builtin_ctzll(ends) / kFpsRun : kFpsRun;
}

// The rows of an example in curve order, by a workgroup of 16 waves: afterwards
// keys[i], i < count, holds the i-th row's number (relative to the example) in its
// REL_BITS low bits, above them its cell of the example's box (6 bits per axis).
//
// Two passes of 9 bits, the keys in registers between them.  A pass counts every
// wave's digits in LDS (two waves to a word: 16 bits each, of at most 16,384 rows),
// turns the counts into places, digit by digit and wave by wave, and writes the keys
// there.  A wave owns a run of places, so a pass keeps the order of the one
// before as far as the counters hand out places lane by lane; where they do not,
// rows of one cell of the curve's upper 9 bits lie in another order, which no
// sample depends on.  4,096 rows, until the first step: 41 us with a bitonic sort of
// the LDS, 16 now, most of it the cells of the rows and their way from memory.
constexpr int kFpsDigits = 512;
struct FpsSort {
  uint32_t count[kFpsWaves / 2][kFpsDigits];
  float part[2 * 3][kFpsWaves];
  uint32_t total[kFpsWaves];
};
template <int DIM, int REL_BITS, int CAP>
__device__ __forceinline__ void
fps_curve_order(const float *__restrict__ rows, int count, int d,
                uint32_t *keys, FpsSort &t) {
  constexpr int W = kFpsWaves;
  constexpr int PER = CAP / kFpsThreads;
  constexpr int AXIS_BITS = 6;
  static_assert(3 * AXIS_BITS + REL_BITS <= 32 && (1 << REL_BITS) >= CAP,
                "row and place in a word");
  static_assert((1 << 3 * AXIS_BITS) == kFpsDigits * kFpsDigits, "two digits");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // (a wave's rows follow each other)
  const int first = wave * (kWave * PER) + lane;
  float v[PER][3], lo[3], hi[3];
#pragma unroll
  for (int i = 0; i < PER; ++i)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      v[i][c] = first + i * kWave < count && c < DIM && c < d
                    ? rows[(size_t)(first + i * kWave) * d + c]
                    : 0.0f;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    lo[c] = hi[c] = 0.0f;
    if (c < DIM) {
      lo[c] = __builtin_inff();
      hi[c] = -__builtin_inff();
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (first + i * kWave < count &&
            __builtin_fabsf(v[i][c]) < __builtin_inff()) {
          lo[c] = __builtin_fminf(lo[c], v[i][c]);
          hi[c] = __builtin_fmaxf(hi[c], v[i][c]);
        }
      lo[c] = -wave_fmax(-lo[c]);
      hi[c] = wave_fmax(hi[c]);
      if (lane == 0) {
        t.part[c][wave] = lo[c];
        t.part[3 + c][wave] = hi[c];
      }
    }
  }
  auto clear = [&]() {
    for (int i = tid; i < W / 2 * kFpsDigits; i += kFpsThreads)
      (&t.count[0][0])[i] = 0u;
  };
  clear();
  __syncthreads();
#pragma unroll
  for (int c = 0; c < DIM && c < 3; ++c) {
    lo[c] = -wave_fmax(-t.part[c][lane & (W - 1)]);
    hi[c] = wave_fmax(t.part[3 + c][lane & (W - 1)]);
  }
  uint32_t key[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i)
    key[i] = curve_place(v[i], lo, hi, d < DIM ? d : DIM, AXIS_BITS)
                 << REL_BITS |
             (uint32_t)(first + i * kWave);
  const int shift = (wave & 1) * 16;
  uint32_t *const mine = t.count[wave / 2];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    uint32_t digit[PER], at[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      digit[i] = key[i] >> (REL_BITS + 9 * pass) & (kFpsDigits - 1);
      at[i] = first + i * kWave < count
                  ? atomicAdd(&mine[digit[i]], 1u << shift) >> shift & 0xffffu
                  : 0u;
    }
    __syncthreads();
    // a thread: eight waves' counts of one digit, two threads a digit
    uint32_t of[4], sum = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      of[i] = t.count[(tid & 1) * 4 + i][tid / 2];
      sum += (of[i] & 0xffffu) + (of[i] >> 16);
    }
    uint32_t before = sum;
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      const uint32_t other = __shfl_up(before, sh);
      before += lane >= sh ? other : 0u;
    }
    if (lane == kWave - 1)
      t.total[wave] = before;
    before -= sum;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w)
      before += w < wave ? t.total[w] : 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t low = before;
      before += of[i] & 0xffffu;
      t.count[(tid & 1) * 4 + i][tid / 2] = before << 16 | low;
      before += of[i] >> 16;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (first + i * kWave < count)
        keys[(mine[digit[i]] >> shift & 0xffffu) + at[i]] = key[i];
    __syncthreads();
    if (pass == 0) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
        key[i] = first + i * kWave < count ? keys[first + i * kWave] : 0u;
      clear();
      __syncthreads();
    }
  }
}

// The order along the curve has to pay: with fewer samples than this every row is
// looked at instead.  Calls, us, all rows / stretches, 16 examples: 400 rows, 100
// samples 63 / 64, 150 83 / 71; 1,024, 60 56 / 61, 100 76 / 68; 2,048, 110 86 / 91, 140
// 104 / 97; 4,096, 110 98 / 106, 140 118 / 113; 8,192, 140 140 / 155, 180 173 / 168;
// of 4 dimensions 2,048, 110 93 / 102, 140 111 / 109; 4,096, 140 129 / 135, 170 152 /
// 148.  Beyond that fps_bucket_kernel, 256 and 512 samples of 8 x 16,384 rows: 342 /
// 398, 669 / 584.
__device__ __forceinline__ int fps_few(int dim, int count) {
  if (dim <= 3)
    return count <= 512    ? 120
           : count <= 1024 ? 90
           : count <= 4096 ? 130
           : count <= 8192 ? 170
                           : 340;
  return count <= 2048 ? 140 : count <= 8192 ? 170 : 480;
}

// Such an example by a workgroup of 1,024 threads.  Up to 512 rows one wave has
// them all; up to 8,192 half of the threads hold the rows, which leaves fewer
// results to hand over per step; the
// others only come to the barriers of fps_every_row (one before the first step
// and one per step; 16 x 2,048 rows, 128 samples: 85 us, by all threads 111).
template <int DIM, int CAP, int T>
__device__ __forceinline__ void fps_few_samples(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int64_t *__restrict__ out, int count, int samples) {
  static_assert(T == 1024 && CAP % T == 0 && CAP <= 16 * T, "rows per thread");
  if constexpr (CAP == 16384) {
    fps_every_row<DIM, 16, T>(src, ptr, out_ptr, start, d, out);
  } else {
    if (CAP == 1024 && count <= 512) {
      if (threadIdx.x < kWave)
        fps_every_row<DIM, 8, kWave>(src, ptr, out_ptr, start, d, out);
      return;
    }
    if (threadIdx.x >= T / 2) {
      for (int m = 0; m < samples; ++m)
        __syncthreads();
      return;
    }
    if (CAP == 4096 && count <= 2048)
      fps_every_row<DIM, 4, T / 2>(src, ptr, out_ptr, start, d, out);
    else
      fps_every_row<DIM, CAP / (T / 2), T / 2>(src, ptr, out_ptr, start, d,
                                               out);
  }
}

// ---- fp32, up to 8,192 rows: a wave's own stretch of the curve ------------------
// (up to 16,384 of sorted rows of up to 3 dimensions, by fps_stream_kernel, in calls of
// many examples)
//
// The rows of an example in curve order are dealt to the 16 waves of a workgroup,
// a stretch each, and stay in registers: row r of a lane is the lane's of the r-th
// 64 rows of the stretch, a "piece" with a box.  A step has several samples (up to
// 16), found as follows.
//
// Every wave has D entries: the row with the largest running minimum of the
// stretch, the one that would have it if that row were sampled too, and so on, each
// with the value it would then have; and `rest`, the first of what would be left
// after all D.  Values with the reference's tie rule below them make one 64-bit
// number (the key), larger ones first, so equal values need no special case.  The
// entries of all waves are ranked.  A sample lowers minima only: while an entry's
// row is at least its value away from all entries ranked before it, those leave its
// value as it is, and while it comes before the `rest` of the waves whose last entry
// is ranked before it, no row without an entry can be ahead of it.  So the samples
// of a step are the longest run of first entries of which that holds for every pair
// -- the same samples, in the same order, as one by one.  (The first of all always
// holds.  A row that does not lower its own minimum -- no finite distance to itself,
// or a minimum of 0 -- is its wave's next entry again, and the `rest` ends the run.)
//
// A wave then tests the boxes of its pieces against all samples at once (16 samples
// x 4 boxes are its lanes) and goes through the pieces that a sample is near to.
//
// Bound by the chain of a step, about 5,250 cycles for nine samples of 4,096 rows (by
// the cycle counter, read after every meeting): 1,100 for the rows of the samples,
// 2,600 from there to the first meeting (1,400 for the entries of a wave whose rows
// changed, ten of sixteen do, the rest waits for the slowest), 850 to the second, 700
// to the third, 400 of them pairs and boxes.  The four waves of a SIMD issue vector
// instructions, some 150 each, in 53 % of it.
// 16 uniform clouds, calls, before (64 buckets in LDS, one entry each, the waves
// sharing the buckets of a step; up to 1,024 rows every row in every step) and now:
// 1,024 rows, 300 samples 180 -> 100 us; 2,048, 512 258 -> 158;
// 4,096 rows, a quarter 386 -> 283, half 609 -> 458, of 4 dimensions 477 -> 365,
// on 33^3 places (ties) 522 -> 294; 8,192 rows, a quarter 702 -> 601, on 33^3
// places 982 -> 621; 1,000 of 4 dimensions, 8 clouds, 1,043 -> 533.  Samples per step (simulated, 4,096 rows, 1,024 samples): 64
// buckets of one entry 5.3; 16 stretches of one entry 4.4, two 9.1, three 10.5 --
// the third costs every changed stretch another pass over its rows (310 us).
constexpr int kFpsBatch = 16; // samples per step at most
constexpr int kFpsOwnLeast = 256; // rows of an example (every wave has some)
template <int D> struct FpsRanks {
  uint64_t key[D * kFpsWaves]; // entry by entry, wave by wave
  // of rank i: coordinates; value, code, rest (0: not the wave's last entry)
  float4 place[kFpsBatch];
  uint4 what[kFpsBatch];
  int end[2]; // the first rank that is no sample of the step (by turns)
};

// The low word of a key: the complement of the tie rule's number of a row of up to
// 2^BITS (BITS + 1 bits of it: never 0, which is no row), then, in 4 bits, the piece
// that it is in.
template <int BITS>
__device__ __forceinline__ uint32_t fps_code(uint32_t rel, int piece) {
  const uint32_t tie = (rel & 255u) << (BITS - 8) | rel >> 8;
  return (~tie & ((2u << BITS) - 1)) << 4 | (uint32_t)piece;
}
template <int BITS>
__device__ __forceinline__ uint32_t fps_row_of(uint32_t code) {
  const uint32_t tie = ~(code >> 4) & ((1u << BITS) - 1);
  return (tie & ((1u << (BITS - 8)) - 1)) << 8 | tie >> (BITS - 8);
}
template <int N, typename F> __device__ __forceinline__ void for_each_of(F f) {
  if constexpr (N > 0) {
    for_each_of<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// The rows of a wave, R of a lane, with the boxes of its pieces and its D entries.
// S: samples of a step at most; BITS: row numbers.
template <int DIM, int R, int D, int S, int BITS> struct FpsHeld {
  static constexpr int BOXES = kWave / S; // a lane per box and sample
  static constexpr int CHUNKS = (R + BOXES - 1) / BOXES;
  static constexpr bool KEEP = R <= 8; // (16 rows: not the registers; formed again)
  // boxes (16 pieces and 32 samples a step: in LDS, as registers they are spilled; with
  // 16 samples a few are, which costs less: 100 x 16,000 rows, 480 samples 441 us, from
  // LDS 448, and with 12 pieces 100 x 12,000, 600 397, 413)
  static constexpr bool IN_REGS = R <= 8 || S <= 16;
  static_assert(R <= 16, "pieces of 4 bits in a code");
  float x[R][DIM];
  // a row's key: running minimum above, code below (minima are in [0, 5e4]: read
  // as doubles the keys order as they should, and none is a NaN); `left`: with the
  // entries found so far sampled
  double low[R], left[KEEP ? R : 1];
  // box BOXES i + lane / S
  float blo[IN_REGS ? CHUNKS : 1][DIM], bhi[IN_REGS ? CHUNKS : 1][DIM];
  // the wave's entries (uniform), and what is left after them
  uint32_t value[D], value_code[D], rest, rest_code;
  float q[D][DIM];

  static __device__ __forceinline__ float minimum(double key) {
    return __int_as_float(__double2hiint(key));
  }
  static __device__ __forceinline__ double with_minimum(double key, float m) {
    return __hiloint2double(__float_as_int(m), __double2loint(key));
  }

  // lower corner, upper corner of a piece's box
  static __device__ __forceinline__ float4 *box_of(int piece) {
    __shared__ float4 boxes[kFpsWaves][R][2];
    return boxes[threadIdx.x / kWave][piece];
  }

  // `row_at`(i, x): number and coordinates of the i-th row along the curve; piece r
  // is the rows from `place`(r) on that are before `to`.  (Lanes without a row: minimum
  // 0 and a code below those of rows, another one in every wave, so that waves without
  // any row have ranks of their own behind all others.)
  template <typename Rows, typename Place>
  __device__ __forceinline__ void load(const Rows &row_at, const Place &place,
                                       int to, const float (&begin_at)[DIM]) {
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int at = place(r) + lane;
      const bool ok = at < to;
      // (where there is none, the last one again)
      const uint32_t rel = row_at(min(at, to - 1), x[r]);
      low[r] = __hiloint2double(
          __float_as_int(ok ? 5e4f : 0.0f),
          (int)(ok ? fps_code<BITS>(rel, r) : threadIdx.x / kWave));
      if (KEEP)
        left[KEEP ? r : 0] = low[r];
    }
#pragma unroll
    for (int i = 0; IN_REGS && i < CHUNKS; ++i)
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        blo[IN_REGS ? i : 0][c] = __builtin_inff();
        bhi[IN_REGS ? i : 0][c] = -__builtin_inff();
      }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool ok = place(r) + lane < to;
      float lo[4] = {}, hi[4] = {};
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        // (a NaN is left out: such a row's minimum never changes)
        const float v = x[r][c];
        const bool in = ok && v == v;
        hi[c] = wave_fmax(in ? v : -__builtin_inff());
        lo[c] = -wave_fmax(in ? -v : -__builtin_inff());
        if (IN_REGS && lane / S == r % BOXES) {
          blo[IN_REGS ? r / BOXES : 0][c] = lo[c];
          bhi[IN_REGS ? r / BOXES : 0][c] = hi[c];
        }
      }
      if (!IN_REGS && lane == 0) {
        box_of(r)[0] = make_float4(lo[0], lo[1], lo[2], lo[3]);
        box_of(r)[1] = make_float4(hi[0], hi[1], hi[2], hi[3]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      low[r] = with_minimum(low[r],
                            fps_lower<DIM>(begin_at, x[r], minimum(low[r])));
  }

  // the first of the rows with the l entries found before sampled
  template <int l>
  __device__ __forceinline__ int best_of(uint32_t &most, uint32_t &its_code) {
    double key = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double with = low[r];
      if constexpr (KEEP && l > 0) {
        left[r] = with_minimum(
            left[r], fps_lower<DIM>(q[l - 1], x[r],
                                    minimum(l == 1 ? low[r] : left[r])));
        with = left[r];
      } else {
#pragma unroll
        for (int j = 0; j < l; ++j)
          with = with_minimum(with, fps_lower<DIM>(q[j], x[r], minimum(with)));
      }
      if (r == 0)
        key = with;
      else
        asm("v_max_f64 %0, %1, %2" : "=v"(key) : "v"(key), "v"(with));
    }
    const uint32_t high = (uint32_t)__double2hiint(key);
    const uint32_t word = (uint32_t)__double2loint(key);
    most = wave_umax(high);
    const uint64_t who = __ballot(high == most);
    int at = (int)__builtin_ctzll(who);
    if (__builtin_expect((who & (who - 1)) != 0, 0)) {
      const uint32_t mine = high == most ? word : 0u;
      const uint32_t top = wave_umax(mine);
      at = (int)__builtin_ctzll(__ballot(mine == top));
    }
    its_code = lane_value(word, at);
    return at;
  }
  __device__ __forceinline__ void find_entries() {
    for_each_of<D>([&](auto which) {
      constexpr int l = decltype(which)::value;
      const int at = this->template best_of<l>(value[l], value_code[l]);
      const int piece = (int)(value_code[l] & 15u);
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (R == 1 || piece == r) {
#pragma unroll
          for (int c = 0; c < DIM; ++c)
            q[l][c] = lane_value(x[r][c], at);
        }
    });
    best_of<D>(rest, rest_code);
  }
  // entry l is the one before it (a row that would be sampled again)
  __device__ __forceinline__ bool again(int l) const {
    return l > 0 && value[l] == value[l > 0 ? l - 1 : 0] &&
           value_code[l] == value_code[l > 0 ? l - 1 : 0];
  }

  // the pieces that a sample is near to, by samples (lane i % S: sample i)
  __device__ __forceinline__ void find_near(const float (&s)[DIM],
                                            uint64_t (&near)[CHUNKS]) const {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      float dd;
      if constexpr (IN_REGS) {
        dd = fps_box_distance<DIM>(s, blo[i], bhi[i]);
      } else {
        const float4 *box =
            box_of(i * BOXES + (int)(threadIdx.x & (kWave - 1)) / S);
        const float4 at[2] = {box[0], box[1]};
        const float lo[4] = {at[0].x, at[0].y, at[0].z, at[0].w};
        const float hi[4] = {at[1].x, at[1].y, at[1].z, at[1].w};
        float l[DIM], u[DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
          l[c] = lo[c];
          u[c] = hi[c];
        }
        dd = fps_box_distance<DIM>(s, l, u);
      }
      near[i] = __ballot(!(dd >= __uint_as_float(value[0])));
    }
  }
  // the first `got` samples; whether a minimum of the wave is another now
  __device__ __forceinline__ bool sample(const float (&s)[DIM],
                                         const uint64_t (&near)[CHUNKS],
                                         int got) {
    bool lower = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      uint32_t some = (uint32_t)(near[r / BOXES] >> (r % BOXES) * S) &
                      (S < 32 ? (1u << got) - 1 : 0xffffffffu >> (32 - got));
      if (some != 0) {
        const float was = minimum(low[r]);
        float now = was;
        do {
          float at[DIM];
#pragma unroll
          for (int c = 0; c < DIM; ++c)
            at[c] = lane_value(s[c], __builtin_ctz(some));
          some &= some - 1;
          now = fps_lower<DIM>(at, x[r], now);
        } while (some != 0);
        lower |= now < was;
        low[r] = with_minimum(low[r], now);
      }
    }
    return __ballot(lower) != 0;
  }
};

template <int DIM, int R, int D, typename Rows>
__device__ __forceinline__ void
fps_own_rows(const Rows &row_at, int count, FpsRanks<D> &t,
             const float (&begin_at)[DIM], int steps, int64_t start_idx,
             int64_t *__restrict__ out) {
  constexpr int W = kFpsWaves;
  constexpr int BITS = 14;
  static_assert(D * W <= kWave, "a lane per entry");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int from = wave * count / W, to = (wave + 1) * count / W;

  typedef FpsHeld<DIM, R, D, kFpsBatch, BITS> Held;
  Held h;
  h.load(row_at, [&](int r) { return from + r * kWave; }, to, begin_at);
  if (tid < 2)
    t.end[tid] = kFpsBatch;

  int m = 1, par = 0;
  bool changed = true;
  while (true) {
    if (changed) {
      h.find_entries();
      if (lane == 0) {
#pragma unroll
        for (int l = 0; l < D; ++l)
          t.key[l * W + wave] = (uint64_t)h.value[l] << 32 | h.value_code[l];
      }
    }
    fps_meet();
    // how many entries come before the wave's
    const uint64_t key = lane < D * W ? t.key[lane] : 0u;
    int rank = 0;
#pragma unroll
    for (int l = 0; l < D; ++l) {
      const uint64_t mine = (uint64_t)h.value[l] << 32 | h.value_code[l];
      rank = h.again(l) ? rank + 1
                        : __builtin_popcountll(__ballot(key > mine));
      if (rank < kFpsBatch && lane == 0) {
        t.place[rank] =
            make_float4(h.q[l][0], DIM > 1 ? h.q[l][DIM > 1 ? 1 : 0] : 0.0f,
                        DIM > 2 ? h.q[l][DIM > 2 ? 2 : 0] : 0.0f,
                        DIM > 3 ? h.q[l][DIM > 3 ? 3 : 0] : 0.0f);
        t.what[rank] = make_uint4(h.value[l], h.value_code[l],
                                  l == D - 1 ? h.rest : 0u,
                                  l == D - 1 ? h.rest_code : 0u);
      }
    }
    fps_meet();
    // lane i % 16: the entry of rank i
    const int a = lane & (kFpsBatch - 1);
    const float4 at = t.place[a];
    const uint4 of = t.what[a];
    const float xs[4] = {at.x, at.y, at.z, at.w};
    float sx[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      sx[c] = xs[c];
    if (wave < kFpsBatch / 4) {
      // sixteen entries against four that may follow them
      const int b = lane / 16 * 4 + wave;
      const float4 at_b = t.place[b];
      const uint4 of_b = t.what[b];
      const float xb[4] = {at_b.x, at_b.y, at_b.z, at_b.w};
      float dd = 0.0f;
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        const float df = sx[c] - xb[c];
        dd = c == 0 ? df * df : __builtin_fmaf(df, df, dd);
      }
      const uint64_t left = (uint64_t)of.z << 32 | of.w;
      const uint64_t key_b = (uint64_t)of_b.x << 32 | of_b.y;
      // (a distance that is NaN ends the run)
      const bool apart =
          (dd >= __uint_as_float(of_b.x)) & (left < key_b);
      const uint64_t ends = __ballot((a < b) & !apart);
      if (ends != 0 && lane == 0)
        atomicMin(&t.end[par], (int)__builtin_ctzll(ends) / 16 * 4 + wave);
    }
    uint64_t near[Held::CHUNKS];
    h.find_near(sx, near);
    fps_meet();
    const int end = t.end[par];
    const int got = min(__builtin_amdgcn_readfirstlane(end), steps - m);
    par ^= 1;
    if (wave == W - 1 && lane < got) {
      // (nobody waits for the stores)
      out[m + lane] = start_idx + fps_row_of<BITS>(of.y);
      if (lane == 0)
        t.end[par] = kFpsBatch;
    }
    m += got;
    if (m >= steps)
      break;
    changed = h.sample(sx, near, got);
  }
}

template <int DIM, int CAP>
__device__ __forceinline__ void
fps_own_example(const float *__restrict__ src, int64_t start_idx, int count,
                int64_t first, int d, int steps, int64_t *__restrict__ out) {
  constexpr int REL_BITS = 13;
  constexpr int D = 2;
  static_assert(CAP <= 8192, "row numbers of 13 bits");
  __shared__ uint32_t keys[CAP];
  __shared__ FpsSort sort;
  __shared__ __align__(16) FpsRanks<D> ranks;
  const float *rows = src + (size_t)start_idx * d;
  fps_curve_order<DIM, REL_BITS, CAP>(rows, count, d, keys, sort);
  if (threadIdx.x == 0)
    out[0] = first;
  float at[DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c)
    at[c] = c < d ? src[(size_t)first * d + c] : 0.0f;
  auto run = [&](auto pieces) {
    fps_own_rows<DIM, decltype(pieces)::value>(
        [&](int i, float (&x)[DIM]) {
          const uint32_t rel = keys[i] & ((1u << REL_BITS) - 1);
#pragma unroll
          for (int c = 0; c < DIM; ++c)
            x[c] = c < d ? rows[(size_t)rel * d + c] : 0.0f;
          return rel;
        },
        count, ranks, at, steps, start_idx, out);
  };
  // (rows of a lane: what the example takes, at most what the launch allows for)
  constexpr int MOST = CAP / kFpsThreads;
  if (MOST > 4 && count > 4 * kFpsThreads)
    run(std::integral_constant<int, MOST>{});
  else if (MOST > 2 && count > 2 * kFpsThreads)
    run(std::integral_constant<int, MOST < 4 ? MOST : 4>{});
  else if (MOST > 1 && count > kFpsThreads)
    run(std::integral_constant<int, MOST < 2 ? MOST : 2>{});
  else
    run(std::integral_constant<int, 1>{});
}

template <int DIM, int CAP>
__global__ __launch_bounds__(kFpsThreads) void fps_own_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int64_t *__restrict__ out) {
  const int b = blockIdx.x;
  const int64_t start_idx = ptr[b];
  // (CAP: the caller's bound on the rows of an example)
  const int count = (int)min(ptr[b + 1] - start_idx, (int64_t)CAP);
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end)
    return;
  const int steps = (int)(o_end - o_begin);
  if (steps < fps_few(DIM, count) || count < kFpsOwnLeast) {
    fps_few_samples<DIM, CAP, kFpsThreads>(src, ptr, out_ptr, start, d, out,
                                           count, steps);
    return;
  }
  const int64_t first = start_idx + (start ? start[b] : 0);
  fps_own_example<DIM, CAP>(src, start_idx, count, first, d, steps,
                            out + o_begin);
}

// Examples of up to 64 W P rows: bucket i of wave w is in the registers of
// that wave (row of a lane in px[.][i], pm[i]), its box and best in lane i.
// For 8,193 - 16,384 rows.  With up to 3 dimensions it is for callers that give
// pca_fps such a bound, the only way to sample such examples in buckets on a stream
// that is being captured; of hundreds of samples the sorted path is faster.  (The
// stretches with 16 rows per lane in its place: 200 - 300 samples 1.03 - 1.4 times as
// fast, but fewer, which look at every row, 2 - 12 % slower beside them.)  8 x 16,384 uniform rows, a quarter sampled: 1.27 -> 0.86 us
// per step (before: every row, from the same registers).
template <int DIM, int W, int P>
__global__ __launch_bounds__(W *kWave) void fps_bucket_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int64_t *__restrict__ out) {
  constexpr int T = W * kWave;
  constexpr int CAP = T * P;
  constexpr int REL_BITS = 14;
  static_assert(CAP <= 16384 && P <= 16 && W <= 16, "row numbers in the keys");
  __shared__ uint32_t keys[CAP];
  __shared__ FpsSort sort;
  __shared__ FpsBest<DIM> table[2][W];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int b = blockIdx.x;
  const int64_t start_idx = ptr[b];
  // (CAP: the caller's bound on the rows of an example)
  const int count = (int)min(ptr[b + 1] - start_idx, (int64_t)CAP);
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end)
    return;
  if (o_end - o_begin < fps_few(DIM, count) || count <= 0) {
    fps_few_samples<DIM, CAP, T>(src, ptr, out_ptr, start, d, out, count,
                                 (int)(o_end - o_begin));
    return;
  }
  const float *rows = src + (size_t)start_idx * d;

  fps_curve_order<DIM, REL_BITS, CAP>(rows, count, d, keys, sort);

  // -- the buckets of this wave -----------------------------------------------
  float px[DIM][P];
  float pm[P];
  uint32_t pr[P];
  float blo[DIM], bhi[DIM];
  FpsBest<DIM> best; // of the bucket of this lane
  best.val = 0u;
  best.rel = kFpsNoRow;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    blo[c] = 0.0f;
    bhi[c] = 0.0f;
    best.x[c] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int pos = (i * W + wave) * kWave + lane;
    const bool ok = pos < count;
    const int rel = ok ? (int)(keys[pos] & (CAP - 1)) : 0;
    pr[i] = ok ? (uint32_t)rel : kFpsNoRow;
    // (lanes without a row: minimum 0 and the last of all ties)
    pm[i] = ok ? 5e4f : 0.0f;
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      const float v = ok && c < d ? rows[(size_t)rel * d + c] : 0.0f;
      px[c][i] = v;
      asm volatile("" : "+v"(px[c][i]));
      // (fminf / fmaxf drop a NaN; such a row's minimum never changes)
      float l = ok ? v : __builtin_inff(), h = ok ? v : -__builtin_inff();
#pragma unroll
      for (int sh = 1; sh < kWave; sh <<= 1) {
        l = __builtin_fminf(l, __shfl_xor(l, sh));
        h = __builtin_fmaxf(h, __shfl_xor(h, sh));
      }
      if (lane == i) {
        blo[c] = l;
        bhi[c] = h;
      }
    }
    if (lane == i && (i * W + wave) * kWave < count)
      best.val = kFpsUnseen;
    // (one bucket after the other: all loads and reductions at once would
    // take several times the registers the loop below needs)
    __builtin_amdgcn_sched_barrier(0);
  }

  const int64_t first = start_idx + (start ? start[b] : 0);
  if (tid == 0)
    out[o_begin] = first;
  float cur[DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c)
    cur[c] = c < d ? src[(size_t)first * d + c] : 0.0f;

  for (int64_t m = o_begin + 1; m < o_end; ++m) {
    const int par = (int)(m & 1);
    uint32_t pass = (uint32_t)__ballot(
        !(fps_box_distance<DIM>(cur, blo, bhi) >= __uint_as_float(best.val)));
    // (every bucket's code with its own registers: a uniform branch each,
    // four at a time where none passes)
#pragma unroll
    for (int g = 0; g < P; g += 4) {
      if ((pass & (0xfu << g)) == 0)
        continue;
#pragma unroll
      for (int i = g; i < (g + 4 < P ? g + 4 : P); ++i) {
        if ((pass & (1u << i)) == 0)
          continue;
        float x[DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          x[c] = px[c][i];
        pm[i] = fps_lower<DIM>(cur, x, pm[i]);
        const uint32_t bits = __float_as_uint(pm[i]);
        const uint32_t top = wave_umax(bits);
        const int at = fps_first(__ballot(bits == top), pr[i]);
        const uint32_t row = lane_value(pr[i], at);
        float at_x[DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          at_x[c] = lane_value(x[c], at);
        const bool mine = lane == i;
        best.val = mine ? top : best.val;
        best.rel = mine ? row : best.rel;
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          best.x[c] = mine ? at_x[c] : best.x[c];
      }
    }
    {
      const uint32_t top =
          (uint32_t)__builtin_amdgcn_readlane((int)row16_umax(best.val), 15);
      const int at =
          fps_first(__ballot(best.val == top) & ((1ull << P) - 1), best.rel);
      if (lane == at)
        table[par][wave] = best;
    }
    fps_meet();
    const FpsBest<DIM> e = table[par][lane & (W - 1)];
    static_assert(W == 16, "one row of 16 lanes looks at the waves' bests");
    const uint32_t top =
        (uint32_t)__builtin_amdgcn_readlane((int)row16_umax(e.val), 15);
    const int at = fps_first(__ballot(e.val == top) & 0xffffull, e.rel);
    const uint32_t row = lane_value(e.rel, at);
    if (tid == 0)
      out[m] = start_idx + (int64_t)row;
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      cur[c] = lane_value(e.x[c], at);
  }
}

// ---- fp32, up to 3 dimensions, larger examples ---------------------------------

// The order of the rows of examples of up to 16,384 (rows beyond that many follow as
// they are, which changes no sample), a workgroup each, in place of a sort in memory.
// 16,384 rows 37 us, most of it their places on the curve and the way from memory,
// by one compute unit each; the sort in memory took 60 us in six launches.  Calls, us,
// before -> now: 200 x 9,000, 450 samples 425 -> 352; 16 x 10,000, 500 360 -> 344; 8 x
// 16,384, 1,000 485 -> 467.  (Rows, minima and boxes written here too, instead of by
// fps_gather_kernel: 8 x 16,384, 240 samples 290 instead of 269.)
__global__ __launch_bounds__(kFpsThreads) void fps_order_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr, int d,
    uint32_t *__restrict__ perm) {
  constexpr int REL_BITS = 14;
  constexpr int CAP = 1 << REL_BITS;
  __shared__ uint32_t keys[CAP];
  __shared__ FpsSort sort;
  const int64_t begin = ptr[blockIdx.x];
  const int64_t all = ptr[blockIdx.x + 1] - begin;
  if (all <= 0)
    return;
  const int count = (int)min(all, (int64_t)CAP);
  const float *rows = src + (size_t)begin * d;
  if (count <= CAP / 2)
    fps_curve_order<3, REL_BITS, CAP / 2>(rows, count, d, keys, sort);
  else if (count <= CAP / 4 * 3)
    fps_curve_order<3, REL_BITS, CAP / 4 * 3>(rows, count, d, keys, sort);
  else
    fps_curve_order<3, REL_BITS, CAP>(rows, count, d, keys, sort);
  for (int64_t i = threadIdx.x; i < all; i += kFpsThreads)
    perm[begin + i] =
        (uint32_t)(begin + (i < count ? keys[i] & (CAP - 1) : i));
}

// Rows in curve order, (x, y, z, row of the example), their running minima, and
// the box of every piece of 64 rows.  The pieces of an example, a multiple of four
// (places beyond the last row: minimum 0 and the last of all ties), follow piece
// number ptr[b] / 64 + 4 b, so that no two examples meet.  A wave per piece.
struct FpsPieces {
  float4 *rows;  // [pieces][64]
  float *minima; // [pieces][64]
  float *boxes;  // [pieces][8]: lower corner, -, upper corner, -
};
constexpr int kFpsPieces = 4;
static_assert(kFpsPieces == kBlock / kWave, "a block of the kernel below");
// What the workgroups of an example tell each other (see fps_shared_kernel): by
// turns two sets of kFpsShareWords, and who they are (fps_crew).
constexpr int kFpsShareMost = 32; // workgroups of an example at most
constexpr int kFpsShareRows = 1;  // rows of a lane that a workgroup is worth
constexpr int kFpsTold = 128;     // entries that they tell each other, of all
constexpr int kFpsShareWords = kFpsTold * 4;
struct FpsShare {
  uint64_t *words; // [examples][2][kFpsShareWords]; NULL: not shared
  uint32_t *state; // [examples]
};
// A state: the workgroups that came, from bit 16 on the number of them that go to work
// where it was closed before all were there, and whether the example is left to
// fps_stream_kernel.
constexpr uint32_t kFpsClosed = 1u << 31, kFpsMarked = 1u << 30;
__host__ __device__ constexpr int64_t fps_first_piece(int64_t begin, int b) {
  return begin / kWave + (int64_t)kFpsPieces * b;
}
__global__ __launch_bounds__(kBlock) void fps_gather_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr, int d,
    int first_segment, const uint32_t *__restrict__ perm, FpsPieces out,
    FpsShare share) {
  const int b = first_segment + blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1);
  if (share.words != nullptr && blockIdx.x == 0) {
    for (int i = threadIdx.x; i < 2 * kFpsShareWords; i += kBlock)
      share.words[(size_t)b * (2 * kFpsShareWords) + i] = 0u;
    if (threadIdx.x == 0)
      share.state[b] = 0u;
  }
  const int64_t begin = ptr[b], end = ptr[b + 1];
  if (begin + (int64_t)blockIdx.x * kBlock >= end)
    return;
  const int64_t rel = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool ok = begin + rel < end;
  const int64_t id = ok ? (int64_t)perm[begin + rel] : begin;
  float v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    v[c] = ok && c < d ? src[(size_t)id * d + c] : 0.0f;
  const int64_t first = fps_first_piece(begin, b);
  out.rows[first * kWave + rel] = make_float4(
      v[0], v[1], v[2],
      __uint_as_float(ok ? (uint32_t)(id - begin) : kFpsNoRow));
  out.minima[first * kWave + rel] = ok ? 5e4f : 0.0f;
  float *box = out.boxes + (first + rel / kWave) * 8;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // (fminf / fmaxf drop a NaN; such a row's minimum never changes)
    float lo = ok ? v[c] : __builtin_inff();
    float hi = ok ? v[c] : -__builtin_inff();
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      lo = __builtin_fminf(lo, __shfl_xor(lo, sh));
      hi = __builtin_fmaxf(hi, __shfl_xor(hi, sh));
    }
    if (lane == 0) {
      box[c] = lo;
      box[4 + c] = hi;
    }
  }
}

// ---- the same, an example by several workgroups -----------------------------------
//
// The pieces of an example are dealt in turn to up to 32 workgroups of 16 waves,
// which hold their rows in registers as in fps_own_kernel: along the curve the next
// piece is another workgroup's, so that the places where samples are found (the thin
// outer parts of a scan) are everybody's.  A workgroup ranks the entries and the
// `rest` of its waves and tells the others the first seven and, as a bound, the
// eighth; no row after a `rest` is told but after it.  All read what all
// told and go on alike: the entries that are before every bound are ranked, up to 32
// of them, and the samples of the step are the longest run of first ones that are
// pairwise apart.  (Three or seven entries of a workgroup are enough: of the scans
// below 18.5 samples per step with seven entries, 17.5 with three, simulated.)
//
// What is told are words of 8 bytes, half of each the step's number, so that a
// reader knows by the word itself that it has arrived: one trip through the
// memory that the XCDs share, no fence, no flag.  A workgroup writes a set again two
// steps later, when all have told the step between, that is, have read the set.
//
// All workgroups of an example have to run at the same time.  The launch asks for no
// more than the device has compute units, but each of them takes a whole one, and
// work on other streams may hold some.  So the workgroups of an example meet first
// (fps_crew), and those that came in time deal the pieces among themselves; one that
// comes later ends at once.  Where too few came to hold the rows, or one waits in vain
// for what another tells (`patience` looks, 1.3 ms, while both run), the example is
// marked, and fps_stream_kernel, launched behind, samples it from the start.
//
// Bound by the chain of a step, about 9,000 cycles for 16 samples of a scan of
// 200,000 rows by 32 workgroups (by the cycle counter, read after every meeting): rows
// of the samples and entries 2,500, of the slowest wave, a workgroup's own ranks 1,000,
// what is told 2,700 (of 16 workgroups 2,050), ranks of all 1,700, pairs and boxes
// 1,100.  Calls, us, one workgroup each -> shared: eight scans of 60,000 - 200,000
// rows, 2 % sampled, 2,795 -> 1,001; one of them 1,198 -> 475; uniform rows, 8 x
// 16,384, 1,000 samples 601 -> 409; 16 x 16,384, a quarter 1,588 -> 741; 64 x 20,000,
// a tenth 1,783 -> 999; 1 x 500,000, 5,000 samples 9,952 -> 2,407; 128 x 20,000, two
// workgroups each, 1,276 -> 1,350: not below four.  What else was tried, eight scans /
// one scan: the words of an entry in four lines that all workgroups write to 2,073 /
// 1,063 (before ranks and layout as they are 1,558 / 763); ranks by a wave of each
// SIMD, an entry after the other, 4,600 cycles; 16 workgroups of an example 1,866 /
// 633; a pause between two looks no change; a workgroup for 2,048 rows at least 1 x
// 16,000, 1,600 samples 581, for 4,096 706, for 1,024 526.
struct FpsTold {
  uint64_t tell[64];           // what this workgroup tells
  uint64_t key[3 * kFpsWaves]; // of this workgroup: entries, then rests
  // of all: value and code (0: none); coordinates; the bounds
  uint64_t first[kFpsTold];
  float at[kFpsTold][3];
  uint64_t bound[kFpsShareMost];
  // of rank i: coordinates and value; code, step that it is of
  float4 place[32];
  uint2 what[32];
  int end[2]; // the first rank that is no sample of the step (by turns)
  int late;
};
template <int R, int S>
__device__ __forceinline__ bool
fps_shared_rows(const float4 *__restrict__ rows, int count, int part, int parts,
                FpsTold &t, uint64_t *words, int patience,
                const float (&begin_at)[3], int steps, int64_t start_idx,
                int64_t *__restrict__ out) {
  constexpr int W = kFpsWaves;
  constexpr int D = 2;
  constexpr int BITS = 19;
  constexpr uint32_t STEP = (1u << 12) - 1; // below a code's 20 bits
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);

  typedef FpsHeld<3, R, D, S, BITS> Held;
  Held h;
  h.load(
      [&](int i, float (&x)[3]) {
        const float4 row = rows[i];
        x[0] = row.x;
        x[1] = row.y;
        x[2] = row.z;
        return __float_as_uint(row.w);
      },
      [&](int r) { return ((r * W + wave) * parts + part) * kWave; }, count,
      begin_at);
  if (tid < 2)
    t.end[tid] = S;
  if (tid == 0)
    t.late = 0;
  if (tid < kFpsTold)
    t.first[tid] = 0u;
  if (tid < kFpsShareMost)
    t.bound[tid] = 0u;
  if (tid < 32)
    t.what[tid] = make_uint2(0u, 0u);

  // (entries of a workgroup)
  const int tells = parts > 16 ? 4 : parts > 8 ? 8 : 16;
  const int slots = parts * tells;
  int m = 1, step = 0;
  bool changed = true;
  while (m < steps) {
    ++step;
    uint64_t *const set = words + (step & 1) * kFpsShareWords;
    if (changed) {
      h.find_entries();
      if (lane == 0) {
#pragma unroll
        for (int l = 0; l < D; ++l)
          t.key[l * W + wave] = (uint64_t)h.value[l] << 32 | h.value_code[l];
        t.key[D * W + wave] = (uint64_t)h.rest << 32 | h.rest_code;
      }
    }
    fps_meet();
    {
      const uint64_t key = lane < (D + 1) * W ? t.key[lane] : 0u;
      int rank = 0;
#pragma unroll
      for (int l = 0; l <= D; ++l) {
        const uint32_t value = l < D ? h.value[l < D ? l : 0] : h.rest;
        const uint32_t code = l < D ? h.value_code[l < D ? l : 0] : h.rest_code;
        const bool again =
            l < D ? h.again(l)
                  : value == h.value[D - 1] && code == h.value_code[D - 1];
        const uint64_t mine = (uint64_t)value << 32 | code;
        const uint64_t more = __ballot(key > mine);
        rank = again ? rank + 1 : __builtin_popcountll(more);
        if (rank < tells && lane < 4) {
          // the first rest, or what there is no room for, is the bound (told in the
          // first place); nothing is told after it
          const bool over = (more >> D * W) != 0;
          const bool bound = !over && (l == D || rank == tells - 1);
          const bool none = over || bound;
          const int n = l < D ? l : 0;
          const uint32_t low = code >> 4 << 12;
          // (by bits: a choice among members would put them in memory)
          uint32_t high = none ? 0u : value;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const uint32_t at = __float_as_uint(h.q[n][c]);
            high = lane == 1 + c ? at : high;
          }
          const uint32_t tag = (uint32_t)step & STEP;
          uint64_t *const to = t.tell + lane;
          if (rank < tells - 1)
            to[(1 + rank) * 4] = (uint64_t)high << 32 |
                                 (lane == 0 ? (none ? 0u : low) | tag
                                            : (uint32_t)step);
          if (bound)
            to[0] = (uint64_t)value << 32 | low | tag;
        }
      }
    }
    fps_meet();
    // (whole lines: written entry by entry, by their waves, the scans took 1,119 us
    // instead of 1,028, 16 x 16,384 rows 865 instead of 770)
    if (tid < tells * 4)
      __hip_atomic_store(set + part * tells * 4 + tid, t.tell[tid],
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < slots * 4) {
      const int slot = tid / 4, c = tid & 3;
      const uint32_t mask = (slot & (tells - 1)) == 0 || c == 0 ? STEP : ~0u;
      uint64_t word;
      bool here;
      int looks = 0;
      do {
        word = __hip_atomic_load(set + tid, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
        here = (((uint32_t)word ^ (uint32_t)step) & mask) == 0;
      } while (!here && ++looks < patience);
      if (!here)
        t.late = 1;
      if (c != 0)
        t.at[slot][c - 1] = __uint_as_float((uint32_t)(word >> 32));
      else if ((slot & (tells - 1)) == 0)
        t.bound[slot / tells] = word & ~(uint64_t)STEP;
      else
        t.first[slot] = word & ~(uint64_t)STEP;
    }
    fps_meet();
    if (t.late != 0)
      return false;
    // eight lanes count what comes before an entry; those before every bound have a
    // rank
    {
      static_assert(kFpsThreads == 8 * kFpsTold, "eight lanes for an entry");
      const int e = tid / 8, j = tid & 7;
      const uint64_t mine = t.first[e];
      if (__ballot(mine != 0u) != 0) {
        uint32_t rank = 0u;
        // (all at once takes registers that the rows need: eight scans 1,255 us)
#pragma unroll 4
        for (int i = 0; i < kFpsTold / 16; ++i) {
          rank += t.first[i * 16 + j * 2] > mine;
          rank += t.first[i * 16 + j * 2 + 1] > mine;
        }
        bool over = false;
#pragma unroll
        for (int i = 0; i < kFpsShareMost / 16; ++i) {
          over |= t.bound[i * 16 + j * 2] > mine;
          over |= t.bound[i * 16 + j * 2 + 1] > mine;
        }
        rank += over ? 256u : 0u;
        rank = row8_sum(rank);
        if (j == 0 && mine != 0u && rank < (uint32_t)S) {
          t.place[rank] = make_float4(t.at[e][0], t.at[e][1], t.at[e][2],
                                      __uint_as_float((uint32_t)(mine >> 32)));
          t.what[rank] = make_uint2((uint32_t)mine >> 12 << 4, (uint32_t)step);
        }
      }
    }
    fps_meet();
    // lane i % S: the entry of rank i
    const int a = lane & (S - 1);
    const float4 at = t.place[a];
    const uint2 of = t.what[a];
    const float sx[3] = {at.x, at.y, at.z};
    {
      // against those that may follow them, 64 / S of a wave
      constexpr int OF = kWave / S;
      const int b = wave * OF + lane / S;
      const float4 at_b = t.place[b & (S - 1)];
      const bool is = t.what[b & (S - 1)].y == (uint32_t)step;
      const float xb[3] = {at_b.x, at_b.y, at_b.z};
      float dd = 0.0f;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float df = sx[c] - xb[c];
        dd = c == 0 ? df * df : __builtin_fmaf(df, df, dd);
      }
      // (a distance that is NaN ends the run)
      const uint64_t ends =
          __ballot((a < b) & (b < S) & !(is & (dd >= at_b.w)));
      if (ends != 0 && lane == 0)
        atomicMin(&t.end[step & 1],
                  wave * OF + (int)__builtin_ctzll(ends) / S);
    }
    uint64_t near[Held::CHUNKS];
    h.find_near(sx, near);
    fps_meet();
    const int end = __builtin_amdgcn_readfirstlane(t.end[step & 1]);
    const int got = min(end, steps - m);
    if (wave == W - 1) {
      if (part == 0 && lane < got)
        out[m + lane] = start_idx + fps_row_of<BITS>(of.x);
      if (lane == 0)
        t.end[(step & 1) ^ 1] = S;
    }
    m += got;
    changed = h.sample(sx, near, got);
  }
  return true;
}

// The workgroups of an example agree on who they are; one thread of each calls this.
// Returns which one it is, of how many (y); -1: it is not needed.  `most`: at most so
// many, `least`: as many as hold the rows.  They wait for each other: `patience`
// looks of 0.12 us (30 us) once half of them are there and hold the rows, and while not
// 16 times as long (0.5 ms) or, if that is more, a patience for every 64 of the `steps`
// samples, since examples that run make room when they are done and one workgroup
// takes about twice that for the samples.  So units that are held by other work cost a
// call that wait and their part of the speed, not the sharing.  One word decides, so
// all see the same.
// Calls, us, alone / beside a wave that sleeps on another stream, without this meeting
// (a held unit cost its example 1.3 ms and the sharing) / now, and beside three: eight
// scans 1,015 / 3,670 / 996, 1,025; 16 x 16,384 rows, a quarter 740 / 1,450 / 749, 787;
// 64 x 20,000, a tenth 798 / 1,380 / 814, 1,385.  Three calls at once, without this
// meeting / with 30 us for all numbers that hold the rows and 0.5 ms for fewer / now:
// 5 x 100,000 rows, 2 % 1,580 / 1,571 - 2,820 / 1,583 - 1,659; 8 x 130,000, 2 % 7,200 /
// 2,079 - 5,268 / 2,084 - 2,881; 16 x 16,384, a quarter 5,300 / 2,130 / 2,160.
constexpr int kFpsCrewWait = 64; // samples that a patience more is waited for
__device__ __forceinline__ int2 fps_crew(uint32_t *state, int most, int least,
                                         int patience, int steps) {
  constexpr uint32_t CAME = 0xffffu;
  const uint32_t before = __hip_atomic_fetch_add(
      state, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int part = (int)(before & CAME);
  if ((before & kFpsClosed) != 0 || part >= most)
    return make_int2(-1, 0);
  const int enough = max(least, most / 2);
  const int64_t for_enough =
      (int64_t)patience * max(16, (steps + kFpsCrewWait - 1) / kFpsCrewWait);
  for (int looks = 0;; ++looks) {
    uint32_t now = __hip_atomic_load(state, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
    const int here = (int)(now & CAME);
    if ((now & kFpsClosed) != 0) {
      const int parts = (int)(now >> 16 & 0xffu);
      return make_int2(parts >= least ? part : -1, parts);
    }
    if (here >= most)
      return make_int2(part, most);
    // (tried again only if one more came, at most `most` times)
    if (looks >= (here >= enough ? (int64_t)patience : for_enough))
      __hip_atomic_compare_exchange_strong(
          state, &now,
          now | kFpsClosed | (here < least ? kFpsMarked : 0u) |
              (uint32_t)here << 16,
          __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// `most` workgroups for every example, those of an example on one XCD where every XCD
// gets as many examples (16 x 16,384 rows, a quarter 742 us, spread over the XCDs 784;
// 64 x 20,000, a tenth 992, 1,056; eight scans 994, 1,032), else in a row.
constexpr int kFpsShareGrid = 256; // all of a launch at most: a compute unit each
template <int R, int S>
__global__ __launch_bounds__(kFpsThreads) void fps_shared_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, int most, FpsPieces p, FpsShare share, int patience, int meeting,
    int64_t *__restrict__ out) {
  __shared__ __align__(16) FpsTold told;
  __shared__ int2 s_crew;
  int b = blockIdx.x / most, index = blockIdx.x % most;
  if (gridDim.x / most % 8 == 0) {
    // (workgroup i is on XCD i % 8)
    const int at_xcd = blockIdx.x / 8;
    b = (int)(blockIdx.x % 8) + 8 * (at_xcd / most);
    index = at_xcd % most;
  }
  const int64_t start_idx = ptr[b];
  const int64_t rows = ptr[b + 1] - start_idx;
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end || rows <= 0)
    return;
  // (Of fewer than 1,024 rows some waves have none.  Such examples were left to
  // fps_stream_kernel, behind the others: 4 x 20,000 rows, a tenth sampled, and 12 x
  // 1,000, all sampled, 1,227 -> 629 us; 8 x 9,000 and 8 x 1,023, a fifth, 567 -> 476.)
  const int64_t parts64 =
      max((int64_t)1, min((int64_t)most,
                          rows / (kFpsWaves * kWave * kFpsShareRows)));
  if (rows > parts64 * R * kFpsThreads) {
    if (threadIdx.x == 0)
      __hip_atomic_store(share.state + b, kFpsMarked, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  if (threadIdx.x == 0)
    s_crew = fps_crew(share.state + b, (int)parts64,
                      (int)((rows + R * kFpsThreads - 1) / (R * kFpsThreads)),
                      meeting, (int)(o_end - o_begin));
  __syncthreads();
  const int parts = __builtin_amdgcn_readfirstlane(s_crew.y);
  // (in order if all came: one scan 420 us of this kernel as they came, 409 in order)
  const int part = parts == most ? index
                                 : __builtin_amdgcn_readfirstlane(s_crew.x);
  if (part < 0)
    return;
  const int64_t first = start_idx + (start ? start[b] : 0);
  if (part == 0 && threadIdx.x == 0)
    out[o_begin] = first;
  float at[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    at[c] = c < d ? src[(size_t)first * d + c] : 0.0f;
  const int need = (int)((rows + parts * kFpsThreads - 1) / (parts * kFpsThreads));
  auto run = [&](auto rows_of_lane) {
    return fps_shared_rows<decltype(rows_of_lane)::value, S>(
        p.rows + fps_first_piece(start_idx, b) * kWave, (int)rows, part, parts,
        told, share.words + (size_t)b * (2 * kFpsShareWords), patience, at,
        (int)(o_end - o_begin), start_idx, out + o_begin);
  };
  bool done;
  if (R > 8 && need > 8)
    done = run(std::integral_constant<int, R>{});
  else if (need > 4)
    done = run(std::integral_constant<int, 8>{});
  else if (need > 2)
    done = run(std::integral_constant<int, 4>{});
  else
    done = run(std::integral_constant<int, 2>{});
  if (!done && threadIdx.x == 0)
    __hip_atomic_fetch_or(share.state + b, kFpsMarked, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
}

// For calls that fps_shared_kernel does not take, and the examples that it marks
// (`only`; NULL: all).
//
// A bucket has R pieces of 64 rows (MANY: a multiple of that) and belongs to a
// lane of the workgroup: its box and its best row are in that lane's registers; the
// rows and their running minima stay in memory, that is in the L2 of the
// workgroup's XCD.  The groups of the samples' table are rows of 16 lanes.  A step
// of up to eight samples: every wave tests its buckets (those samples only that
// are near to any of them), the buckets that pass go on a list, all waves share
// the list, the owners take the results, the entries are ranked.
//
// Eight ragged LiDAR-like scans of 60,000 - 200,000 rows, 2 % sampled: 5.75 ->
// 2.79 ms per call, 1.47 -> 0.71 us per sample of the longest scan (before: one
// sample per step).  Uniform rows, samples: 8 x 20,000, 2,000 each 2.22 -> 1.16
// ms; 8 x 60,000, 600 each 1.27 -> 0.83; 2 x 300,000, 900 each 4.54 -> 2.93.
// Where nearly every maximum is a tie (4 x 200,000 rows on 33^3 places, 2,000 samples
// each) 5.2 -> 3.2 ms; without the tie of `rest` a step there ends with its first
// sample (6.0 ms).
// Bound by the chain of a step, about 7,000 cycles for five samples of a scan of
// 200,000 rows: 1,400 to the list, 2,500 + 1,200 for the 21 buckets of the list
// (their rows at the 64 bytes per clock that a compute unit gets from the L2, and
// the wait for the slowest wave), 1,800 for entries and ranks, of which most is
// instructions that all sixteen waves execute.  Figures behind the choices, on
// the scans: with the owners looking at their own buckets 3.1 ms, two thirds of
// it waits for the wave with the most; minima stored where nothing changed 3.4;
// up to four samples per step 3.7; buckets of 128 rows 2.9 (16-lane groups of
// 64 rows could not hold 200,000).
template <int W, int R, bool MANY, bool OWN>
__global__ __launch_bounds__(W *kWave) void fps_stream_kernel(
    const float *__restrict__ src, const int64_t *__restrict__ ptr,
    const int64_t *__restrict__ out_ptr, const int64_t *__restrict__ start,
    int d, FpsPieces p, const uint32_t *__restrict__ only,
    int64_t *__restrict__ out) {
  constexpr int DIM = 3;
  static_assert(W * 4 == kWave, "a group per row of 16 lanes");
  static_assert(kFpsPieces % R == 0, "whole buckets");
  __shared__ FpsTable table;
  // the buckets of a step, with the samples that they are near to, and what was
  // found in them
  __shared__ uint32_t list[kWave * W];
  __shared__ float4 found_head[kWave * W]; // value, row, x, y
  __shared__ float4 found_tail[kWave * W]; // z, rest, its tie, -
  __shared__ int items[2];
  __shared__ uint32_t sampled[2 * kWave];
  __shared__ __align__(16) FpsRanks<OWN ? 2 : 1> ranks;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int b = blockIdx.x;
  const int64_t start_idx = ptr[b];
  const int count = (int)(ptr[b + 1] - start_idx);
  const int64_t o_begin = out_ptr[b];
  const int64_t o_end = out_ptr[b + 1];
  if (o_begin >= o_end || count <= 0 ||
      (only != nullptr && (only[b] & kFpsMarked) == 0u))
    return;
  const int64_t first_piece = fps_first_piece(start_idx, b);
  const float4 *rows = p.rows + first_piece * kWave;
  // Examples whose rows fit the registers after all (a bound of 16,385: 8 x 16,384
  // rows, 1,000 samples 727 -> 589 us, 8,300 666 -> 521; 200 x 9,000, 450 samples, with
  // 16 rows of a lane 468, with 12 425).  Not in calls of larger ones: the registers
  // make those 1 % slower.
  if (OWN && count >= kFpsOwnLeast && count <= 16 * kFpsThreads) {
    float at[DIM];
    const int64_t first = start_idx + (start ? start[b] : 0);
    if (tid == 0)
      out[o_begin] = first;
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      at[c] = c < d ? src[(size_t)first * d + c] : 0.0f;
    auto run = [&](auto rows_of_lane) {
      fps_own_rows<DIM, decltype(rows_of_lane)::value>(
          [&](int i, float (&x)[DIM]) {
            const float4 row = rows[i];
            x[0] = row.x;
            x[1] = row.y;
            x[2] = row.z;
            return __float_as_uint(row.w);
          },
          count, ranks, at, (int)(o_end - o_begin), start_idx, out + o_begin);
    };
    if (count > 12 * kFpsThreads)
      run(std::integral_constant<int, 16>{});
    else if (count > 8 * kFpsThreads)
      run(std::integral_constant<int, 12>{});
    else
      run(std::integral_constant<int, 8>{});
    return;
  }
  float *minima = p.minima + first_piece * kWave;
  const int pieces = (count + kWave - 1) / kWave;
  const int chunks =
      MANY ? max(1, (pieces + kWave * W * R - 1) / (kWave * W * R)) : 1;
  const int per_bucket = chunks * R;
  const int buckets = (pieces + per_bucket - 1) / per_bucket;
  const int last = (pieces - 1) / R * (R * kWave) + lane;
  // The buckets of a wave follow each other along the curve, so that most
  // samples are far from all of them; neighbours, of which one sample often
  // changes several, are in different groups.
  const int run = (buckets + W - 1) / W;
  const int slot = (lane & 15) * 4 + lane / 16;
  const int bucket = wave * run + slot;

  float blo[DIM], bhi[DIM], bx[DIM];
  uint32_t val, rest = 0u, rest_tie = kFpsAnyTie, rel = kFpsNoRow;
  {
    const int k = bucket;
    const bool any = slot < run && k < buckets;
    val = any ? kFpsUnseen : 0u;
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      blo[c] = __builtin_inff();
      bhi[c] = -__builtin_inff();
      bx[c] = 0.0f;
    }
    const float *box = p.boxes + (first_piece + (int64_t)k * per_bucket) * 8;
    for (int i = 0; any && i < per_bucket && k * per_bucket + i < pieces; ++i) {
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        blo[c] = __builtin_fminf(blo[c], box[i * 8 + c]);
        bhi[c] = __builtin_fmaxf(bhi[c], box[i * 8 + 4 + c]);
      }
    }
  }

  // of all buckets of the wave: box, largest value
  float wlo[DIM], whi[DIM];
  uint32_t wave_val = kFpsUnseen;
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    wlo[c] = blo[c];
    whi[c] = bhi[c];
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) {
      wlo[c] = __builtin_fminf(wlo[c], __shfl_xor(wlo[c], sh));
      whi[c] = __builtin_fmaxf(whi[c], __shfl_xor(whi[c], sh));
    }
  }
  if (tid < 2)
    items[tid] = 0;
  __syncthreads();
  float sx[DIM]; // lane i: sample i of the step
  int got = 1, turn = 0;
  {
    const int64_t first = start_idx + (start ? start[b] : 0);
    if (tid == 0)
      out[o_begin] = first;
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      sx[c] = c < d ? src[(size_t)first * d + c] : 0.0f;
  }

  const int steps = (int)(o_end - o_begin);
  int m = 1;
  while (m < steps) {
    uint32_t hits = 0; // bit i: sample i may lower a minimum of this bucket
    uint32_t near = (uint32_t)__ballot(
        lane < got && !(fps_box_distance<DIM>(sx, wlo, whi) >=
                        __uint_as_float(wave_val)));
    while (near != 0) {
      const int i = __builtin_ctz(near);
      near &= near - 1;
      float q[DIM];
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        q[c] = lane_value(sx[c], i);
      const bool passes =
          !(fps_box_distance<DIM>(q, blo, bhi) >= __uint_as_float(val));
      hits |= passes ? 1u << i : 0u;
    }
    // the buckets to look at, for all waves
    const uint64_t pass = __ballot(hits != 0);
    int item = 0;
    if (pass != 0) {
      int base = 0;
      if (lane == 0)
        base = atomicAdd(&items[turn], __builtin_popcountll(pass));
      item = __builtin_amdgcn_readfirstlane(base) +
             __builtin_amdgcn_mbcnt_hi(
                 (uint32_t)(pass >> 32),
                 __builtin_amdgcn_mbcnt_lo((uint32_t)pass, 0u));
      if (hits != 0)
        list[item] = (uint32_t)bucket | hits << 16;
    }
    // (with the rows' minima of the step before, which any wave may read now)
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(items[turn]);
    turn ^= 1;
    if (tid == 0)
      items[turn] = 0;
    // U buckets at a time, so that their rows are on the way together
    auto look = [&](auto many, const int first_item) {
      constexpr int U = decltype(many)::value;
      uint32_t todo[U];
      int bucket[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t what = (uint32_t)__builtin_amdgcn_readfirstlane(
            (int)list[first_item + u * W]);
        bucket[u] = (int)(what & 0xffffu);
        todo[u] = what >> 16;
      }
      // a lane's largest minimum of each bucket and the second
      uint32_t f_val[U], f_rest[U], f_rel[U];
      float f_x[U][DIM];
      int i_last[U];
      float4 v[U][R];
      float low[U][R];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        i_last[u] = (pieces - 1) / R - bucket[u] * chunks;
        f_val[u] = 0u;
        f_rest[u] = 0u;
      }
      for (int i = 0; i < chunks; ++i) {
        float was[U][R];
        int at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          at[u] = (bucket[u] * chunks + i) * (R * kWave) + lane;
          // (MANY: the pieces may end inside the bucket; then the last ones
          // again, which are not looked at below)
          if (MANY)
            at[u] = min(at[u], last);
#pragma unroll
          for (int r = 0; r < R; ++r)
          {
            v[u][r] = rows[at[u] + r * kWave];
            was[u][r] = minima[at[u] + r * kWave];
            low[u][r] = was[u][r];
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          uint32_t some = todo[u];
          do {
            float q[DIM];
#pragma unroll
            for (int c = 0; c < DIM; ++c)
              q[c] = lane_value(sx[c], __builtin_ctz(some));
            some &= some - 1;
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const float x[DIM] = {v[u][r].x, v[u][r].y, v[u][r].z};
              low[u][r] = fps_lower<DIM>(q, x, low[u][r]);
            }
          } while (some != 0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t before = f_val[u];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (low[u][r] < was[u][r])
              minima[at[u] + r * kWave] = low[u][r];
            const uint32_t bits =
                !MANY || i <= i_last[u] ? __float_as_uint(low[u][r]) : 0u;
            // (the middle one of three: the second largest is not below it)
            f_rest[u] = max(f_rest[u], min(f_val[u], bits));
            f_val[u] = max(f_val[u], bits);
          }
          // which row it is (the last one of equal ones)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const bool is = __float_as_uint(low[u][r]) == f_val[u] &&
                            (!MANY || f_val[u] > before);
            if (r == 0 && !MANY) {
              f_rel[u] = __float_as_uint(v[u][r].w);
              f_x[u][0] = v[u][r].x;
              f_x[u][1] = v[u][r].y;
              f_x[u][2] = v[u][r].z;
            } else {
              f_rel[u] = is ? __float_as_uint(v[u][r].w) : f_rel[u];
              f_x[u][0] = is ? v[u][r].x : f_x[u][0];
              f_x[u][1] = is ? v[u][r].y : f_x[u][1];
              f_x[u][2] = is ? v[u][r].z : f_x[u][2];
            }
          }
        }
      }
      uint32_t top[U], next[U];
      uint64_t who[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        top[u] = f_val[u];
      wave_umax_of<U>(top);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool is = f_val[u] == top[u];
        who[u] = __ballot(is);
        next[u] = is ? f_rest[u] : f_val[u];
      }
      wave_umax_of<U>(next);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint32_t next_tie = kFpsAnyTie;
        int at = (int)__builtin_ctzll(who[u]);
        if (__builtin_expect((who[u] & (who[u] - 1)) != 0 || next[u] == top[u],
                             0)) {
          // rows of equal value: the one that comes first in the reference's
          // order
          next[u] = top[u];
          uint32_t first = 0u, second = 0u; // (complements of smallest ties)
          auto among = [&](const float4(&row)[R], const float(&m)[R]) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const bool is = __float_as_uint(m[r]) == top[u];
              const uint32_t t = is ? ~fps_tie(__float_as_uint(row[r].w)) : 0u;
              const bool take = t > first;
              second = max(second, min(first, t));
              first = max(first, t);
              f_rel[u] = take ? __float_as_uint(row[r].w) : f_rel[u];
              f_x[u][0] = take ? row[r].x : f_x[u][0];
              f_x[u][1] = take ? row[r].y : f_x[u][1];
              f_x[u][2] = take ? row[r].z : f_x[u][2];
            }
          };
          if (R > 1 && !MANY) {
            among(v[u], low[u]);
          } else {
#pragma unroll 1
            for (int i = 0; i < chunks; ++i) {
              float4 row[R];
              float m[R];
              const int to = min(
                  (bucket[u] * chunks + i) * (R * kWave) + lane, last);
#pragma unroll
              for (int r = 0; r < R; ++r) {
                row[r] = rows[to + r * kWave];
                m[r] = minima[to + r * kWave];
              }
              among(row, m);
            }
          }
          const uint32_t most = wave_umax(first);
          at = (int)__builtin_ctzll(__ballot(first == most));
          next_tie = wave_umax(lane == at ? second : first);
        }
        if (lane == at) {
          found_head[first_item + u * W] =
              make_float4(__uint_as_float(top[u]), __uint_as_float(f_rel[u]),
                          f_x[u][0], f_x[u][1]);
          found_tail[first_item + u * W] =
              make_float4(f_x[u][2], __uint_as_float(next[u]),
                          __uint_as_float(next_tie), 0.0f);
        }
      }
    };
    int i = wave;
    for (; i + W < total; i += 2 * W)
      look(std::integral_constant<int, 2>{}, i);
    if (i < total)
      look(std::integral_constant<int, 1>{}, i);
    fps_meet();
    if (hits != 0) {
      const float4 h = found_head[item];
      const float4 t = found_tail[item];
      val = __float_as_uint(h.x);
      rel = __float_as_uint(h.y);
      bx[0] = h.z;
      bx[1] = h.w;
      bx[2] = t.x;
      rest = __float_as_uint(t.y);
      rest_tie = __float_as_uint(t.z);
    }
    if (pass != 0 || m == 1) {
      // the best of every group
      const uint32_t top = row16_umax_all(val);
      bool is = val == top;
      uint32_t next = row16_umax_all(is ? rest : val);
      uint32_t next_tie = next == top ? rest_tie : kFpsAnyTie;
      if (__builtin_expect(__builtin_popcountll(__ballot(is)) > 4, 0)) {
        // several of a group
        const uint32_t t = is ? ~fps_tie(rel) : 0u;
        const uint32_t first = row16_umax_all(t);
        const bool it = is && t == first;
        const uint32_t other =
            row16_umax_all(it ? (rest == top ? rest_tie : 0u) : t);
        next = other != 0u ? top : next;
        next_tie = other != 0u ? other : next_tie;
        is = it;
      }
      wave_val = max(max(lane_value(top, 0), lane_value(top, 16)),
                     max(lane_value(top, 32), lane_value(top, 48)));
      if (is) {
        fps_enter<DIM>(table, wave * 4 + lane / 16, top, rel, bx, next,
                       next_tie);
      }
    }
    uint32_t chosen;
    got = fps_rank<kWave / W, DIM>(
        table, wave, [](uint32_t row) { return row; }, sx, chosen);
    got = min(got, steps - m);
    if (wave == 0) {
      // (64 samples are written out at a time)
      if (lane < got)
        sampled[(m + lane) & (2 * kWave - 1)] = chosen;
      const int from = m & ~(kWave - 1), to = m + got;
      if (to >= from + kWave || to == steps) {
        // (the last step may end one block of samples and begin another)
        for (int k = from + lane; k < to; k += kWave)
          if (k > 0 && (k < from + kWave || to == steps))
            out[o_begin + k] =
                start_idx + (int64_t)sampled[k & (2 * kWave - 1)];
      }
    }
    m += got;
  }
}

// Up to 1,024 rows the kernels that look at every row take less of a compute unit:
// for more examples than this.  Every row / stretches, us: 400 rows, 200 samples, 256
// examples 102 / 84, 300 105 / 133; 1,024 rows, 60 samples 56 / 56, 63 / 89.
constexpr int kFpsOwnMost = 256;

template <int DIM>
hipError_t launch_fps_on_chip(const float *src, const int64_t *ptr,
                              const int64_t *out_ptr, const int64_t *start,
                              int d, int num_segments, int64_t max_rows,
                              int64_t *out, hipStream_t stream) {
#define PCA_FPS_LAUNCH(kernel_, threads_)                                      \
  hipLaunchKernelGGL((kernel_), dim3(num_segments), dim3(threads_), 0, stream, \
                     src, ptr, out_ptr, start, d, out)
  // (shapes by measurement: 16 examples of each size on one device; the
  // kernels' comments give the times on both sides of a limit)
  const bool many = num_segments > kFpsOwnMost;
  if (max_rows <= 256)
    PCA_FPS_LAUNCH((fps_reg_kernel<DIM, 4, 64>), 64);
  else if (max_rows <= 512 && many)
    PCA_FPS_LAUNCH((fps_reg_kernel<DIM, 8, 64>), 64);
  else if (max_rows <= 1024 && many)
    PCA_FPS_LAUNCH((fps_reg_kernel<DIM, 2, 512>), 512);
  else if (max_rows <= 1024)
    PCA_FPS_LAUNCH((fps_own_kernel<DIM, 1024>), 1024);
  else if (max_rows <= 2048)
    PCA_FPS_LAUNCH((fps_own_kernel<DIM, 2048>), 1024);
  else if (max_rows <= 4096)
    PCA_FPS_LAUNCH((fps_own_kernel<DIM, 4096>), 1024);
  else if (max_rows <= 8192)
    PCA_FPS_LAUNCH((fps_own_kernel<DIM, 8192>), 1024);
  else
    PCA_FPS_LAUNCH((fps_bucket_kernel<DIM, 16, 16>), 1024);
#undef PCA_FPS_LAUNCH
  return hipGetLastError();
}

template <typename Tr>
hipError_t launch_fps_any(const void *src, const int64_t *ptr,
                          const int64_t *out_ptr, const int64_t *start, int d,
                          int num_segments, void *dist, int64_t *out,
                          hipStream_t stream) {
  hipLaunchKernelGGL((fps_any_kernel<Tr>), dim3(num_segments),
                     dim3(kFpsThreads), 0, stream,
                     static_cast<const typename Tr::store_t *>(src), ptr,
                     out_ptr, start, d,
                     static_cast<typename Tr::calc_t *>(dist), out);
  return hipGetLastError();
}

} // namespace

// Examples of up to 16,384 rows of up to 4 dimensions.
static bool fps_on_chip(int dtype, int d, int64_t max_rows) {
  return dtype == 0 && d >= 1 && d <= 4 && max_rows >= 1 &&
         max_rows <= 16 * kFpsThreads;
}

// Larger examples of up to three dimensions: rows in curve order in memory.
static bool fps_streams(int dtype, int d, int64_t max_rows) {
  return dtype == 0 && d >= 1 && d <= 3 && max_rows > 16 * kFpsThreads;
}

static size_t fps_align(size_t v) { return (v + 255) & ~(size_t)255; }

// Workgroups of an example, for calls of few enough examples (else 0).
static int fps_share_most(int num_segments) {
  const int most = std::min(kFpsShareMost, kFpsShareGrid / num_segments);
  return most >= 4 ? most : 0;
}
static size_t fps_share_bytes(int num_segments) {
  if (fps_share_most(num_segments) == 0)
    return 0;
  return fps_align(sizeof(uint64_t) * 2 * kFpsShareWords *
                   (size_t)num_segments) +
         fps_align(sizeof(uint32_t) * (size_t)num_segments);
}

static size_t fps_pieces_bytes(size_t pieces) {
  return fps_align(sizeof(float4) * kWave * pieces) +
         fps_align(sizeof(float) * kWave * pieces) +
         fps_align(sizeof(float) * 8 * pieces);
}
size_t fps_states_at(int n, int num_segments) {
  return fps_pieces_bytes((size_t)fps_first_piece(n, num_segments)) +
         fps_align(sizeof(uint64_t) * 2 * kFpsShareWords *
                   (size_t)num_segments);
}

size_t fps_scratch_bytes(int dtype, int n, int d, int num_segments,
                         int64_t max_rows) {
  if (fps_on_chip(dtype, d, max_rows))
    return 0;
  const size_t dist = fps_align(sizeof(double) * (size_t)n);
  if (!fps_streams(dtype, d, max_rows))
    return dist;
  const size_t pieces = (size_t)fps_first_piece(n, num_segments);
  // (a stream that is being captured takes fps_any_kernel and its `dist`)
  return std::max(dist, fps_pieces_bytes(pieces) +
                            fps_share_bytes(num_segments) +
                            std::max(curve_order_bytes(n, num_segments),
                                     fps_align(sizeof(uint32_t) * (size_t)n)));
}

namespace {
hipError_t launch_fps_stream(const float *src, const int64_t *ptr,
                             const int64_t *out_ptr, const int64_t *start,
                             int n, int d, int num_segments, int64_t max_rows,
                             void *scratch, FpsPatience patience, int64_t *out,
                             hipStream_t stream) {
  char *cursor = static_cast<char *>(scratch);
  auto take = [&cursor](size_t bytes) {
    char *piece = cursor;
    cursor += fps_align(bytes);
    return static_cast<void *>(piece);
  };
  FpsPieces p;
  const size_t pieces = (size_t)fps_first_piece(n, num_segments);
  p.rows = static_cast<float4 *>(take(sizeof(float4) * kWave * pieces));
  p.minima = static_cast<float *>(take(sizeof(float) * kWave * pieces));
  p.boxes = static_cast<float *>(take(sizeof(float) * 8 * pieces));
  const int64_t rows = std::min(max_rows, (int64_t)n);
  const int most = fps_share_most(num_segments);
  FpsShare share = {nullptr, nullptr};
  if (most > 0) {
    void *words = take(sizeof(uint64_t) * 2 * kFpsShareWords *
                       (size_t)num_segments);
    void *state = take(sizeof(uint32_t) * (size_t)num_segments);
    int device = 0, units = 0;
    if (rows <= (int64_t)most * 16 * kFpsThreads &&
        hipGetDevice(&device) == hipSuccess &&
        hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount,
                              device) == hipSuccess &&
        units >= kFpsShareGrid)
      share = {static_cast<uint64_t *>(words), static_cast<uint32_t *>(state)};
  }
  const uint32_t *perm = nullptr;
  if (rows <= 16 * kFpsThreads + 1) {
    uint32_t *order = reinterpret_cast<uint32_t *>(cursor);
    perm = order;
    hipLaunchKernelGGL(fps_order_kernel, dim3(num_segments), dim3(kFpsThreads),
                       0, stream, src, ptr, d, order);
  } else {
    hipError_t err = launch_curve_order(src, ptr, n, d, num_segments, cursor,
                                        &perm, stream);
    if (err != hipSuccess)
      return err;
  }
  for (int b0 = 0; b0 < num_segments; b0 += 65535) {
    const int some = std::min(65535, num_segments - b0);
    hipLaunchKernelGGL(fps_gather_kernel,
                       dim3((unsigned)((rows + kBlock - 1) / kBlock), some),
                       dim3(kBlock), 0, stream, src, ptr, d, b0, perm,
                       p, share);
  }
  if (share.words != nullptr) {
#define PCA_FPS_SHARED(R_, S_)                                                 \
  hipLaunchKernelGGL((fps_shared_kernel<R_, S_>), dim3(num_segments *most),    \
                     dim3(kFpsThreads), 0, stream, src, ptr, out_ptr, start,   \
                     d, most, p, share, patience.told, patience.came, out)
    // (rows of a lane at most: with 16 a quarter of the workgroups can do what all do
    // with four; where two rows are enough for all, eight are that many.  The kernel
    // without 16 is the faster one there, calls, us, with / without: 16 x 16,384 rows, a
    // quarter 740 / 730; 16 x 8,000, 1,200 samples 372 / 365)
    if (rows <= (int64_t)most * 2 * kFpsThreads)
      PCA_FPS_SHARED(8, 32);
    else
      PCA_FPS_SHARED(16, 32);
#undef PCA_FPS_SHARED
  }
  // (half as many rows to a bucket where the lanes suffice: 8 x 60,000 rows, 600
  // samples each, R = 1 / 2 910 / 840 us, 8 x 20,000 1,160 / 1,240; the scans, at
  // most 200,000 rows, R = 4 2.8 ms, 2 x 4 2.9)
#define PCA_FPS_STREAM(S_, MANY_, OWN_)                                        \
  hipLaunchKernelGGL((fps_stream_kernel<kFpsWaves, S_, MANY_, OWN_>),          \
                     dim3(num_segments), dim3(kFpsThreads), 0, stream, src,    \
                     ptr, out_ptr, start, d, p, share.state, out)
  if (rows <= 16 * kFpsThreads + 1)
    PCA_FPS_STREAM(1, false, true);
  else if (rows <= kWave * kFpsThreads / 2)
    PCA_FPS_STREAM(1, false, false);
  else if (rows <= kWave * kFpsThreads)
    PCA_FPS_STREAM(2, false, false);
  else if (rows <= 4 * kWave * kFpsThreads)
    PCA_FPS_STREAM(4, false, false);
  else
    PCA_FPS_STREAM(4, true, false);
#undef PCA_FPS_STREAM
  return hipGetLastError();
}
} // namespace

hipError_t launch_fps(int dtype, const void *src, const int64_t *ptr,
                      const int64_t *out_ptr, const int64_t *start, int n,
                      int d, int num_segments, int64_t max_rows, void *scratch,
                      bool captured, int64_t *out, hipStream_t stream,
                      FpsPatience patience) {
  if (fps_on_chip(dtype, d, max_rows)) {
    const float *s = static_cast<const float *>(src);
    if (d <= 2)
      return launch_fps_on_chip<2>(s, ptr, out_ptr, start, d, num_segments,
                                   max_rows, out, stream);
    if (d == 3)
      return launch_fps_on_chip<3>(s, ptr, out_ptr, start, d, num_segments,
                                   max_rows, out, stream);
    return launch_fps_on_chip<4>(s, ptr, out_ptr, start, d, num_segments,
                                 max_rows, out, stream);
  }
  if (fps_streams(dtype, d, max_rows) && !captured)
    return launch_fps_stream(static_cast<const float *>(src), ptr, out_ptr,
                             start, n, d, num_segments, max_rows, scratch,
                             patience, out, stream);
  switch (dtype) {
  case 0:
    return launch_fps_any<FpsF32>(src, ptr, out_ptr, start, d, num_segments,
                                  scratch, out, stream);
  case 1:
    return launch_fps_any<FpsF64>(src, ptr, out_ptr, start, d, num_segments,
                                  scratch, out, stream);
  case 2:
    return launch_fps_any<FpsF16>(src, ptr, out_ptr, start, d, num_segments,
                                  scratch, out, stream);
  default:
    return hipErrorInvalidValue;
  }
}

} // namespace pca
