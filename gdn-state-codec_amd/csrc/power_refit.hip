// Rank-4 window-boundary refit (window_boundary_launch_v1 with
// power_iterations in 1..32; native/ascendc/gdn_state_codec/kernel/
// gdn_state_codec_window_boundary.cpp:253-366).
//
// For a state whose 16-record window is full, the window's residual operator
//   R = boundary * S + old compensators * S + sum_j key_j corr_j^T * suffix_j
// is fitted with four rank-one terms by deflated power iteration (the start
// vector of rank r is ((r+1)(c+3)) mod 17 - 8, normalized with the reference's
// Newton square root, newton_sqrt), stored as fp16 compensators; R minus the fit is then
// re-encoded with fresh smoothing sqrt(mean |row|), absmax scales and
// round-half-away codes, and the window is cleared.
//
// Every dot product of the reference is a sequential fp32 sum; this kernel
// keeps each one on a single thread in the reference's order, so the result is
// bit-identical to the CPU statement of the reference kernel.
//
// One workgroup per state, in two forms (takes_split_form says which):
//   split, 256 threads: threads 0..127 own the key rows and 128..255 the value
//     columns, each with its line's 128 boundary values code / 127 * s * scale
//     in VGPRs (168, so three states per CU).  An operator application sums on
//     the side that owns its outputs, while a wavefront of the other side forms
//     the 24 projections of the compensators, records and fitted ranks.
//   whole, 128 threads: thread t owns row t and column t, with their codes in
//     64 VGPRs and the first 48 of the row's values in 48 more; the other
//     values are formed again in every application (eight instructions a value
//     instead of three).  Five states per CU (31,920 bytes of LDS each).
// In both one wavefront sums a vector's squared norm and normalizes it.  The
// chains of one state bound the kernel when there are few states (per
// application 128 products and adds, 24 more terms and 128 adds), VALU issue
// when there are many.  The fitted residual is evaluated once per cell, one key
// row per thread held in registers for the smoothing, scale and code passes,
// and written once to the workspace.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "pipelined_sum.h"
#include "codec_math.h"
#include "gdn_state_codec_window.h"
#include "lane_exchange.h"
#include "launch.h"
#include "window_common.h"

namespace gdn {
namespace {

constexpr int kThreads = 128;       // one thread per row (and column)
constexpr int kSplitThreads = 256;  // one thread per row, one per column
constexpr int kCodeStride = kDim + 4;
constexpr float kBoundaryFloor = 1.0e-8f;
// The split form up to one round of the chip, and with two iterations or more
// wherever it takes no more rounds than the whole one, its round being the
// shorter: from 1,281 to 1,536 states.  Split / whole form with the window's 16
// steps (before both, with each value formed from LDS by a thread for row and
// column), us, 4 iterations: 512 states 319 / 377 (427), 768 332 / 387 (432),
// 800 478 / 399 (439), 1,280 571 / 514 (554), 1,282 580 / 647, 1,408 590 / 660
// (777), 1,536 598 / 663 (779), 1,792 750 / 760 (837), 2,048 794 / 778 (868),
// 2,304 876 / 857 (937), 4,096 1,521 / 1,373 (1,567), 8,192 2,876 / 2,543
// (2,866).  1,536 states with 1 iteration 429 / 425 (472), with 2 490 / 508, with
// 16 1,287 / 1,649 (2,006).
constexpr uint32_t kSplitRound = 3 * 256;
constexpr uint32_t kWholeRound = 5 * 256;
constexpr bool takes_split_form(uint32_t states, uint32_t iterations) {
  return states <= kSplitRound ||
         (iterations > 1 && (states + kSplitRound - 1) / kSplitRound <=
                                (states + kWholeRound - 1) / kWholeRound);
}

// In the form with codes in registers, the values of a row's first columns are
// held as well: what three wavefronts per SIMD leave of the registers.  Such a
// value costs an application three VALU instructions, one formed from its code
// eight.  8,192 states, 4 iterations, with the window's 16 steps: 2,660 us with
// none held, 2,555 with 48, 2,606 with 64 and 2,729 with 80, where more values
// are spilled (11, 19 and 35 VGPRs).
constexpr int kHeldCells = 48;

// f(std::integral_constant<int, c>) for c = 0 .. kDim - 1, expanded at compile
// time: a body that indexes a register array by c keeps the array in VGPRs,
// where a loop the compiler declines to unroll fully would move it to scratch.
template <int kColumn = 0, typename F>
__device__ __forceinline__ void each_column(F&& f) {
  if constexpr (kColumn < kDim) {
    f(std::integral_constant<int, kColumn>{});
    each_column<kColumn + 1>(f);
  }
}

struct PowerArgs {
  const int8_t* residual;
  const float* smoothing;
  const float* scales;
  const uint16_t* comp_keys;
  const uint16_t* comp_values;
  float* record_decay;
  uint16_t* record_keys;
  uint16_t* record_corrections;
  uint32_t* positions;
  int8_t* next_residual;
  float* next_smoothing;
  float* next_scales;
  uint16_t* next_comp_keys;
  uint16_t* next_comp_values;
  float* workspace;
  uint32_t power_iterations;
};

// Compensators and records are fp16 values (the fitted ranks are rounded to
// fp16 when formed), so they are kept as fp16 bits and widened exactly when
// read: 31,920 bytes, five workgroups per CU.
struct PowerShared {
  int8_t code[kDim * kCodeStride];  // [value column][key row]
  alignas(8) uint16_t ck[kDim * kRank];
  alignas(8) uint16_t cv[kDim * kRank];
  alignas(8) uint16_t nk[kDim * kRank];
  alignas(8) uint16_t nv[kDim * kRank];
  // Records as [dimension][record]: a dimension's 16 records are 32
  // contiguous bytes, so the record projections (lane j walks record j)
  // read consecutive words and a cell reads its 16 records as two 16-byte
  // words.
  alignas(16) uint16_t rk[kDim * kWindow];
  alignas(16) uint16_t rc[kDim * kWindow];
  float smoothing[kDim], scales[kDim];
  alignas(16) float left[kDim];
  alignas(16) float right[kDim];
  alignas(16) float square[kDim];  // of the vector just formed, for its norm
  // The projections of an application: old ranks, fitted ranks, records.
  alignas(16) float projection[2 * kRank + kWindow];
  alignas(16) float record_suffix[kWindow];
  float scalar;  // the singular value
  int flag;      // whether the vector could be normalized
};
static_assert(workgroups_by_lds(sizeof(PowerShared)) >= 5, "five workgroups per CU");

// code / 127 by the two-part division (div_by_127, exact for every integer in
// [-128, 127]): two VALU instructions, where a table of the 256 quotients
// would cost a second LDS read whose address depends on the first.
__device__ __forceinline__ float code_value_arith(int8_t code) {
  return div_by_127(static_cast<float>(code));
}

// The sequential sum of sh.square, evaluated identically by every lane.
__device__ __forceinline__ float squared_norm(const PowerShared& sh) {
  float squared = 0.0f;
  struct Group {
    float x[16];
  };
  pipelined<kDim / 16, Group>(
      [&](auto g, Group& r) {
        unrolled<4>([&](auto q) {
          *reinterpret_cast<float4*>(r.x + 4 * decltype(q)::value) =
              *reinterpret_cast<const float4*>(sh.square + 16 * decltype(g)::value +
                                               4 * decltype(q)::value);
        });
      },
      [&](auto, const Group& r) { unrolled<16>([&](auto i) { squared += r.x[i]; }); });
  return squared;
}

// Normalize (:25-37) of `vector` by one wavefront; a vector whose norm is not
// usable stays as it is.
__device__ __forceinline__ void normalize(PowerShared& sh, float* vector, int lane) {
  const float squared = squared_norm(sh);
  const bool ok = !(squared <= 1.0e-20f);
  if (ok) {
    const float inverse = 1.0f / newton_sqrt(squared);
    vector[lane] *= inverse;
    vector[64 + lane] *= inverse;
  }
  if (lane == 0) sh.flag = ok ? 1 : 0;
}

// The projections of an application (old compensator side, fitted ranks,
// records) by one wavefront: one sequential sum per lane in the reference's
// loop order, a product of an fp16 and an fp32 value being one v_fma_mix_f32
// (adding -0 changes nothing).  Ranks not fitted yet are zero in LDS and their
// sums are not used.
__device__ __forceinline__ void projections(PowerShared& sh, const float* vector,
                                            const uint16_t* old_basis,
                                            const uint16_t* record_basis,
                                            const uint16_t* fitted_basis, int lane) {
  if (lane >= 2 * kRank + kWindow) return;
  const uint16_t* const basis = lane < kRank ? old_basis + lane
                                : lane < 2 * kRank ? fitted_basis + (lane - kRank)
                                                   : record_basis + (lane - 2 * kRank);
  const int stride = lane < 2 * kRank ? kRank : kWindow;
  const float neg_zero = opaque_negative_zero();
  float acc = 0.0f;
  struct Group {
    float x[8];
    uint16_t b[8];
  };
  Group now, ahead;
  const auto load = [&](int i, Group& g) {
    *reinterpret_cast<float4*>(g.x) = *reinterpret_cast<const float4*>(vector + i);
    *reinterpret_cast<float4*>(g.x + 4) = *reinterpret_cast<const float4*>(vector + i + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) g.b[e] = basis[(i + e) * stride];
  };
  load(0, now);
#pragma unroll 2
  for (int i = 0; i < kDim; i += 8) {
    load((i + 8) & (kDim - 1), ahead);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      acc += __builtin_fmaf(half_bits_to_float(now.b[e]), now.x[e], neg_zero);
    }
    now = ahead;
  }
  sh.projection[lane] = acc;
}

// The sum of an application's boundary part (:113-142, :168-197) over a line's
// values: value = ((code / 127 * s) * scale) * vector * bs, in order.
__device__ __forceinline__ float line_sum(const float (&cell)[kDim], const float* vector,
                                          float bs) {
  float value = 0.0f;
  struct Group {
    float x[8];
  };
  pipelined<kDim / 8, Group>(
      [&](auto g, Group& r) {
        constexpr int first = 8 * decltype(g)::value;
        *reinterpret_cast<float4*>(r.x) = *reinterpret_cast<const float4*>(vector + first);
        *reinterpret_cast<float4*>(r.x + 4) = *reinterpret_cast<const float4*>(vector + first + 4);
      },
      [&](auto g, const Group& r) {
        unrolled<8>([&](auto i) {
          value += cell[8 * decltype(g)::value + decltype(i)::value] * r.x[i] * bs;
        });
      });
  return value;
}

// The same sum with the line's codes packed four to a word in place of its
// values, but for the first kHeld of them, which are in held[]; `own` is the
// line's factor, `across` the other axis' factors, and `rows` tells which of
// the two is the smoothing (code / 127 * s * scale).
template <bool kRows, int kHeld>
__device__ __forceinline__ float code_sum(const float (&held)[kDim],
                                          const uint32_t (&codes)[kDim / 4], const float* vector,
                                          const float* across, float own, float bs) {
  static_assert(kHeld % 4 == 0, "whole code words");
  float value = 0.0f;
  struct Group {
    float x[4], f[4];
  };
  pipelined<kDim / 4, Group>(
      [&](auto g, Group& r) {
        constexpr int first = 4 * decltype(g)::value;
        *reinterpret_cast<float4*>(r.x) = *reinterpret_cast<const float4*>(vector + first);
        if constexpr (first >= kHeld) {
          *reinterpret_cast<float4*>(r.f) = *reinterpret_cast<const float4*>(across + first);
        }
      },
      [&](auto g, const Group& r) {
        if constexpr (4 * decltype(g)::value < kHeld) {
          unrolled<4>([&](auto i) {
            value += held[4 * decltype(g)::value + decltype(i)::value] * r.x[i] * bs;
          });
          return;
        }
        // Opaque, so that the widened codes are not formed once for all
        // applications and held (spilled) between them.
        uint32_t word = codes[decltype(g)::value];
        asm volatile("" : "+v"(word));
        unrolled<4>([&](auto i) {
          constexpr int b = decltype(i)::value;
          const float code = code_value_arith(static_cast<int8_t>(word >> (8 * b)));
          const float cell = kRows ? code * own * r.f[b] : code * r.f[b] * own;
          value += cell * r.x[b] * bs;
        });
      });
  return value;
}

// The rest of an application for line `line` (:143-165, :198-220): the old
// compensators, the records, less the fitted ranks.
__device__ __forceinline__ float line_terms(const PowerShared& sh, float value, int line,
                                            const uint16_t* old_basis,
                                            const uint16_t* record_basis,
                                            const uint16_t* fitted_basis, float bs, int fitted) {
  const float neg_zero = opaque_negative_zero();
  const auto half = [](uint32_t pair, int i) { return i & 1 ? pair >> 16 : pair; };
  const auto times = [&](uint32_t bits, float x) {
    return __builtin_fmaf(half_bits_to_float(bits), x, neg_zero);
  };
  const uint2 old2 = *reinterpret_cast<const uint2*>(old_basis + line * kRank);
  const uint2 new2 = *reinterpret_cast<const uint2*>(fitted_basis + line * kRank);
  const uint4 r0 = reinterpret_cast<const uint4*>(record_basis + line * kWindow)[0];
  const uint4 r1 = reinterpret_cast<const uint4*>(record_basis + line * kWindow)[1];
  const uint32_t olds[2] = {old2.x, old2.y}, news[2] = {new2.x, new2.y};
  const uint32_t records[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
  for (int r = 0; r < kRank; ++r) value += times(half(olds[r / 2], r), sh.projection[r]) * bs;
#pragma unroll
  for (int j = 0; j < kWindow; ++j) {
    value += times(half(records[j / 2], j), sh.projection[2 * kRank + j]) * sh.record_suffix[j];
  }
#pragma unroll
  for (int r = 0; r < kRank; ++r) {
    if (r < fitted) value -= times(half(news[r / 2], r), sh.projection[kRank + r]);
  }
  return value;
}

// The re-encode of R minus the fit, for 128 threads of a workgroup (those with
// `active`, whole wavefronts; the others only meet its barriers) whose LDS
// holds the state (codes [value column][key row] at kCodeStride, the old
// and fitted compensators ck / cv / nk / nv [dim][rank], the records rk / rc
// [dim][record], smoothing, scales and record suffixes).  With kFromCodes the
// boundary values come from the codes in LDS, else cell[] holds them already.
// Thread t owns key row t, whose 128 fitted cells stay in registers through
// the smoothing, scale and code passes.  Writes the fitted residual to
// workspace [key row][value column], next_smoothing[key], next_scales[value],
// and hands every code of row t to sink(integral_constant column, code).  Each
// cell is the reference's ResidualCell (window_boundary.cpp:223-251;
// encoded_requantize.cpp:72-100 is the same expression), evaluated in its
// order.  The column loops are unrolled at compile time (each_column) so that
// cell[] is only ever indexed by constants and lives in VGPRs.  Uses sh.left
// and sh.right as scratch for the column maxima.
template <bool kFromCodes, typename Sink>
__device__ __forceinline__ void reencode_rows(PowerShared& sh, float (&cell)[kDim], bool active,
                                              float bs, int t, float* workspace,
                                              float* next_smoothing, float* next_scales,
                                              Sink&& sink) {
  const int row = t;
  if (active) {
    {
      // The row's operands stay as fp16 pairs (widened where used) and the
      // window suffix products, the same for every thread, in scalar
      // registers, leaving the vector registers to the cells.
      [[maybe_unused]] const float s = sh.smoothing[row];
      uint32_t ck2[kRank / 2], nk2[kRank / 2], rk2[kWindow / 2];
      float suffix[kWindow];
#pragma unroll
      for (int i = 0; i < kRank / 2; ++i) {
        ck2[i] = reinterpret_cast<const uint32_t*>(sh.ck + row * kRank)[i];
        nk2[i] = reinterpret_cast<const uint32_t*>(sh.nk + row * kRank)[i];
      }
#pragma unroll
      for (int i = 0; i < kWindow / 2; ++i) rk2[i] = reinterpret_cast<const uint32_t*>(sh.rk + row * kWindow)[i];
#pragma unroll
      for (int j = 0; j < kWindow; ++j) {
        suffix[j] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(sh.record_suffix[j])));
      }
      // Every compensator and record product is of two fp16 values, exact in
      // fp32: one v_fma_mix_f32 each (half_product), and the fitted ranks'
      // `value -= nk * nv` one fma (minus_half_product), the reference's
      // roundings throughout.
      const float neg_zero = opaque_negative_zero();
      const auto half = [](uint32_t pair, int i) { return i & 1 ? pair >> 16 : pair; };
      // A column's LDS operands; the next column's are read while this one's
      // cell is evaluated, so their latency overlaps the arithmetic.
      struct Operands {
        int code;     // with kFromCodes
        float scale;  // with kFromCodes
        uint2 cv, nv;
        uint4 r0, r1;
      };
      const auto fetch = [&](int column) {
        Operands o;
        if constexpr (kFromCodes) {
          o.code = sh.code[column * kCodeStride + row];
          o.scale = sh.scales[column];
        }
        o.cv = *reinterpret_cast<const uint2*>(sh.cv + column * kRank);
        o.nv = *reinterpret_cast<const uint2*>(sh.nv + column * kRank);
        const uint4* const rc4 = reinterpret_cast<const uint4*>(sh.rc + column * kWindow);
        o.r0 = rc4[0];
        o.r1 = rc4[1];
        return o;
      };
      Operands next = fetch(0);
      each_column([&](auto c) {
        constexpr int column = decltype(c)::value;
        // Opaque to the compiler, so the pairs stay packed in registers.
#pragma unroll
        for (int i = 0; i < kRank / 2; ++i) asm volatile("" : "+v"(ck2[i]), "+v"(nk2[i]));
#pragma unroll
        for (int i = 0; i < kWindow / 2; ++i) asm volatile("" : "+v"(rk2[i]));
        const Operands o = next;
        if constexpr (column + 1 < kDim) next = fetch(column + 1);
        // Issued here, ahead of this column's arithmetic, not sunk to its end.
        __builtin_amdgcn_sched_barrier(0);
        // code / 127 by the two-part division (exact for every integer code).
        float value;
        if constexpr (kFromCodes) {
          value = code_value_arith(static_cast<int8_t>(o.code)) * s * o.scale * bs;
        } else {
          value = cell[column] * bs;
        }
        const uint32_t cvp[kRank / 2] = {o.cv.x, o.cv.y}, nvp[kRank / 2] = {o.nv.x, o.nv.y};
#pragma unroll
        for (int r = 0; r < kRank; ++r) {
          value += half_product(half(ck2[r / 2], r), half(cvp[r / 2], r), neg_zero) * bs;
          value = minus_half_product(value, half(nk2[r / 2], r), half(nvp[r / 2], r));
        }
        const uint32_t rc2[kWindow / 2] = {o.r0.x, o.r0.y, o.r0.z, o.r0.w,
                                           o.r1.x, o.r1.y, o.r1.z, o.r1.w};
#pragma unroll
        for (int j = 0; j < kWindow; ++j) {
          value += half_product(half(rk2[j / 2], j), half(rc2[j / 2], j), neg_zero) * suffix[j];
        }
        cell[column] = value;
        // One column ahead at a time: the scheduler would otherwise hoist the
        // LDS reads of many columns ahead of their use.
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    {
      float4* const work = reinterpret_cast<float4*>(workspace + row * kDim);
#pragma unroll
      for (int q = 0; q < kDim / 4; ++q) {
        work[q] = make_float4(cell[4 * q], cell[4 * q + 1], cell[4 * q + 2], cell[4 * q + 3]);
      }
    }

    // ---- fresh smoothing (row t): sequential sum of |cell| over the columns ----
    float s_new;
    {
      float mean_absolute = 0.0f;
      each_column([&](auto c) { mean_absolute += fabsf(cell[decltype(c)::value]); });
      const float mean = mean_absolute / 128.0f;
      s_new = newton_sqrt(mean > kBoundaryFloor ? mean : kBoundaryFloor);
      next_smoothing[row] = s_new;
    }
    // From here on cell[] holds m = cell / s_new (the cells themselves are in the
    // workspace already): the scale pass divides once and stores m in place.

    // ---- scales: max over rows of |cell / s| per column -------------------------
    // The reference keeps `value > maximum ? value : maximum` from 0 over the
    // rows, which skips NaNs; fmaxf(|m|, 0) maps a NaN to 0 and leaves every
    // other |m| alone, and a maximum of those is exact in any order.  Each
    // wavefront reduces its 64 rows with quarter-width reduce-scatters (32
    // columns across 64 lanes: lane L ends with column L % 32), then the two
    // wavefronts' maxima meet in LDS.
    const int lane = t & 63;
    const int wave = t >> 6;
#pragma unroll
    for (int quarter = 0; quarter < 4; ++quarter) {
#pragma unroll
      for (int i = 0; i < 32; ++i) cell[32 * quarter + i] = cell[32 * quarter + i] / s_new;
      const auto magnitude = [&](int i) { return fmaxf(fabsf(cell[32 * quarter + i]), 0.0f); };
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float lo = fold_max<16>(magnitude(i), magnitude(16 + i), lane);
        const float hi = fold_max<16>(magnitude(8 + i), magnitude(24 + i), lane);
        v[i] = fold_max<8>(lo, hi, lane);
        if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = fold_max<4>(v[i], v[i + 4], lane);
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = fold_max<2>(v[i], v[i + 2], lane);
      v[0] = fold_max<1>(v[0], v[1], lane);
      v[0] = max_partner<32>(v[0]);
      if (lane < 32) {
        (wave == 0 ? sh.left : sh.right)[32 * quarter + lane] = v[0];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // both wavefronts' column maxima; every cell has been evaluated
  if (active) {
    // Thread t's own slots: no other thread reads them before the barrier.
    const float maximum = fmaxf(sh.left[t], sh.right[t]);
    next_scales[t] = maximum;
    sh.left[t] = maximum;
    // The certified codes' factor RN(127 / maximum) (code_lift in codec_math.h)
    // for a maximum of 0 or in [2^-90, 2^90]; NaN otherwise, which sends every
    // cell of the column to the exact path below.
    sh.right[t] = maximum == 0.0f ? 0.0f
                  : (maximum >= 0x1p-90f && maximum <= 0x1p90f) ? kQuantizedMaximum / maximum
                                                                : __builtin_nanf("");
  }
  __syncthreads();

  // ---- codes: round-half-away (:336-345), handed to the caller's sink ------
  // The reference's q = m / maximum * 127, then trunc(q +- 0.5) clamped to
  // +-127.  Where the lift u = fma(m, RN(127 / maximum), 0.5 + 2^-14) has a
  // fraction of at least 2^-13, q + 0.5 lies at least 2^-15 inside
  // (floor(u), floor(u) + 1), so the rounded q +- 0.5 truncates to floor(u)
  // (the certificate of codec_math.h; |m| <= maximum since the maximum is
  // over these same m).  The other cells, NaN and infinite ones among them,
  // take the reference's expression.
  if (!active) return;
  each_column([&](auto c) {
    constexpr int column = decltype(c)::value;
    const float m = cell[column];
    const float u = code_lift(m, sh.right[column]);
    int code;
    if (lift_fraction(u) >= kCodeLiftMargin) {
      code = lifted_code(u);
    } else {
      const float maximum = sh.left[column];
      float q = maximum == 0.0f ? 0.0f : m / maximum * 127.0f;
      q += q >= 0.0f ? 0.5f : -0.5f;
      q = q > 127.0f ? 127.0f : q;
      q = q < -127.0f ? -127.0f : q;
      code = static_cast<int>(q);
    }
    sink(c, static_cast<int8_t>(code));
    if constexpr (column % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  });
}

template <bool kSplit>
__global__ __launch_bounds__(kSplit ? kSplitThreads : kThreads) __attribute__((amdgpu_waves_per_eu(3))) void power_refit_kernel(PowerArgs a) {
  constexpr int kFitThreads = kSplit ? kSplitThreads : kThreads;
  extern __shared__ __align__(16) unsigned char dynamic[];
  PowerShared& sh = *reinterpret_cast<PowerShared*>(dynamic);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int line = t & (kDim - 1);   // the thread's row or column
  const bool rows = !kSplit || wave < 2;     // it owns a key row,
  const bool columns = !kSplit || wave > 1;  // a value column
  const uint64_t state = blockIdx.x;
  if (a.positions[state * kPositionStride] != static_cast<uint32_t>(kWindow)) return;  // uniform
  const uint64_t vb = state * kDim;
  const uint64_t rb = state * kWindow;

  // ---- stage the state in LDS -----------------------------------------------
  for (int i = t; i < kTile / 4; i += kFitThreads) {
    const uint32_t w = reinterpret_cast<const uint32_t*>(a.residual + state * kTile)[i];
    const int column = (4 * i) / kDim, row = (4 * i) % kDim;
    *reinterpret_cast<uint32_t*>(&sh.code[column * kCodeStride + row]) = w;
  }
  for (int i = t; i < kDim * kRank; i += kFitThreads) {
    sh.ck[i] = a.comp_keys[vb * kRank + i];
    sh.cv[i] = a.comp_values[vb * kRank + i];
    sh.nk[i] = 0u;
    sh.nv[i] = 0u;
  }
  for (int i = t; i < kWindow * kDim; i += kFitThreads) {
    const int j = i / kDim, dimension = i % kDim;
    sh.rk[dimension * kWindow + j] = a.record_keys[rb * kDim + i];
    sh.rc[dimension * kWindow + j] = a.record_corrections[rb * kDim + i];
  }
  if (rows) sh.smoothing[line] = (a.smoothing + vb)[line];
  if (columns) sh.scales[line] = (a.scales + vb)[line];
  // BuildSuffix (:102-111), computed identically by every thread.
  float bs = 1.0f;
  for (int j = kWindow - 1; j >= 0; --j) {
    if (t == 0) sh.record_suffix[j] = bs;
    bs *= a.record_decay[rb + j];
  }
  // The same value in every lane: keep it in a scalar register.
  bs = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(bs)));
  __syncthreads();

  // ---- the lines' boundary values (code / 127 * s * scale), or their codes ----
  float cell[kDim];
  uint32_t row_codes[kDim / 4], column_codes[kDim / 4];
  if constexpr (!kSplit) {
    each_column([&](auto c) {
      constexpr int column = decltype(c)::value;
      const uint32_t code = static_cast<uint8_t>(sh.code[column * kCodeStride + line]);
      row_codes[column / 4] =
          column % 4 == 0 ? code : row_codes[column / 4] | (code << (8 * (column % 4)));
      if constexpr (column % 4 == 0) {
        column_codes[column / 4] =
            *reinterpret_cast<const uint32_t*>(&sh.code[line * kCodeStride + column]);
      }
      if constexpr (column < kHeldCells) {
        cell[column] = code_value_arith(static_cast<int8_t>(code)) * sh.smoothing[line] *
                       sh.scales[column];
      }
    });
  } else if (rows) {
    const float s = sh.smoothing[line];
    each_column([&](auto c) {
      constexpr int column = decltype(c)::value;
      cell[column] = code_value_arith(sh.code[column * kCodeStride + line]) * s * sh.scales[column];
      if constexpr (column % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    });
  } else {
    const float scale = sh.scales[line];
    each_column([&](auto c) {
      constexpr int row = decltype(c)::value;
      cell[row] = code_value_arith(sh.code[line * kCodeStride + row]) * sh.smoothing[row] * scale;
      if constexpr (row % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    });
  }

  // ---- deflated power iteration ---------------------------------------------
  // ApplyRight (:113-166, forward: right vector in, one row's sum out) and
  // ApplyTranspose (:168-221): the sums on the side that owns the outputs, the
  // projections in a wavefront of the other side; the result and its squares
  // are published by the last barrier.
  const auto apply = [&](bool forward, int fitted) {
    const float* const in = forward ? sh.right : sh.left;
    float* const out = forward ? sh.left : sh.right;
    const bool own = forward ? rows : columns;
    float value = 0.0f;
    // Split: a wavefront of the other side, while this one sums.
    if (wave == (kSplit ? (forward ? 2 : 0) : (forward ? 1 : 0))) {
      projections(sh, in, forward ? sh.cv : sh.ck, forward ? sh.rc : sh.rk,
                  forward ? sh.nv : sh.nk, lane);
    }
    if (own) {
      if constexpr (kSplit) {
        value = line_sum(cell, in, bs);
      } else if (forward) {
        value = code_sum<true, kHeldCells>(cell, row_codes, in, sh.scales, sh.smoothing[line], bs);
      } else {
        value = code_sum<false, 0>(cell, column_codes, in, sh.smoothing, sh.scales[line], bs);
      }
    }
    __syncthreads();
    if (own) {
      value = line_terms(sh, value, line, forward ? sh.ck : sh.cv, forward ? sh.rk : sh.rc,
                         forward ? sh.nk : sh.nv, bs, fitted);
      out[line] = value;
      sh.square[line] = value * value;
    }
    __syncthreads();
  };
  const auto normalized = [&](float* vector) {
    if (wave == 1) normalize(sh, vector, lane);
    __syncthreads();
    return sh.flag != 0;  // uniform
  };
  for (int rank = 0; rank < kRank; ++rank) {
    if (rows) {
      const float v = static_cast<float>(static_cast<int>(((rank + 1) * (line + 3)) % 17) - 8);
      sh.right[line] = v;
      sh.square[line] = v * v;
    }
    __syncthreads();
    (void)normalized(sh.right);
    for (uint32_t it = 0; it < a.power_iterations; ++it) {
      apply(true, rank);
      if (!normalized(sh.left)) break;
      apply(false, rank);
      if (!normalized(sh.right)) break;
    }
    apply(true, rank);
    if (wave == 1) {
      const float singular = newton_sqrt(squared_norm(sh));
      if (lane == 0) sh.scalar = singular;
    }
    __syncthreads();
    const float singular = sh.scalar;
    if (singular > 1.0e-20f) {
      const float inverse = 1.0f / singular;
      if (rows) {
        sh.nk[line * kRank + rank] =
            static_cast<uint16_t>(float_to_half_bits(sh.left[line] * inverse * singular));
      }
      if (columns) {
        sh.nv[line * kRank + rank] = static_cast<uint16_t>(float_to_half_bits(sh.right[line]));
      }
    }
    __syncthreads();
  }

  // ---- R minus the fit, re-encoded; codes staged in the code area ------------
  // The workspace is written once and never read back.
  reencode_rows<!kSplit>(sh, cell, rows, bs, line, a.workspace + state * kTile,
                       a.next_smoothing + vb, a.next_scales + vb, [&](auto c, int8_t code) {
                         sh.code[decltype(c)::value * kCodeStride + line] = code;
                       });
  __syncthreads();
  // next_residual [value column][key row], eight lanes to a whole 128-byte
  // column.
#pragma unroll
  for (int first = 0; first < kDim; first += kFitThreads / 8) {
    const int column = first + (t >> 3);
    const int offset = 16 * (t & 7);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&sh.code[column * kCodeStride + offset]);
    *reinterpret_cast<uint4*>(a.next_residual + state * kTile + column * kDim + offset) =
        make_uint4(src[0], src[1], src[2], src[3]);
  }

  // ---- new compensators, cleared window, position ----------------------------
  for (int i = t; i < kDim * kRank; i += kFitThreads) {
    a.next_comp_keys[vb * kRank + i] = sh.nk[i];
    a.next_comp_values[vb * kRank + i] = sh.nv[i];
  }
  for (int i = t; i < kWindow * kDim / 2; i += kFitThreads) {
    reinterpret_cast<uint32_t*>(a.record_keys + rb * kDim)[i] = 0u;
    reinterpret_cast<uint32_t*>(a.record_corrections + rb * kDim)[i] = 0u;
  }
  if (t < kWindow) a.record_decay[rb + t] = 0.0f;
  __syncthreads();  // every thread has read the position word above
  if (t == 0) a.positions[state * kPositionStride] = 0u;
}

// ---- encoded_requantize -----------------------------------------------------

struct RequantizeArgs {
  const int8_t* residual;  // [state][row = smoothing axis][column = scale axis]
  const float* smoothing;
  const float* scales;
  const uint16_t* old_left;  // [state][dim][rank]
  const uint16_t* old_right;
  const float* record_decay;
  const uint16_t* record_left;  // [state][record][dim]
  const uint16_t* record_right;
  const uint16_t* new_left;  // [state][rank][dim]
  const uint16_t* new_right;
  int8_t* next_residual;  // [state][row][column]
  float* next_smoothing;
  float* next_scales;
  uint16_t* next_left;  // [state][dim][rank]
  uint16_t* next_right;
  float* workspace;  // [state][row][column]
};

// EncodedRequantize::Process (encoded_requantize.cpp:102-166): the window
// operator minus the committed ranks re-encoded.  The state is staged in the
// power refit's LDS layout (codes transposed to [column][row], the [rank][dim]
// bases to [dim][rank], the records to [dim][record]) and re-encoded by the
// same reencode_rows; the codes go back through the code area to 16-byte
// row stores (168 VGPRs, three wavefronts per SIMD: five workgroups per CU,
// as the LDS allows).
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3))) void encoded_requantize_kernel(
    RequantizeArgs a) {
  extern __shared__ __align__(16) unsigned char dynamic[];
  PowerShared& sh = *reinterpret_cast<PowerShared*>(dynamic);
  const int t = threadIdx.x;
  const uint64_t state = blockIdx.x;
  const uint64_t vb = state * kDim;
  const uint64_t rb = state * kWindow;

  const uint32_t* words = reinterpret_cast<const uint32_t*>(a.residual + state * kTile);
  for (int i = t; i < kTile / 4; i += kThreads) {
    const uint32_t w = words[i];
    const int row = (4 * i) / kDim, column = (4 * i) % kDim;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      sh.code[(column + b) * kCodeStride + row] = static_cast<int8_t>(w >> (8 * b));
    }
  }
  for (int i = t; i < kDim * kRank; i += kThreads) {
    const int dimension = i / kRank, rank = i % kRank;
    sh.ck[i] = a.old_left[vb * kRank + i];
    sh.cv[i] = a.old_right[vb * kRank + i];
    sh.nk[i] = a.new_left[(state * kRank + rank) * kDim + dimension];
    sh.nv[i] = a.new_right[(state * kRank + rank) * kDim + dimension];
  }
  for (int i = t; i < kWindow * kDim; i += kThreads) {
    const int j = i / kDim, dimension = i % kDim;
    sh.rk[dimension * kWindow + j] = a.record_left[rb * kDim + i];
    sh.rc[dimension * kWindow + j] = a.record_right[rb * kDim + i];
  }
  sh.smoothing[t] = (a.smoothing + vb)[t];
  sh.scales[t] = (a.scales + vb)[t];
  // The suffix products (:106-111), computed identically by every thread.
  float bs = 1.0f;
  for (int j = kWindow - 1; j >= 0; --j) {
    if (t == 0) sh.record_suffix[j] = bs;
    bs *= a.record_decay[rb + j];
  }
  bs = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(bs)));
  __syncthreads();

  // The codes of row t, four to a word, staged row-major in the code area
  // (free once every cell has been evaluated; a 132-byte row stride keeps the
  // 64 lanes' word writes in distinct banks), so that only one packed word is
  // live at a time.
  uint32_t quad = 0u;
  float cell[kDim];
  reencode_rows<true>(sh, cell, true, bs, t, a.workspace + state * kTile, a.next_smoothing + vb,
                      a.next_scales + vb, [&](auto c, int8_t code) {
                  constexpr int column = decltype(c)::value;
                  quad |= static_cast<uint32_t>(static_cast<uint8_t>(code)) << (8 * (column % 4));
                  if constexpr (column % 4 == 3) {
                    *reinterpret_cast<uint32_t*>(&sh.code[t * kCodeStride + column - 3]) = quad;
                    quad = 0u;
                  }
                });
  __syncthreads();
  // next_residual [row][column]: each round of 16 rows, eight lanes write one
  // whole 128-byte row.
#pragma unroll
  for (int round = 0; round < kDim / 16; ++round) {
    const int row = 16 * round + (t >> 3);
    const int offset = 16 * (t & 7);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&sh.code[row * kCodeStride + offset]);
    *reinterpret_cast<uint4*>(a.next_residual + state * kTile + row * kDim + offset) =
        make_uint4(src[0], src[1], src[2], src[3]);
  }
  // The committed bases in the [dim][rank] layout: the LDS copies already are.
  for (int i = t; i < kDim * kRank; i += kThreads) {
    a.next_left[vb * kRank + i] = sh.nk[i];
    a.next_right[vb * kRank + i] = sh.nv[i];
  }
}

// The residual workspace of the allocation-free refit entry point: room for
// kNoAllocMaxStates states (32 MiB), one copy per GPU, held by every GPU this
// library runs on until the process ends.  In host code `scratch` names a
// host-side stand-in, never the device array: host code uses only the address
// hipGetSymbolAddress returns for the GPU in question (scratch_on_device).
constexpr uint32_t kNoAllocMaxStates = 512;
static __device__ __align__(256) float scratch[kNoAllocMaxStates * kTile];

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
float* scratch_address[kMaxDevices] = {};

// The device address of `scratch` on the GPU that `stream` runs on, looked up
// once per GPU with that GPU current (and the caller's current GPU restored).
int32_t scratch_on_device(void* stream, float** address) {
  int device = 0;
  if (hipStreamGetDevice(static_cast<hipStream_t>(stream), &device) != hipSuccess ||
      device < 0 || device >= kMaxDevices) {
    return kStatusLaunchFailed;
  }
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_address[device] == nullptr) {
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess) return kStatusLaunchFailed;
    if (current != device && hipSetDevice(device) != hipSuccess) return kStatusLaunchFailed;
    void* found = nullptr;
    const hipError_t status = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
    if (current != device && hipSetDevice(current) != hipSuccess) return kStatusLaunchFailed;
    if (status != hipSuccess || found == nullptr) return kStatusLaunchFailed;
    scratch_address[device] = static_cast<float*>(found);
  }
  *address = scratch_address[device];
  return kStatusOk;
}

}  // namespace

int32_t launch_power_refit(void* stream, const int8_t* residual, const float* smoothing,
                           const float* scales, const uint16_t* comp_keys,
                           const uint16_t* comp_values, float* record_decay,
                           uint16_t* record_keys, uint16_t* record_corrections,
                           uint32_t* positions, int8_t* next_residual, float* next_smoothing,
                           float* next_scales, uint16_t* next_comp_keys,
                           uint16_t* next_comp_values, float* residual_workspace,
                           uint32_t states, uint32_t power_iterations) {
  const PowerArgs args{residual, smoothing, scales, comp_keys, comp_values, record_decay,
                       record_keys, record_corrections, positions, next_residual, next_smoothing,
                       next_scales, next_comp_keys, next_comp_values, residual_workspace,
                       power_iterations};
  void* pointers[] = {const_cast<PowerArgs*>(&args)};
  const bool split = takes_split_form(states, power_iterations);
  const hipError_t status = hipLaunchKernel(
      split ? reinterpret_cast<const void*>(power_refit_kernel<true>)
            : reinterpret_cast<const void*>(power_refit_kernel<false>),
      dim3(states), dim3(split ? kSplitThreads : kThreads), pointers, sizeof(PowerShared),
      static_cast<hipStream_t>(stream));
  return status == hipSuccess ? kStatusOk : kStatusLaunchFailed;
}

int32_t launch_quant_only_refit(void* stream, const int8_t* residual, const float* smoothing,
                                const float* scales, float* record_decay,
                                uint16_t* record_keys, uint16_t* record_corrections,
                                uint32_t* positions, int8_t* next_residual,
                                float* next_smoothing, float* next_scales,
                                uint16_t* next_comp_keys, uint16_t* next_comp_values,
                                uint32_t states);

}  // namespace gdn

// The window-boundary refit without a caller workspace: the power refit's
// fitted residual goes to the library's own scratch array, so the call
// allocates nothing.  Calls that overlap on one GPU share that array and race.
extern "C" int32_t statecentric_gdn_state_codec_window_boundary_noalloc_launch_v1(
    void* stream, const int8_t* residual, const float* smoothing, const float* scales,
    const uint16_t* compensator_keys, const uint16_t* compensator_values,
    float* record_decay, uint16_t* record_keys, uint16_t* record_corrections,
    uint32_t* positions, int8_t* next_residual, float* next_smoothing, float* next_scales,
    uint16_t* next_compensator_keys, uint16_t* next_compensator_values, uint32_t states,
    uint32_t power_iterations) {
  if (!residual || !smoothing || !scales || !compensator_keys || !compensator_values ||
      !record_decay || !record_keys || !record_corrections || !positions || !next_residual ||
      !next_smoothing || !next_scales || !next_compensator_keys || !next_compensator_values ||
      states == 0 || states > gdn::kMaxWindowStates || power_iterations > 32 ||
      (power_iterations > 0 && states > gdn::kNoAllocMaxStates) ||
      !gdn::aligned16(residual, smoothing, scales, compensator_keys, compensator_values,
                      record_decay, record_keys, record_corrections, positions, next_residual,
                      next_smoothing, next_scales, next_compensator_keys,
                      next_compensator_values)) {
    return gdn::kStatusInvalidArgument;
  }
  if (power_iterations == 0) {  // the quant-only refit uses no workspace
    return gdn::launch_quant_only_refit(stream, residual, smoothing, scales, record_decay,
                                        record_keys, record_corrections, positions,
                                        next_residual, next_smoothing, next_scales,
                                        next_compensator_keys, next_compensator_values, states);
  }
  float* workspace = nullptr;
  const int32_t found = gdn::scratch_on_device(stream, &workspace);
  if (found != gdn::kStatusOk) return found;
  return gdn::launch_power_refit(stream, residual, smoothing, scales, compensator_keys,
                                 compensator_values, record_decay, record_keys,
                                 record_corrections, positions, next_residual, next_smoothing,
                                 next_scales, next_compensator_keys, next_compensator_values,
                                 workspace, states, power_iterations);
}

// encoded_requantize_launch_v1 (encoded_requantize.cpp:102-166, admission
// :189-215): every state re-encoded; see the kernel above.
extern "C" int32_t statecentric_gdn_state_codec_encoded_requantize_launch_v1(
    void* stream, const int8_t* residual, const float* smoothing, const float* scales,
    const uint16_t* old_left, const uint16_t* old_right, const float* record_decay,
    const uint16_t* record_left, const uint16_t* record_right, const uint16_t* new_left,
    const uint16_t* new_right, int8_t* next_residual, float* next_smoothing,
    float* next_scales, uint16_t* next_left, uint16_t* next_right,
    float* residual_workspace, uint32_t states) {
  if (!residual || !smoothing || !scales || !old_left || !old_right || !record_decay ||
      !record_left || !record_right || !new_left || !new_right || !next_residual ||
      !next_smoothing || !next_scales || !next_left || !next_right || !residual_workspace ||
      states == 0 || states > gdn::kMaxWindowStates ||
      !gdn::aligned16(residual, smoothing, scales, old_left, old_right, record_decay,
                      record_left, record_right, new_left, new_right, next_residual,
                      next_smoothing, next_scales, next_left, next_right, residual_workspace)) {
    return gdn::kStatusInvalidArgument;
  }
  const gdn::RequantizeArgs args{residual, smoothing, scales, old_left, old_right,
                                 record_decay, record_left, record_right, new_left, new_right,
                                 next_residual, next_smoothing, next_scales, next_left,
                                 next_right, residual_workspace};
  void* pointers[] = {const_cast<gdn::RequantizeArgs*>(&args)};
  const hipError_t status = hipLaunchKernel(
      reinterpret_cast<const void*>(gdn::encoded_requantize_kernel), dim3(states),
      dim3(gdn::kThreads), pointers, sizeof(gdn::PowerShared), static_cast<hipStream_t>(stream));
  return status == hipSuccess ? gdn::kStatusOk : gdn::kStatusLaunchFailed;
}
