// The device rank-4 chain over an encoded boundary, whole, in one launch.
//
// The reference drives this chain from the host, one stage per launch
// (host/gdn_state_codec_encoded_projection_probe.cpp:611-636): for each rank
// r = 0..3 the seed vector is copied in, then `iterations` times the vector
// is projected through the int8 boundary and finished forward and transposed
// (prepare_int8_vector -> int8_cube_matmul -> finish_encoded_projection, with
// r fitted ranks), and the last vector is projected once more and committed
// as rank r (commit_encoded_rank).  Every stage reads and writes [S][128][16]
// device vectors of which one column is used.
//
// Here one 256-thread workgroup owns one state for the whole chain.  The
// state's int8 boundary is read from HBM once, into registers in both
// orientations: threads 0..127 hold row t, threads 128..255 column t - 128 (32
// words each); the bases, records, scales and the vector live in LDS; and each
// stage is the reference's arithmetic in the reference's order, so every output
// is bit-identical to the launch-per-stage chain (the stages are restated from
// the kernels in decode_pair.hip and encoded_rank.hip):
//   prepare : x = fp16(v) * axis, scale = max|x| > 1e-20 ? max|x| / 127 : 1,
//             q = round(x / scale) (add +-0.5, clamp to +-127, truncate);
//   product : p = A q or A^T q, exact in int32 (v_dot4_i32_i8);
//   finish  : the 24 coefficient sums (old ranks, fitted ranks, records) as
//             sequential fp32 sums, the rows' value with the window's gates,
//             the sequential squared norm, its Newton square root and the fp16
//             output v / |v|;
//   commit  : the rows' value written as the rank's left basis (fp16) and as
//             the corrected vector (fp32), the vector as its right basis.
//
// A step is bound by its serial chain and, with eight states per CU, by the
// VALU issue of the stages that use one wavefront, so the four wavefronts take
// different parts of it:
//   1. one wavefront prepares q while another forms the coefficients (both
//      need only the vector);
//   2. the pair of wavefronts whose lines the product runs over forms it and
//      the rows' values, one line per thread, and their squares;
//   3. one wavefront sums the norm and writes the next vector.
// Parts 1 and 3 run on the pair that part 2 leaves free.  2,048 states, 8
// iterations, the chain with its requantize: 529 us with one wavefront
// per sequential stage and the lines split over thread pairs, 418 us so.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "codec_math.h"
#include "gdn_state_codec_window.h"
#include "lane_exchange.h"
#include "launch.h"
#include "pipelined_sum.h"
#include "window_common.h"

namespace gdn {
namespace {

constexpr int kChainThreads = 256;
constexpr int kCoefficientRows = 2 * kRank + kWindow;  // old, fitted, records
constexpr uint32_t kMaxChainIterations = 64;

struct ChainArgs {
  const int8_t* residual;       // [S][128 left][128 right]
  const float* smoothing;       // [S][128] (left axis)
  const float* scales;          // [S][128] (right axis)
  const uint16_t* old_left;     // fp16 [S][128][4]
  const uint16_t* old_right;    // fp16 [S][128][4]
  const float* record_decay;    // [S][16]
  const uint16_t* record_left;  // fp16 [S][16][128]
  const uint16_t* record_right;
  const uint16_t* seeds;        // fp16 [S][4][128]
  uint16_t* new_left;           // fp16 [S][4][128]
  uint16_t* new_right;          // fp16 [S][4][128]
  float* corrected;             // [S][4][128]
  uint32_t iterations;
};

// Side 0 is the right (value / scale) axis, side 1 the left (key / smoothing)
// axis.  A finish with transpose T takes its input on side T and writes on
// side 1 - T; the forward product (T = 0) maps a right-side vector to the
// left side.
// Basis rows are padded to 136 fp16 (68 words): the 24 coefficient lanes, each
// reading 16 bytes of its own row, then start on banks 4c; unpadded 256-byte
// rows put all 24 on one bank.
constexpr int kBasisStride = kDim + 8;

struct ChainShared {
  // basis[side][row][dim], fp16: rows 0..3 the old compensators of that side
  // (transposed from [dim][rank]), 4..7 the fitted ranks, 8..23 the records.
  __attribute__((aligned(16))) uint16_t basis[2][kCoefficientRows][kBasisStride];
  float axis[2][kDim];
  float suffix[kCoefficientRows];  // of each record's coefficient; 1 for the ranks
  float boundary_suffix;           // the whole window's decay product
  __attribute__((aligned(16))) uint16_t vector[kDim];  // the current vector, fp16 bits
  __attribute__((aligned(16))) uint32_t q[kDim / 4];  // the quantized vector
  __attribute__((aligned(16))) float values[kDim];   // the rows' values
  __attribute__((aligned(16))) float squares[kDim];  // and their squares, for the norm
  __attribute__((aligned(16))) float coefficients[kCoefficientRows];
  float dynamic_scale;
};
static_assert(workgroups_by_lds(sizeof(ChainShared)) >= 8, "eight states per CU");

// Vector quantizer rounding of the reference: add +-0.5, clamp, truncate.
__device__ __forceinline__ int chain_round(float value) {
  float r = value + (value >= 0.0f ? 0.5f : -0.5f);
  r = r > 127.0f ? 127.0f : r;
  r = r < -127.0f ? -127.0f : r;
  return static_cast<int>(r);
}

// prepare_int8_vector of the current vector on input side `side`
// (decode_pair.hip prepare_vector_kernel): one wavefront, rows 2l, 2l + 1.
__device__ void chain_prepare(ChainShared& sh, int side, int lane) {
  float x[2];
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int row = 2 * lane + e;
    x[e] = half_bits_to_float(sh.vector[row]) * sh.axis[side][row];
    m = fmaxf(m, fabsf(x[e]));
  }
  m = wave_max_valu(m);
  const float scale = m > 1.0e-20f ? m / 127.0f : 1.0f;
  const uint32_t c0 = static_cast<uint32_t>(chain_round(x[0] / scale)) & 0xFFu;
  const uint32_t c1 = static_cast<uint32_t>(chain_round(x[1] / scale)) & 0xFFu;
  // Rows 2l, 2l + 1 are bytes 2 (l & 1), +1 of word l / 2.
  reinterpret_cast<uint16_t*>(sh.q)[lane] = static_cast<uint16_t>(c0 | (c1 << 8));
  if (lane == 0) sh.dynamic_scale = scale;
}

// The coefficients of a vector on side `in_side`, one per lane 0..23 of one
// wavefront: sequential sums over the vector, the records' times their suffix.
// Each term is an fp16 basis value times an fp16 vector value, a product exact
// in fp32, so `coefficient += b * x` rounds exactly what
// fma(b, x, coefficient) rounds: one v_fma_mix_f32 per term, reading both
// halves of the packed words itself.
__device__ void chain_coefficients(ChainShared& sh, int in_side, int lane) {
  if (lane >= kCoefficientRows) return;
  const uint16_t* const basis = sh.basis[in_side][lane];
  const auto term = [](uint32_t b, uint32_t x, float total) {
    return __builtin_fmaf(half_bits_to_float(b), half_bits_to_float(x), total);
  };
  struct Terms8 {
    uint4 b, x;
  };
  float coefficient = 0.0f;
  pipelined<kDim / 8, Terms8>(
      [&](auto g, Terms8& r) {
        r.b = *reinterpret_cast<const uint4*>(basis + 8 * decltype(g)::value);
        r.x = *reinterpret_cast<const uint4*>(sh.vector + 8 * decltype(g)::value);
      },
      [&](auto, const Terms8& r) {
        coefficient = term(r.b.x, r.x.x, coefficient);
        coefficient = term(r.b.x >> 16, r.x.x >> 16, coefficient);
        coefficient = term(r.b.y, r.x.y, coefficient);
        coefficient = term(r.b.y >> 16, r.x.y >> 16, coefficient);
        coefficient = term(r.b.z, r.x.z, coefficient);
        coefficient = term(r.b.z >> 16, r.x.z >> 16, coefficient);
        coefficient = term(r.b.w, r.x.w, coefficient);
        coefficient = term(r.b.w >> 16, r.x.w >> 16, coefficient);
      });
  sh.coefficients[lane] = coefficient * sh.suffix[lane];
}

// The row's value of finish_encoded_projection / commit_encoded_rank
// (encoded_rank.hip encoded_rows_kernel) from its projection p, on the output
// side, with `ranks` fitted ranks.  A basis value times a coefficient is
// fma(b, c, -0): the rounded product of the widened half in one v_fma_mix_f32.
__device__ __forceinline__ float chain_row(const ChainShared& sh, int out_side, uint32_t ranks,
                                           int row, int p, float neg_zero) {
  float c[kCoefficientRows];
  unrolled<2 * kRank / 4>([&](auto g) {
    const float4 v = *reinterpret_cast<const float4*>(sh.coefficients + 4 * decltype(g)::value);
    c[4 * g] = v.x, c[4 * g + 1] = v.y, c[4 * g + 2] = v.z, c[4 * g + 3] = v.w;
  });
  const auto product = [&](int r, float coefficient) {
    return __builtin_fmaf(half_bits_to_float(sh.basis[out_side][r][row]), coefficient, neg_zero);
  };
  const float boundary_suffix = sh.boundary_suffix;
  float value = static_cast<float>(p) * sh.dynamic_scale / 127.0f * sh.axis[out_side][row] *
                boundary_suffix;
#pragma unroll
  for (int r = 0; r < kRank; ++r) {
    value += product(r, c[r]) * boundary_suffix;
    const float fitted = product(kRank + r, c[kRank + r]);
    value -= static_cast<uint32_t>(r) < ranks ? fitted : 0.0f;  // x - 0 is x for every x
  }
#pragma unroll
  for (int j = 0; j < kWindow; j += 4) {
    const float4 v = *reinterpret_cast<const float4*>(sh.coefficients + 2 * kRank + j);
    value += product(2 * kRank + j, v.x);
    value += product(2 * kRank + j + 1, v.y);
    value += product(2 * kRank + j + 2, v.z);
    value += product(2 * kRank + j + 3, v.w);
  }
  return value;
}

// The end of finish_encoded_projection: the new vector v / |v| in fp16, by one
// wavefront, rows 2l, 2l + 1.
__device__ void chain_normalize(ChainShared& sh, int lane) {
  struct Squares8 {
    float4 a, b;
  };
  float squared_norm = 0.0f;
  pipelined<kDim / 8, Squares8>(
      [&](auto g, Squares8& r) {
        r.a = *reinterpret_cast<const float4*>(sh.squares + 8 * decltype(g)::value);
        r.b = *reinterpret_cast<const float4*>(sh.squares + 8 * decltype(g)::value + 4);
      },
      [&](auto, const Squares8& r) {
        squared_norm += r.a.x;
        squared_norm += r.a.y;
        squared_norm += r.a.z;
        squared_norm += r.a.w;
        squared_norm += r.b.x;
        squared_norm += r.b.y;
        squared_norm += r.b.z;
        squared_norm += r.b.w;
      });
  const float inverse = squared_norm > 1.0e-20f ? 1.0f / newton_sqrt(squared_norm) : 0.0f;
  const float2 v = *reinterpret_cast<const float2*>(sh.values + 2 * lane);
  reinterpret_cast<uint32_t*>(sh.vector)[lane] =
      (float_to_half_bits(v.x * inverse) & 0xFFFFu) | (float_to_half_bits(v.y * inverse) << 16);
}

// Signed byte dot product of the thread's line and q, exact in int32.
__device__ __forceinline__ int chain_dot(const uint32_t (&codes)[kDim / 4], const uint32_t* q) {
  int acc = 0;
#pragma unroll
  for (int i = 0; i < kDim / 4; i += 4) {
    const uint4 qw = *reinterpret_cast<const uint4*>(q + i);
    acc = __builtin_amdgcn_sdot4(static_cast<int>(codes[i]), static_cast<int>(qw.x), acc, false);
    acc = __builtin_amdgcn_sdot4(static_cast<int>(codes[i + 1]), static_cast<int>(qw.y), acc,
                                 false);
    acc = __builtin_amdgcn_sdot4(static_cast<int>(codes[i + 2]), static_cast<int>(qw.z), acc,
                                 false);
    acc = __builtin_amdgcn_sdot4(static_cast<int>(codes[i + 3]), static_cast<int>(qw.w), acc,
                                 false);
  }
  return acc;
}

// Eight waves per SIMD (64 VGPRs): two states per SIMD at a time and 2,048 in
// flight, so 8,192 states run in four full rounds.
__global__ __launch_bounds__(kChainThreads, 8) void encoded_chain_kernel(ChainArgs a) {
  __shared__ ChainShared sh;
  const int t = threadIdx.x;
  const int wave = t >> 6;
  const int lane = t & 63;
  const int pair = t >> 7;            // 0: the rows' wavefronts, 1: the columns'
  const int line = t & (kDim - 1);
  const uint64_t state = blockIdx.x;

  // ---- the boundary in registers, both orientations ------------------------
  // codes[i]: A[line][4i ..+3] in a row's thread, A[4i ..+3][line] in a
  // column's, whose bytes come through LDS, half the tile at a time, staged in
  // the basis area before the bases are loaded.
  const int8_t* const tile = a.residual + state * kTile;
  uint32_t codes[kDim / 4];
  if (pair == 0) {
    const uint4* src = reinterpret_cast<const uint4*>(tile + line * kDim);
#pragma unroll
    for (int i = 0; i < kDim / 16; ++i) {
      const uint4 w = src[i];
      codes[4 * i] = w.x, codes[4 * i + 1] = w.y, codes[4 * i + 2] = w.z, codes[4 * i + 3] = w.w;
    }
  }
  uint8_t* const stage = reinterpret_cast<uint8_t*>(&sh.basis[0][0][0]);
  static_assert(sizeof(sh.basis) >= kDim / 2 * kDim, "staging area");
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (wave == h) {
      uint4* const to = reinterpret_cast<uint4*>(stage + lane * kDim);
#pragma unroll
      for (int i = 0; i < kDim / 16; ++i) {
        to[i] = make_uint4(codes[4 * i], codes[4 * i + 1], codes[4 * i + 2], codes[4 * i + 3]);
      }
    }
    __syncthreads();
    if (pair == 1) {
#pragma unroll
      for (int i = 0; i < kDim / 8; ++i) {
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          word |= static_cast<uint32_t>(stage[(4 * i + j) * kDim + line]) << (8 * j);
        }
        codes[kDim / 8 * h + i] = word;
      }
    }
    __syncthreads();  // the staging area becomes the second half, then the bases
  }

  // ---- bases, records, scales, gates, zero fitted ranks --------------------
  const uint64_t basis_base = state * kDim * kRank;
  const uint64_t record_base = state * kWindow * kDim;
  for (int i = t; i < kDim * kRank; i += kChainThreads) {
    const int dim = i >> 2, r = i & 3;  // [dim][rank] -> [rank][dim]
    sh.basis[0][r][dim] = a.old_right[basis_base + i];
    sh.basis[1][r][dim] = a.old_left[basis_base + i];
    sh.basis[0][kRank + r][dim] = 0;
    sh.basis[1][kRank + r][dim] = 0;
  }
  for (int i = t; i < kWindow * kDim; i += kChainThreads) {
    const int j = i >> 7, dim = i & (kDim - 1);
    sh.basis[0][2 * kRank + j][dim] = a.record_right[record_base + i];
    sh.basis[1][2 * kRank + j][dim] = a.record_left[record_base + i];
  }
  if (t < kDim) {
    sh.axis[0][t] = a.scales[state * kDim + t];
    sh.axis[1][t] = a.smoothing[state * kDim + t];
    sh.vector[t] = a.seeds[state * kRank * kDim + t];
  }
  if (t == kDim) {
    float suffix = 1.0f;
    for (int j = kWindow - 1; j >= 0; --j) {
      sh.suffix[2 * kRank + j] = suffix;
      suffix *= a.record_decay[state * kWindow + j];
    }
    for (int r = 0; r < 2 * kRank; ++r) sh.suffix[r] = 1.0f;
    sh.boundary_suffix = suffix;
  }
  __syncthreads();

  // ---- the chain -----------------------------------------------------------
  const float neg_zero = opaque_negative_zero();
  for (uint32_t rank = 0; rank < static_cast<uint32_t>(kRank); ++rank) {
    const uint32_t steps = 2 * a.iterations + 1;  // forward, transposed, ..., commit
    for (uint32_t step = 0; step < steps; ++step) {
      // Input side 0 forward, 1 transposed; the product's lines are those of
      // pair `side`, the other pair's two wavefronts take the parts beside it,
      // exchanged from one iteration to the next.
      const int side = static_cast<int>(step & 1u);
      const int first = 2 * (1 - side) + static_cast<int>((step >> 1) & 1u);
      const int second = first ^ 1;
      if (wave == first) chain_prepare(sh, side, lane);
      if (wave == second) chain_coefficients(sh, side, lane);
      __syncthreads();
      if (pair == side) {
        const int p = chain_dot(codes, sh.q);
        const float value = chain_row(sh, 1 - side, rank, line, p, neg_zero);
        if (step + 1 < steps) {
          sh.values[line] = value;
          sh.squares[line] = value * value;
        } else {  // commit_encoded_rank, the vector on the right side
          const uint64_t at = (state * kRank + rank) * kDim + line;
          const uint16_t left = static_cast<uint16_t>(float_to_half_bits(value));
          const uint16_t right = sh.vector[line];
          a.corrected[at] = value;
          a.new_left[at] = left;
          a.new_right[at] = right;
          sh.basis[1][kRank + rank][line] = left;
          sh.basis[0][kRank + rank][line] = right;
          if (rank + 1 < static_cast<uint32_t>(kRank)) sh.vector[line] = a.seeds[at + kDim];
        }
      }
      __syncthreads();
      if (step + 1 < steps) {
        if (wave == second) chain_normalize(sh, lane);
        __syncthreads();
      }
    }
  }
}

}  // namespace
}  // namespace gdn

extern "C" int32_t statecentric_gdn_state_codec_encoded_rank_chain_launch_v4(
    void* stream, const int8_t* residual, const float* smoothing, const float* scales,
    const uint16_t* old_left, const uint16_t* old_right, const float* record_decay,
    const uint16_t* record_left, const uint16_t* record_right, const uint16_t* seeds,
    uint16_t* new_left, uint16_t* new_right, float* corrected, uint32_t states,
    uint32_t iterations) {
  if (!residual || !smoothing || !scales || !old_left || !old_right || !record_decay ||
      !record_left || !record_right || !seeds || !new_left || !new_right || !corrected ||
      states == 0 || states > gdn::kMaxWindowStates || iterations == 0 ||
      iterations > gdn::kMaxChainIterations ||
      !gdn::aligned16(residual, smoothing, scales, old_left, old_right, record_decay,
                      record_left, record_right, seeds, new_left, new_right, corrected)) {
    return gdn::kStatusInvalidArgument;
  }
  const gdn::ChainArgs args{residual, smoothing, scales, old_left, old_right, record_decay,
                            record_left, record_right, seeds, new_left, new_right, corrected,
                            iterations};
  return gdn::launch(gdn::encoded_chain_kernel, dim3(states), dim3(gdn::kChainThreads), stream,
                     args);
}
