// The exact-SVD boundary initializer: the reference runtime's
// GdnStateCodecRuntime._encode_dense_boundary(dense, "exact_svd")
// (src/gdn_state_codec/runtime.py:335-389), which takes the rank-4 truncated
// SVD of each dense [key][value] head D with torch.linalg.svd,
//   compensator_keys[k][r] = U[k][r] * S[r],   compensator_values[v][r] = V[v][r]
// (r = 0..3 by decreasing singular value, stored as fp16), quantizes the fp32
// residual D - keys * values^T and stores the codes in [value][key] order.
//
// Two kernels share the work, both in double up to their outputs.  The direct
// form (Gram matrix, Householder tridiagonal form, the four largest
// eigenpairs; described at its kernel) serves every head but those it marks
// (rows orthogonal from the start, an eigenpair not at rounding level), which
// the Jacobi form behind it takes; a caller's own sweep limit means Jacobi
// throughout.
//
// The decomposition is unique only up to the signs of each (u, v) pair and,
// for equal singular values, the basis of their subspace; the product
// keys * values^T, which is all the codec uses, is not.  The residual then
// goes through the batched quant-only encode (codec.hip) in the provider
// layout.
//
// The Jacobi form is a one-sided (Hestenes) iteration on the provider tile
// P = D^T ([value][key], as the runtime holds it): rotating pairs of P's rows
// until every pair is orthogonal turns row v into u_v * s_v, so the four rows
// of largest norm are the four left singular vectors times their singular
// values, i.e. the compensator keys, and the matching right singular vectors
// are D^T u = P w, normalized.
//
// One 512-thread workgroup per head.  The 128 rows live in LDS in double
// (stride 130, so every row starts 16-byte aligned; 130 KiB, one workgroup
// per CU).  A sweep visits every pair of rows once in 127 rounds of 64
// disjoint pairs (the round-robin tournament: in round r, row 127 meets row r
// and row (r + p) mod 127 meets (r - p) mod 127 for p = 1..63); eight lanes
// serve one pair, each holding 16 values of both rows.  The time is the
// rounds' dependent latency, not issue: two waves per SIMD and short sums
// (two accumulators per lane) hide part of it.  The rotation follows
// Rutishauser's formula for the smaller angle.  Everything up to the outputs
// is double: with fp32 rows the rounding of the rotations, amplified by the
// gap between the fourth and fifth singular values (1-5% on Gaussian heads),
// left the rank-4 product 1e-5..6e-5 of the largest singular value off; in
// double it is the fp32 rounding of the outputs.  Before the sweeps the head
// is scaled by a power of two so that its largest magnitude lies in [1/2, 1),
// and the scaling is undone exactly on the keys.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "gdn_state_codec_kernel.h"
#include "lane_exchange.h"
#include "launch.h"
#include "window_common.h"
#include "work_order.h"

namespace gdn {
namespace {

constexpr int kSvdThreads = 512;
constexpr int kLanesPerPair = 8;
constexpr int kSvdRowStride = kDim + 2;  // doubles
constexpr int kRounds = kDim - 1;          // rounds per sweep (128 rows, odd 127)
constexpr int kSpan = kDim / kLanesPerPair;  // values of a row per lane
constexpr int kMaxSweeps = 30;
constexpr int kSvdRank = 4;
constexpr uint64_t kCus = 256;
// A pair is rotated when its cosine exceeds 2^-36; this converges in 10-13
// sweeps on the test heads.
constexpr double kCosineTolerance = 0x1p-36;
// Rows whose squared norm (after scaling) is below 2^-96 -- every value below
// 2^-48 of the head's largest -- are taken as converged: their share of any
// singular value is below the fp32 rounding of the outputs.
constexpr double kNegligibleSquare = 0x1p-96;

// Per-head outcomes written to `status`.
constexpr int32_t kSvdOk = 0;
constexpr int32_t kSvdNonFiniteInput = 1;
constexpr int32_t kSvdNotConverged = 2;  // a rotation still happened in the last sweep
// Between the two kernels of a call: the head is left to the Jacobi kernel.
constexpr int32_t kSvdPending = -1;

struct SvdArgs {
  const float* provider;   // [heads][value][key]
  float* residual;         // [heads][value][key]
  uint16_t* keys;          // fp16 [heads][key][4]
  uint16_t* values;        // fp16 [heads][value][4]
  int32_t* status;         // [heads]
  uint64_t heads;
  int max_sweeps;          // 1..kMaxSweeps
  bool pending_only;       // Jacobi: only the heads the direct form left
};

struct SvdShared {
  double w[kDim * kSvdRowStride];  // the rows being orthogonalized
  double norm[kDim];              // their squared norms after the sweeps
  double y[kSvdRank][kDim];       // P w_r for the four selected rows
  double y_norm[kSvdRank];
  float right[kDim][kSvdRank];
  float wave_max[kSvdThreads / 64];
  uint64_t pending[kSvdThreads / 64];
  int top[kSvdRank];
};

// x * 2^-exponent in double (exact for every fp32 x).
__device__ __forceinline__ double scaled(float x, int exponent) {
  return ldexp(static_cast<double>(x), -exponent);
}

// One head by Jacobi sweeps; every thread of the workgroup.
__device__ void jacobi_head(SvdShared& sh, const SvdArgs& a, uint64_t head, int t) {
  const float* const p = a.provider + head * kTile;

  // ---- load, finiteness, largest magnitude --------------------------------
  constexpr int kLoads = kTile / 4 / kSvdThreads;  // 8 float4 per thread
  float4 v[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) v[i] = reinterpret_cast<const float4*>(p)[i * kSvdThreads + t];
  bool finite = true;
  float largest = 0.0f;
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    finite = finite && isfinite(v[i].x) && isfinite(v[i].y) && isfinite(v[i].z) &&
             isfinite(v[i].w);
    largest = fmaxf(largest, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)),
                                   fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
  }
  if (__syncthreads_and(finite) == 0) {  // uniform
    if (t == 0) a.status[head] = kSvdNonFiniteInput;
    return;
  }
  largest = wave_max(largest);
  if ((t & 63) == 0) sh.wave_max[t >> 6] = largest;
  __syncthreads();
  largest = sh.wave_max[0];
#pragma unroll
  for (int w = 1; w < kSvdThreads / 64; ++w) largest = fmaxf(largest, sh.wave_max[w]);
  int exponent = 0;  // largest = f * 2^exponent, f in [1/2, 1)
  frexpf(largest, &exponent);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int f = i * kSvdThreads + t;  // float4 index: row f / 32, column 4 (f % 32)
    double* const to = sh.w + (f >> 5) * kSvdRowStride + 4 * (f & 31);
    *reinterpret_cast<double2*>(to) = make_double2(scaled(v[i].x, exponent),
                                                   scaled(v[i].y, exponent));
    *reinterpret_cast<double2*>(to + 2) = make_double2(scaled(v[i].z, exponent),
                                                       scaled(v[i].w, exponent));
  }
  __syncthreads();

  // ---- Jacobi sweeps ------------------------------------------------------
  const int pair = t / kLanesPerPair;
  const int lane = t % kLanesPerPair;
  bool converged = false;
  for (int sweep = 0; sweep < a.max_sweeps; ++sweep) {
    bool rotated = false;
    for (int round = 0; round < kRounds; ++round) {
      int first = kDim - 1, second = round;
      if (pair != 0) {
        first = round + pair;
        if (first >= kRounds) first -= kRounds;
        second = round - pair;
        if (second < 0) second += kRounds;
      }
      double* const row_a = sh.w + first * kSvdRowStride;
      double* const row_b = sh.w + second * kSvdRowStride;
      double x[kSpan], y[kSpan];
#pragma unroll
      for (int e = 0; e < kSpan / 2; ++e) {  // double2 chunks lane, lane + 8, ...
        const double2 xa = *reinterpret_cast<const double2*>(row_a + 2 * (lane + 8 * e));
        const double2 yb = *reinterpret_cast<const double2*>(row_b + 2 * (lane + 8 * e));
        x[2 * e] = xa.x, x[2 * e + 1] = xa.y;
        y[2 * e] = yb.x, y[2 * e + 1] = yb.y;
      }
      double a2[2] = {0.0, 0.0}, b2[2] = {0.0, 0.0}, g2[2] = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < kSpan; ++i) {
        a2[i & 1] = fma(x[i], x[i], a2[i & 1]);
        b2[i & 1] = fma(y[i], y[i], b2[i & 1]);
        g2[i & 1] = fma(x[i], y[i], g2[i & 1]);
      }
      double alpha = a2[0] + a2[1], beta = b2[0] + b2[1], gamma = g2[0] + g2[1];
      // The pair's eight lanes add their partial sums in the same commuted
      // order, so all eight hold identical totals and take the same branch.
      alpha += dpp_xor<1>(alpha), beta += dpp_xor<1>(beta), gamma += dpp_xor<1>(gamma);
      alpha += dpp_xor<2>(alpha), beta += dpp_xor<2>(beta), gamma += dpp_xor<2>(gamma);
      alpha += dpp_xor<4>(alpha), beta += dpp_xor<4>(beta), gamma += dpp_xor<4>(gamma);
      const bool active = alpha > kNegligibleSquare && beta > kNegligibleSquare &&
                          gamma * gamma > kCosineTolerance * kCosineTolerance * alpha * beta;
      if (active) {
        // Rotate (x, y) -> (c x - s y, s x + c y) by the angle of magnitude
        // at most pi/4 that makes the rows orthogonal: t = s/c solves
        // t^2 + 2 zeta t - 1 = 0 with zeta = (beta - alpha) / (2 gamma), and
        // the smaller root sign(zeta) / (|zeta| + sqrt(1 + zeta^2)), times
        // |2 gamma| above and below, is 2 gamma sign(d) / (|d| + sqrt(d^2 +
        // 4 gamma^2)) with d = beta - alpha: one dependent division fewer.
        // After the head's scaling alpha, beta <= 128 and gamma^2 > 2^-264, so
        // neither square overflows or underflows.
        const double d = beta - alpha;
        const double two_gamma = 2.0 * gamma;
        // sign(zeta) |2 gamma| = 2 gamma sign(d), with sign(+0) = +1 (for
        // d = 0, zeta = +0 / (2 gamma) carries the sign of gamma).
        const double tangent = (d < 0.0 ? -two_gamma : two_gamma) /
                               (fabs(d) + sqrt(fma(d, d, two_gamma * two_gamma)));
        const double c = 1.0 / sqrt(fma(tangent, tangent, 1.0));
        const double s = c * tangent;
#pragma unroll
        for (int i = 0; i < kSpan; ++i) {
          const double xi = x[i], yi = y[i];
          x[i] = fma(c, xi, -(s * yi));
          y[i] = fma(s, xi, c * yi);
        }
#pragma unroll
        for (int e = 0; e < kSpan / 2; ++e) {
          *reinterpret_cast<double2*>(row_a + 2 * (lane + 8 * e)) =
              make_double2(x[2 * e], x[2 * e + 1]);
          *reinterpret_cast<double2*>(row_b + 2 * (lane + 8 * e)) =
              make_double2(y[2 * e], y[2 * e + 1]);
        }
        rotated = true;
      }
      __syncthreads();
    }
    if (__syncthreads_or(rotated) == 0) {  // uniform
      converged = true;
      break;
    }
  }

  // ---- the four rows of largest norm --------------------------------------
  if (t < kDim) {
    const double* const row = sh.w + t * kSvdRowStride;
    double sum = 0.0;
    for (int k = 0; k < kDim; ++k) sum = fma(row[k], row[k], sum);
    sh.norm[t] = sum;
  }
  __syncthreads();
  if (t == 0) {
    // Decreasing norm; equal norms in increasing row order.
    uint64_t taken[2] = {0, 0};
    for (int r = 0; r < kSvdRank; ++r) {
      int best = 0;
      double best_norm = -1.0;
      for (int row = 0; row < kDim; ++row) {
        const bool used = (taken[row >> 6] >> (row & 63)) & 1u;
        if (!used && sh.norm[row] > best_norm) best_norm = sh.norm[row], best = row;
      }
      taken[best >> 6] |= uint64_t{1} << (best & 63);
      sh.top[r] = best;
    }
  }
  __syncthreads();
  int top[kSvdRank];
#pragma unroll
  for (int r = 0; r < kSvdRank; ++r) top[r] = sh.top[r];

  // ---- right vectors: y_r = P w_r (scaled P), four lanes per row ----------
  static_assert(kSvdThreads == 4 * kDim, "four lanes per row");
  {
    const int row = t >> 2;
    const int part = t & 3;  // keys 32 part .. 32 part + 31
    const float4* const source = reinterpret_cast<const float4*>(p + row * kDim + 32 * part);
    double acc[kSvdRank] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int j = 0; j < 8; ++j) {
      const float4 q = source[j];
      const double qs[4] = {scaled(q.x, exponent), scaled(q.y, exponent),
                            scaled(q.z, exponent), scaled(q.w, exponent)};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = 32 * part + 4 * j + c;
#pragma unroll
        for (int r = 0; r < kSvdRank; ++r) {
          acc[r] = fma(qs[c], sh.w[top[r] * kSvdRowStride + k], acc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) {
      acc[r] += dpp_xor<1>(acc[r]);
      acc[r] += dpp_xor<2>(acc[r]);
      if (part == 0) sh.y[r][row] = acc[r];
    }
  }
  __syncthreads();
  if (t < kSvdRank) {
    double sum = 0.0;
    for (int row = 0; row < kDim; ++row) sum = fma(sh.y[t][row], sh.y[t][row], sum);
    sh.y_norm[t] = sqrt(sum);
  }
  __syncthreads();
  if (t < kDim) {
    uint32_t bits[kSvdRank];
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) {
      // A zero product (a head of rank below r + 1 whose row r is zero)
      // leaves a zero vector; its key is zero as well.
      const double n = sh.y_norm[r];
      const float right = n > 0.0 ? static_cast<float>(sh.y[r][t] / n) : 0.0f;
      sh.right[t][r] = right;
      bits[r] = float_to_half_bits(right);
    }
    *reinterpret_cast<uint2*>(a.values + (head * kDim + t) * kSvdRank) =
        make_uint2(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16));
  }

  // ---- keys and residual ----------------------------------------------------
  const int key = t & (kDim - 1);
  float left[kSvdRank];
#pragma unroll
  for (int r = 0; r < kSvdRank; ++r) {
    left[r] = static_cast<float>(ldexp(sh.w[top[r] * kSvdRowStride + key], exponent));
  }
  if (t < kDim) {
    uint32_t bits[kSvdRank];
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) bits[r] = float_to_half_bits(left[r]);
    *reinterpret_cast<uint2*>(a.keys + (head * kDim + key) * kSvdRank) =
        make_uint2(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16));
  }
  __syncthreads();  // sh.right
  float* const out = a.residual + head * kTile;
  for (int row = t >> 7; row < kDim; row += kSvdThreads / kDim) {
    float fit = left[0] * sh.right[row][0];
#pragma unroll
    for (int r = 1; r < kSvdRank; ++r) fit = fmaf(left[r], sh.right[row][r], fit);
    out[row * kDim + key] = p[row * kDim + key] - fit;
  }
  // An unconverged head still gets the fit of its last sweep, flagged.
  if (t == 0) a.status[head] = converged ? kSvdOk : kSvdNotConverged;
}

// The Jacobi form over the batch: every head, or the pending ones, whose marks
// a workgroup reads 512 at a time (one per thread) before it starts on them.
// The heads are dealt out by dealt_item: pending ones often recur at a period.
__global__ __launch_bounds__(kSvdThreads) void exact_svd_jacobi_kernel(SvdArgs a) {
  extern __shared__ __align__(16) unsigned char dynamic[];
  SvdShared& sh = *reinterpret_cast<SvdShared*>(dynamic);
  const int t = threadIdx.x;
  for (uint64_t turn = 0; turn * gridDim.x < a.heads; turn += kSvdThreads) {
    const uint64_t own = dealt_item(blockIdx.x, turn + t, gridDim.x);
    const bool wanted = own < a.heads && (!a.pending_only || a.status[own] == kSvdPending);
    const uint64_t mask = __ballot(wanted);
    if ((t & 63) == 0) sh.pending[t >> 6] = mask;
    __syncthreads();
    for (int w = 0; w < kSvdThreads / 64; ++w) {
      uint64_t left = sh.pending[w];
      while (left != 0) {  // uniform
        const int bit = __builtin_ctzll(left);
        left &= left - 1;
        jacobi_head(sh, a, dealt_item(blockIdx.x, turn + 64 * w + bit, gridDim.x), t);
        __syncthreads();  // the next head reuses the rows
      }
    }
    __syncthreads();  // every thread has read the marks
  }
}

// ---- the direct form: Gram matrix, tridiagonal form, four eigenpairs -------
//
// The batch's kernel.  Only four singular triplets are kept, so instead of
// orthogonalizing all 128 rows (about 11 sweeps x 127 barrier-separated rounds
// that move every row through LDS) it forms G = P P^T, reduces it to
// tridiagonal form by 126 Householder reflections, finds the four largest
// eigenvalues by 64-way multisection on Sturm counts and their eigenvectors by
// twisted factorization, and maps those back: the right vectors (values) are
// the eigenvectors q, the keys P^T q, so that the product of each pair is
// q q^T P whatever the last bits of the eigenvalue are.
//
// What bounds it: the 126 reflections are a serial chain (two barriers, a
// 16-lane norm, an fp64 square root and reciprocal, one matrix-vector product
// each; 0.5 us to 1.3 us, about half of a head's 0.2 ms) that issues up to 500
// vector instructions a step, so the layout keeps it short: G stays in
// registers (256 threads x 64 doubles), block-cyclic over the threads so that
// the shrinking active part stays spread over all of them, in the layout the
// fp64 MFMA leaves it in; a row's sum is finished inside one 16-lane DPP row
// and the only traffic through LDS is the vector u and the product G u.  Two
// heads share a CU (256 VGPRs, under 80 KiB of LDS).  Jacobi -> this form:
// 32 heads 2.35 -> 0.20 ms, 960 heads 9.2 -> 0.52 ms, 8,192 heads 72.7 -> 3.71
// ms; 32 heads of rank three (two passes) 3.09 -> 0.39 ms.
//
// Squaring P costs accuracy only where a singular value is far below the
// first: its vector's error is about 2^-52 (sigma_1 / sigma_r)^2.  A pass
// therefore keeps only the triplets with lambda_r > 2^-20 lambda_1 (sigma_r >
// 2^-10 sigma_1).  A head with fewer than four of them (a state of fewer than
// four tokens has that rank) takes another pass over what is left of P without
// the triplets found, which the Gram matrix forms in double from P itself (2^-53
// of sigma_1 is lost, as in any double form; nothing is kept in fewer bits); it
// costs as much as the first.  Where vectors lean on each other (repeated
// eigenvalues), those up to the first that does are kept and another pass finds
// the rest: at most four passes, 0.2 ms each for 32 heads, where the Jacobi
// kernel takes about 2 ms.  A head whose first vector's residual is not at
// rounding level, or whose rows look orthogonal from the start, is marked
// pending for that kernel.
constexpr int kDirectThreads = 256;
constexpr int kStageStride = kDim + 4;                    // floats
constexpr int kVectorStride = 10;                         // doubles: 16 rows of 8, bank-spread
constexpr int kReflectors = kDim - 2;
constexpr int kReflectorWords = (kDim - 1) * kDim / 2;  // sum of 127 - k, k = 0..125, and one
constexpr int kSections = 9;                              // 65^9 > 2^54
constexpr double kTinyPivot = 1e-30;
constexpr double kTinyCoupling = 1e-40;                   // floor of a squared off-diagonal
constexpr double kZeroColumn = 1e-200;                    // a squared column norm taken as zero
constexpr double kSmallestRatio = 0x1p-20;                // lambda_4 / lambda_1
constexpr double kLargestOverlap = 1e-4;                  // |z_r . z_s| before orthogonalization
constexpr double kSmallestRemainder = 0.5;                // |q|^2 behind the earlier vectors
constexpr double kLargestResidual = 1e-12;                // |T z - lambda z|, |T| <= 1

typedef double Double4 __attribute__((ext_vector_type(4)));

struct DirectShared {
  union {
    float stage[kDim * kStageStride];       // P, while G is formed
    struct {
      double reflector[kReflectorWords];    // u_k, 127 - k doubles each, from reflector_at(k)
      double2 chain[kDim];                  // scaled {d_i, e_(i-1)^2}
    };
    double partial[2][kDim][kSvdRank];      // half sums of P^T q, at the end
  };
  union {
    struct {
      double u[16 * kVectorStride];         // element i at [i % 16][i / 16]
      double product[16 * kVectorStride];   // G u, the same layout
    };
    double pivot[kSvdRank][2][kDim];        // forward and backward pivots, then the vectors
  };
  union {
    struct {
      double inverse_h[kDim];               // 2 / u.u (0: no reflection)
      double d[kDim];                       // diagonal
      double e[kDim];                       // e_i couples i and i + 1; scaled after the reduction
    };
    double fit[kSvdRank - 1][kDim];         // P^T q of the triplets found, between passes
  };
  double lambda[kSvdRank];
  double scaled_minor[kSvdRank][2][kDim / 8];
  float wave_max[kDirectThreads / 64];
};
static_assert(workgroups_by_lds(sizeof(DirectShared)) >= 2, "two heads per CU");

// (One place is left free in front, which the masked read of u_0 touches.)
constexpr int reflector_at(int k) { return 1 + k * (kDim - 1) - k * (k - 1) / 2; }

// 1 / x and sqrt(x) for normal x: the hardware estimate (relative error at most
// 2^-24, measured) and one step of the third order, r (1 + e + e^2) and
// y (1 + e / 2 + 3 e^2 / 8), which leaves only the rounding of the steps.
__device__ __forceinline__ double fast_reciprocal(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
__device__ __forceinline__ double fast_sqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double root = x * y;
  const double e = fma(-root, y, 1.0);
  return fma(root * e, fma(e, 0.375, 0.5), root);
}

// x of the lane a DPP control names, every lane of the wavefront having one
// (so no old value need be kept); kRowBroadcast + n names lane n of the row,
// and moves both dwords in one instruction.
constexpr int kRowBroadcast = 0x150;
template <int kCtrl>
__device__ __forceinline__ double dpp_move(double x) {
  return __builtin_amdgcn_mov_dpp(x, kCtrl, 0xF, 0xF, true);
}

// Sum over the 16 lanes of a DPP row, the same in every lane: once the lanes of
// a quad agree, mirroring a half row names the other quad's sum, and rotating
// by 8 the other half's.
__device__ __forceinline__ double row_sum(double x) {
  x += dpp_move<kDppQuadSwap1>(x);
  x += dpp_move<kDppQuadSwap2>(x);
  x += dpp_move<kDppHalfMirror>(x);
  return x + dpp_move<kDppRowRotate8>(x);
}
__device__ __forceinline__ double wave_sum_f64(double x) {
  const auto add = [](double p, double q) { return p + q; };
  x = row_sum(x);
  x = combine_with_partner<16>(x, add);
  return combine_with_partner<32>(x, add);
}

// A lane with `up` clear ends with lo + partner's lo, one with it set with
// hi + partner's hi.
template <int kCtrl>
__device__ __forceinline__ double fold_row(double lo, double hi, bool up) {
  const double send = up ? lo : hi;
  const double keep = up ? hi : lo;
  return keep + dpp_move<kCtrl>(send);
}

// Sums v[kFirst .. 7] over the 16 lanes of a DPP row; lane c gets the sum of
// slot slot_of<kFirst>(c).  (Mirroring a half row pairs c with 7 - c, which
// the two quad exchanges behind it complete to all eight lanes.)
template <int kFirst>
__device__ __forceinline__ int slot_of(int c) {
  constexpr int count = kFirst < 4 ? 8 : kFirst < 6 ? 4 : kFirst < 7 ? 2 : 1;
  return 8 - count + ((c >> 1) & (count - 1));
}
template <int kFirst>
__device__ __forceinline__ double row_scatter_sum(const double (&v)[8], int c) {
  double four[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    four[i] = kFirst < 4 ? fold_row<kDppRowRotate8>(v[i], v[i + 4], (c & 8) != 0) : v[i + 4];
  }
  double two[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    two[i] = kFirst < 6 ? fold_row<kDppHalfMirror>(four[i], four[i + 2], (c & 4) != 0)
                        : four[i + 2];
  }
  double one;
  if constexpr (kFirst < 7) {
    one = fold_row<kDppQuadSwap2>(two[0], two[1], (c & 2) != 0);
  } else {
    one = two[1] + dpp_move<kDppQuadSwap2>(two[1]);
  }
  one += dpp_move<kDppQuadSwap1>(one);
  if constexpr (kFirst >= 6) {  // lane ^ 4: the mirror alone would change the slot
    one += dpp_move<kDppHalfMirror>(dpp_move<kDppQuadReverse>(one));
  }
  if constexpr (kFirst >= 4) one += dpp_move<kDppRowRotate8>(one);
  return one;
}

// values[a] = slot a's value, for a >= kFirst, of a row whose lane c holds slot
// slot_of(c).
template <int kFirst, int kSlot = kFirst, typename Lane>
__device__ __forceinline__ void spread_slots(double own, double (&values)[8], Lane) {
  if constexpr (kSlot < 8) {
    values[kSlot] = dpp_move<kRowBroadcast + Lane::of(kSlot)>(own);
    spread_slots<kFirst, kSlot + 1>(own, values, Lane{});
  }
}
struct DirectLane {  // lane c holds slot c % 8
  static constexpr int of(int slot) { return slot; }
};
template <int kFirst>
struct ScatterLane {  // lane c holds slot_of<kFirst>(c)
  static constexpr int of(int slot) {
    return kFirst < 4 ? 2 * slot : kFirst < 6 ? 2 * (slot - 4) : kFirst < 7 ? 2 * (slot - 6) : 0;
  }
};

// Reflections 16 kFirst .. 16 kFirst + 15: rows and columns below 16 kFirst
// are finished, so slots 0 .. kFirst - 1 of both are skipped.  Thread (wave w,
// lane group g, lane c) holds G[16 a + 4 w + g][16 b + c] in m[a][b].  A step
// reads u and G u from LDS once per column (four 16-byte reads each); the row
// entries come out of one 8-byte read, or of the row's own sums, by DPP
// broadcasts (as LDS reads they doubled the LDS time, which bound the first
// blocks).  The product is taken with the column itself, so that it overlaps
// the norm's chain, and corrected for the one element that u changes.
template <int kFirst>
__device__ __forceinline__ void reflect_block(DirectShared& sh, double (&m)[8][8], int row,
                                              int c) {
  constexpr int kLast = kFirst == 7 ? kReflectors : 16 * kFirst + 16;
  constexpr int kNext = kFirst < 7 ? kFirst + 1 : 7;
#pragma unroll 1
  for (int k = 16 * kFirst; k < kLast; ++k) {
    const int at = k & 15;
    if (c == at) {  // column k, below the diagonal
      double* const to = sh.u + row * kVectorStride;
      to[kFirst] = row > at ? m[kFirst][kFirst] : 0.0;
#pragma unroll
      for (int a = kFirst + 1; a < 8; ++a) to[a] = m[a][kFirst];
      if (row == at) sh.d[k] = m[kFirst][kFirst];
    }
    __syncthreads();
    double ur[8], uc[8];
#pragma unroll
    for (int a = kFirst & ~1; a < 8; a += 2) {
      const double2 q = *reinterpret_cast<const double2*>(sh.u + c * kVectorStride + a);
      uc[a] = q.x, uc[a + 1] = q.y;
    }
    const double row_part = sh.u[row * kVectorStride + (c & 7)];
    const int next = (k + 1) & 15;  // element k + 1 lives in row / lane `next`,
    const bool carry = next == 0;   // in slot kFirst + 1 instead of kFirst
    const double x0 = sh.u[next * kVectorStride + kFirst + (carry ? 1 : 0)];
    double square = 0.0;
#pragma unroll
    for (int b = kFirst; b < 8; ++b) square = fma(uc[b], uc[b], square);
    square = row_sum(square);
    double sums[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int b = kFirst; b < 8; ++b) {
#pragma unroll
      for (int a = kFirst; a < 8; ++a) sums[a] = fma(m[a][b], uc[b], sums[a]);
    }
    // u = x - alpha e_1 with alpha = -sign(x0) |x|, 2 / u.u = 1 / (|x|^2 + |x0| |x|).
    const bool reflects = square > kZeroColumn;
    const double norm = fast_sqrt(square);
    const double alpha = reflects ? -copysign(norm, x0) : 0.0;
    const double inverse_h = reflects ? fast_reciprocal(fma(fabs(x0), norm, square)) : 0.0;
    const double change = c == next ? -alpha : 0.0;
    if (carry) {  // uniform
#pragma unroll
      for (int a = kFirst; a < 8; ++a) sums[a] = fma(m[a][kNext], change, sums[a]);
    } else {
#pragma unroll
      for (int a = kFirst; a < 8; ++a) sums[a] = fma(m[a][kFirst], change, sums[a]);
    }
    const double sum = row_scatter_sum<kFirst>(sums, c);
    if ((c & 1) == 0) sh.product[row * kVectorStride + slot_of<kFirst>(c)] = sum;
    spread_slots<kFirst>(row_part, ur, DirectLane{});
    const double head = reflects ? x0 - alpha : 0.0;
    if (row == next) {
      if (carry) ur[kNext] = head; else ur[kFirst] = head;
    }
    if (c == next) {
      if (carry) uc[kNext] = head; else uc[kFirst] = head;
    }
    if (row == 0) {  // the reflector, for the way back
      double* const to = sh.reflector + reflector_at(k) - (k + 1) + c;
      if (c > at) to[16 * kFirst] = uc[kFirst];
#pragma unroll
      for (int b = kFirst + 1; b < 8; ++b) to[16 * b] = uc[b];
      if (c == 0) {
        sh.e[k] = alpha;
        sh.inverse_h[k] = inverse_h;
      }
    }
    __syncthreads();
    double pr[8], pc[8];
#pragma unroll
    for (int a = kFirst & ~1; a < 8; a += 2) {
      const double2 q = *reinterpret_cast<const double2*>(sh.product + c * kVectorStride + a);
      pc[a] = q.x, pc[a + 1] = q.y;
    }
    spread_slots<kFirst>(sum, pr, ScatterLane<kFirst>{});
    double along = 0.0;
#pragma unroll
    for (int b = kFirst; b < 8; ++b) along = fma(uc[b], pc[b], along);
    along = row_sum(along);
    const double shift = -0.5 * along * inverse_h * inverse_h;
#pragma unroll
    for (int a = kFirst; a < 8; ++a) {
      pr[a] = fma(shift, ur[a], pr[a] * inverse_h);
      pc[a] = fma(shift, uc[a], pc[a] * inverse_h);
    }
#pragma unroll
    for (int b = kFirst; b < 8; ++b) {
#pragma unroll
      for (int a = kFirst; a < 8; ++a) {
        m[a][b] = fma(-ur[a], pc[b], fma(-pr[a], uc[b], m[a][b]));
      }
    }
  }
}

// The number of eigenvalues below x of the scaled tridiagonal matrix: sign
// changes of the leading principal minors, by their three-term recurrence
// (rescaled every 8 rows; a squared coupling is at least kTinyCoupling, so two
// neighbouring minors never both vanish).
__device__ __forceinline__ int count_below(const DirectShared& sh, double x) {
  double before = 1.0, minor = sh.chain[0].x - x;
  uint32_t signs = static_cast<uint32_t>(__double2hiint(minor)) >> 31;
  int count = __popc(signs);
  constexpr int kRows = 8;
  double2 links[kRows], ahead[kRows];
#pragma unroll
  for (int j = 0; j < kRows; ++j) links[j] = sh.chain[j];
#pragma unroll 2
  for (int i0 = 0; i0 < kDim; i0 += kRows) {
    // The next rows' links are read while these rows' chain runs.
    const double2* const from = sh.chain + ((i0 + kRows) & (kDim - 1));
#pragma unroll
    for (int j = 0; j < kRows; ++j) ahead[j] = from[j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      double following = fma(links[j].x - x, minor, -(links[j].y * before));
      double kept = minor;
      if (j == 0) {  // row 0 is the start of the recurrence
        following = i0 == 0 ? minor : following;
        kept = i0 == 0 ? before : kept;
      }
      before = kept;
      minor = following;
      signs = (signs << 1) | (static_cast<uint32_t>(__double2hiint(minor)) >> 31);
    }
    // Sign changes between the nine latest minors (row 0 repeats its own).
    count += __popc((signs ^ (signs >> 1)) & 0xFFu);
    const int exponent = max(__builtin_amdgcn_frexp_exp(minor), __builtin_amdgcn_frexp_exp(before));
    minor = __builtin_amdgcn_ldexp(minor, -exponent);
    before = __builtin_amdgcn_ldexp(before, -exponent);
#pragma unroll
    for (int j = 0; j < kRows; ++j) links[j] = ahead[j];
  }
  return count;
}

// G = P P^T on the fp64 MFMA (16x16x4), times 2^(-2 exponent).
// Operand lane (k group l / 16, index l % 16); result register v of lane l is
// row 4 v + l / 16, column l % 16 of its block.  The row operand takes the
// rows 16 (4 half + i / 4) + 4 wave + i % 4, so that register v of half h is
// slot 4 h + v of reflect_block's layout.  fp32 products are exact in double
// and neither overflow nor vanish, so P is used unscaled and G scaled: its
// entries are then at most 128.  With kDeflated the operands are what is left
// of P without the triplets found, formed in double where they are read
// (q [row][4] and fit [triplet][key], zero for those not found).
template <bool kDeflated>
__device__ __forceinline__ void gram_matrix(const DirectShared& sh, const double* q,
                                            double (&m)[8][8], int wave, int lane, int exponent) {
  const int c = lane & 15;
  Double4 block[2][8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int b = 0; b < 8; ++b) block[h][b] = Double4{0.0, 0.0, 0.0, 0.0};
  }
  const int left = 16 * (c >> 2) + 4 * wave + (c & 3);
  const int keys = 4 * (lane >> 4);
#pragma unroll 1
  for (int k = 0; k < kDim; k += 16) {
    using Operand = std::conditional_t<kDeflated, double, float>;
    Operand l[2][4], r[4][4];
    double fit[kSvdRank - 1][4];
    if constexpr (kDeflated) {
#pragma unroll
      for (int i = 0; i < kSvdRank - 1; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fit[i][j] = sh.fit[i][k + keys + j];
      }
    }
    const auto load = [&](Operand(&to)[4], int row) {
      float cells[4];
      *reinterpret_cast<float4*>(cells) =
          *reinterpret_cast<const float4*>(sh.stage + row * kStageStride + k + keys);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        to[j] = cells[j];
        if constexpr (kDeflated) {
#pragma unroll
          for (int i = 0; i < kSvdRank - 1; ++i) {
            to[j] = fma(-q[row * kSvdRank + i], fit[i][j], to[j]);
          }
        }
      }
    };
#pragma unroll
    for (int h = 0; h < 2; ++h) load(l[h], left + 64 * h);
    // Four blocks of columns, one key of every lane group at a time:
    // successive products go to different accumulators.
#pragma unroll
    for (int b0 = 0; b0 < 8; b0 += 4) {
#pragma unroll
      for (int b = 0; b < 4; ++b) load(r[b], 16 * (b0 + b) + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            block[h][b0 + b] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(l[h][j], r[b][j], block[h][b0 + b], 0, 0, 0);
          }
        }
      }
    }
  }
  const double scale = ldexp(1.0, -2 * exponent);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      for (int b = 0; b < 8; ++b) m[4 * h + v][b] = block[h][b][v] * scale;
    }
  }
}

// The tridiagonal matrix scaled by a power of two to |T| <= 1 (chain, e);
// returns the Gershgorin bound of its eigenvalues.
__device__ __forceinline__ double scale_chain(DirectShared& sh, int wave, int lane) {
  const double e0 = sh.e[lane], e1 = lane < 63 ? sh.e[64 + lane] : 0.0;
  const double b0 = lane > 0 ? sh.e[lane - 1] : 0.0, b1 = sh.e[63 + lane];
  const double d0 = sh.d[lane], d1 = sh.d[64 + lane];
  double reach = fmax(fabs(d0) + fabs(e0) + fabs(b0), fabs(d1) + fabs(e1) + fabs(b1));
  const auto maximum = [](double x, double y) { return fmax(x, y); };
  reach = combine_with_partner<1>(reach, maximum);
  reach = combine_with_partner<2>(reach, maximum);
  reach = combine_with_partner<4>(reach, maximum);
  reach = combine_with_partner<8>(reach, maximum);
  reach = combine_with_partner<16>(reach, maximum);
  reach = combine_with_partner<32>(reach, maximum);
  const int power = reach > 0.0 ? -__builtin_amdgcn_frexp_exp(reach) : 0;
  const double top = ldexp(reach, power) * (1.0 + 0x1p-40);
  __syncthreads();  // every wave has read d and e
  if (wave == 0) {
    const double s0 = ldexp(b0, power), s1 = ldexp(b1, power);
    sh.chain[lane] = make_double2(ldexp(d0, power), fmax(s0 * s0, kTinyCoupling));
    sh.chain[64 + lane] = make_double2(ldexp(d1, power), fmax(s1 * s1, kTinyCoupling));
    sh.e[lane] = ldexp(e0, power);
    sh.e[64 + lane] = ldexp(e1, power);
  }
  __syncthreads();
  return top;
}

// Eigenvalue `index` (0 the largest) by 64-way multisection of one wavefront.
__device__ __forceinline__ double section(DirectShared& sh, double top, int index, int lane) {
  double low = -0x1p-20, high = top;
#pragma unroll 1
  for (int section = 0; section < kSections; ++section) {
    const double step = (high - low) * (1.0 / 65.0);
    const double x = fma(step, static_cast<double>(lane + 1), low);
    // x is at or below eigenvalue `index` while at least index + 1 lie above it.
    const uint64_t below = __ballot(count_below(sh, x) <= kDim - 1 - index);
    const int inside = ~below == 0 ? 64 : __builtin_ctzll(~below);  // leading lanes
    const double from = low;
    low = inside > 0 ? fma(step, static_cast<double>(inside), from) : from;
    high = inside < 64 ? fma(step, static_cast<double>(inside + 1), from) : high;
  }
  const double lambda = 0.5 * (low + high);
  if (lane == 0) sh.lambda[index] = lambda;
  return lambda;
}

// The unit eigenvector of eigenvalue `lambda` of one wavefront, by twisted
// factorization, to pivot[index][0]; its residual to pivot[index][1][0].
// Lane 0 forms the leading principal minors of T - lambda from the top, lane 1
// the trailing ones from the bottom, by count_below's recurrence; neighbours'
// quotients are the pivots of the two triangular factorizations (dividing
// afterwards, all lanes at once, keeps the division out of the chain: 128
// dependent reciprocals took 62,000 cycles).  The twist is where the two meet
// with the smallest remainder, and the vector follows from it outwards (every
// row but the twist's holds to rounding).
__device__ __forceinline__ void twisted_vector(DirectShared& sh, double lambda, int index,
                                               int lane) {
  double* const forward = sh.pivot[index][0];
  double* const backward = sh.pivot[index][1];
  if (lane < 2) {
    double* const minors = lane == 0 ? forward : backward;
    double before = 0.0, minor = 1.0, coupling = 0.0;
#pragma unroll 1
    for (int s0 = 0; s0 < kDim; s0 += 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int i = lane == 0 ? s0 + j : kDim - 1 - s0 - j;
        const double2 link = sh.chain[i];
        const double into = lane == 0 ? link.y : coupling;  // couples row i and the one before
        const double following = fma(link.x - lambda, minor, -(into * before));
        before = minor;
        minor = following;
        coupling = link.y;
        minors[i] = minor;
      }
      const int exponent =
          max(__builtin_amdgcn_frexp_exp(minor), __builtin_amdgcn_frexp_exp(before));
      minor = __builtin_amdgcn_ldexp(minor, -exponent);
      before = __builtin_amdgcn_ldexp(before, -exponent);
      // The scale of the next eight rows: a minor at a multiple of eight is
      // divided by its neighbour at this scale.
      if (s0 + 8 < kDim) sh.scaled_minor[index][lane][s0 / 8] = minor;
    }
  }
  wave_lds_sync();
  // The pivots of rows lane and 64 + lane; a vanishing one counts as
  // kTinyPivot, and the row behind it follows from that.
  const auto pivot = [&](int side, int i) {
    const double* const minors = side == 0 ? forward : backward;
    const int s = side == 0 ? i : kDim - 1 - i;       // rows from this side's start
    const int prior = side == 0 ? i - 1 : i + 1;
    const double diagonal = sh.chain[i].x - lambda;
    if (s == 0) return diagonal == 0.0 ? kTinyPivot : diagonal;
    const double below = s % 8 == 0 ? sh.scaled_minor[index][side][s / 8 - 1] : minors[prior];
    const double coupling = sh.chain[side == 0 ? i : i + 1].y;
    const double quotient = below == 0.0 ? diagonal - coupling / kTinyPivot
                                         : minors[i] * fast_reciprocal(below);
    return quotient == 0.0 ? kTinyPivot : quotient;
  };
  const double f0 = pivot(0, lane), f1 = pivot(0, 64 + lane);
  const double r0 = pivot(1, lane), r1 = pivot(1, 64 + lane);
  const double g0 = fabs((f0 + r0) - (sh.chain[lane].x - lambda));
  const double g1 = fabs((f1 + r1) - (sh.chain[64 + lane].x - lambda));
  double best = fmin(g0, g1);
  const auto minimum = [](double x, double y) { return fmin(x, y); };
  best = combine_with_partner<1>(best, minimum);
  best = combine_with_partner<2>(best, minimum);
  best = combine_with_partner<4>(best, minimum);
  best = combine_with_partner<8>(best, minimum);
  best = combine_with_partner<16>(best, minimum);
  best = combine_with_partner<32>(best, minimum);
  const uint64_t first = __ballot(g0 == best), second = __ballot(g1 == best);
  const int twist = first != 0 ? __builtin_ctzll(first)
                               : second != 0 ? 64 + __builtin_ctzll(second) : 0;
  // z_i = -(e_i / forward_i) z_(i+1) above the twist, -(e_(i-1) / backward_i)
  // z_(i-1) below it: the factors in place of the minors.
  wave_lds_sync();
  forward[lane] = -sh.e[lane] * fast_reciprocal(f0);
  forward[64 + lane] = -sh.e[64 + lane] * fast_reciprocal(f1);
  backward[lane] = lane > 0 ? -sh.e[lane - 1] * fast_reciprocal(r0) : 0.0;
  backward[64 + lane] = -sh.e[63 + lane] * fast_reciprocal(r1);
  wave_lds_sync();
  if (lane < 2) {
    double* const factors = lane == 0 ? forward : backward;
    const int steps = lane == 0 ? twist : kDim - 1 - twist;
    const int direction = lane == 0 ? -1 : 1;
    double z = 1.0;
    for (int s = 1; s <= steps; s += 8) {
      // Past the end the twist's own place, which nothing reads, takes part.
      double factor[8];
      double* at[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        at[j] = factors + twist + (s + j <= steps ? direction * (s + j) : 0);
        factor[j] = *at[j];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        z *= factor[j];
        *at[j] = z;
      }
    }
  }
  wave_lds_sync();
  const auto element = [&](int i) {
    return i == twist ? 1.0 : i < twist ? forward[i] : backward[i];
  };
  double z0 = element(lane), z1 = element(64 + lane);
  const double length = sqrt(wave_sum_f64(fma(z0, z0, z1 * z1)));
  z0 /= length;
  z1 /= length;
  wave_lds_sync();
  forward[lane] = z0;
  forward[64 + lane] = z1;
  if (lane == 0) backward[0] = best / length;
}

// The first `fresh` vectors made orthogonal, the same in every wavefront, and
// vector `wave` left in z0 (element lane) and z1 (64 + lane).  Returns how many
// of them are sound: residuals at rounding level, vectors near orthogonal to
// begin with.  (The vectors of equal eigenvalues come out as the same vector,
// or leaning on each other.)
__device__ __forceinline__ int orthogonal_vectors(const DirectShared& sh, int fresh, int wave,
                                                  int lane, double& z0, double& z1) {
  double q0[kSvdRank], q1[kSvdRank];
#pragma unroll
  for (int r = 0; r < kSvdRank; ++r) {
    q0[r] = sh.pivot[r][0][lane];
    q1[r] = sh.pivot[r][0][64 + lane];
  }
  bool sound = sh.lambda[0] > 0.0 && sh.pivot[0][1][0] < kLargestResidual;  // false for NaN
  int count = sound ? 1 : 0;
#pragma unroll
  for (int r = 1; r < kSvdRank; ++r) {
    if (r >= fresh) break;
    sound = sound && sh.pivot[r][1][0] < kLargestResidual;
#pragma unroll
    for (int s = 0; s < r; ++s) {
      const double overlap = wave_sum_f64(fma(q0[r], q0[s], q1[r] * q1[s]));
      sound = sound && fabs(overlap) < kLargestOverlap;
      q0[r] = fma(-overlap, q0[s], q0[r]);
      q1[r] = fma(-overlap, q1[s], q1[r]);
    }
    const double inverse = 1.0 / sqrt(wave_sum_f64(fma(q0[r], q0[r], q1[r] * q1[r])));
    q0[r] *= inverse;
    q1[r] *= inverse;
    count += sound ? 1 : 0;
  }
  z0 = wave == 0 ? q0[0] : wave == 1 ? q0[1] : wave == 2 ? q0[2] : q0[3];
  z1 = wave == 0 ? q1[0] : wave == 1 ? q1[1] : wave == 2 ? q1[2] : q1[3];
  return count;
}

// Reflections 16 kFirst .. 16 kFirst + 15 undone, in one wavefront for all four
// vectors: lane (g, c) holds elements 16 b + c of vector g in z[b].  Two at a
// time: the three sums of a pair are independent, so their latencies overlap.
template <int kFirst>
__device__ __forceinline__ void unreflect_block(const DirectShared& sh, double (&z)[8], int c) {
  constexpr int kLast = kFirst == 7 ? kReflectors - 1 : 16 * kFirst + 15;
  struct Pair {
    double u[8], v[8];
  };
  const auto load = [&](int k, Pair& p) {
    const double* const u = sh.reflector + reflector_at(k) - (k + 1) + c;
    const double* const v = sh.reflector + reflector_at(k - 1) - k + c;
#pragma unroll
    for (int b = kFirst; b < 8; ++b) p.u[b] = u[16 * b], p.v[b] = v[16 * b];
  };
  Pair now;
  load(kLast, now);
#pragma unroll 2
  for (int k = kLast; k > 16 * kFirst; k -= 2) {
    Pair ahead;
    load(max(k - 2, 16 * kFirst + 1), ahead);
    __builtin_amdgcn_sched_barrier(0);
    now.u[kFirst] = 16 * kFirst + c > k ? now.u[kFirst] : 0.0;
    now.v[kFirst] = 16 * kFirst + c > k - 1 ? now.v[kFirst] : 0.0;
    double uz = 0.0, vz = 0.0, uv = 0.0;
#pragma unroll
    for (int b = kFirst; b < 8; ++b) {
      uz = fma(now.u[b], z[b], uz);
      vz = fma(now.v[b], z[b], vz);
      uv = fma(now.u[b], now.v[b], uv);
    }
    const double first = row_sum(uz) * sh.inverse_h[k];
    const double second = fma(-first, row_sum(uv), row_sum(vz)) * sh.inverse_h[k - 1];
#pragma unroll
    for (int b = kFirst; b < 8; ++b) {
      z[b] = fma(-second, now.v[b], fma(-first, now.u[b], z[b]));
    }
    now = ahead;
  }
}

// The vectors q_found .. q_(found + fresh - 1) made orthogonal to the earlier
// ones (twice, so that the result is at rounding level): the rounding of what
// an earlier pass left lets them lean on those, and P^T q would hold that part
// of the larger triplets.  A vector most of which lies in the
// earlier ones' span belongs to rounding noise: what is left of P has no part
// along that span but noise, so its singular value (and every later one) is at
// the noise's level, and it and all later vectors become zero.  (Left as it
// is, normalized back to length one, it would add a triplet of P a second
// time.)  Returns whether every vector stands; the same in every thread.
__device__ __forceinline__ bool clear_earlier(double* q, int found, int fresh, int wave,
                                              int lane) {
  double q0[kSvdRank], q1[kSvdRank];
#pragma unroll
  for (int r = 0; r < kSvdRank; ++r) {
    q0[r] = q[lane * kSvdRank + r];
    q1[r] = q[(64 + lane) * kSvdRank + r];
  }
  bool stands = true;
#pragma unroll
  for (int r = 1; r < kSvdRank; ++r) {
    if (r >= found && r < found + fresh) {  // uniform
      for (int twice = 0; twice < 2; ++twice) {
#pragma unroll
        for (int s = 0; s < r; ++s) {
          const double overlap = wave_sum_f64(fma(q0[r], q0[s], q1[r] * q1[s]));
          q0[r] = fma(-overlap, q0[s], q0[r]);
          q1[r] = fma(-overlap, q1[s], q1[r]);
        }
      }
      const double square = wave_sum_f64(fma(q0[r], q0[r], q1[r] * q1[r]));
      stands = stands && square > kSmallestRemainder;  // false for NaN
      const double inverse = 1.0 / sqrt(square);
      q0[r] = stands ? q0[r] * inverse : 0.0;
      q1[r] = stands ? q1[r] * inverse : 0.0;
    }
  }
  __syncthreads();  // every wave has read q
  if (wave >= found && wave < found + fresh) {
    q[lane * kSvdRank + wave] = wave == 1 ? q0[1] : wave == 2 ? q0[2] : q0[3];
    q[(64 + lane) * kSvdRank + wave] = wave == 1 ? q1[1] : wave == 2 ? q1[2] : q1[3];
  }
  __syncthreads();
  return stands;
}

__global__ __launch_bounds__(kDirectThreads, 2) void exact_svd_direct_kernel(SvdArgs a) {
  extern __shared__ __align__(16) unsigned char dynamic[];
  DirectShared& sh = *reinterpret_cast<DirectShared*>(dynamic);
  int t = threadIdx.x;
  const uint64_t head = blockIdx.x;
  double* const q = &sh.pivot[0][0][0];  // the right vectors, [row][4]

  // ---- P to LDS, finiteness, largest magnitude ----------------------------
  float largest = 0.0f;
  {
    constexpr int kLoads = kTile / 4 / kDirectThreads;  // 16 float4 per thread
    float4 v[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      v[i] = reinterpret_cast<const float4*>(a.provider + head * kTile)[i * kDirectThreads + t];
    }
    bool finite = true;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      finite = finite && isfinite(v[i].x) && isfinite(v[i].y) && isfinite(v[i].z) &&
               isfinite(v[i].w);
      largest = fmaxf(largest, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)),
                                     fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
      const int f = i * kDirectThreads + t;  // float4 index: row f / 32, column 4 (f % 32)
      *reinterpret_cast<float4*>(sh.stage + (f >> 5) * kStageStride + 4 * (f & 31)) = v[i];
    }
    if (__syncthreads_and(finite) == 0) {  // uniform
      if (t == 0) a.status[head] = kSvdNonFiniteInput;
      return;
    }
  }

  // Each pass finds `fresh` triplets behind the `found` ones; wave r keeps q_r
  // from pass to pass.
  double own0 = 0.0, own1 = 0.0;
  int found = 0;
  while (true) {
    // Opaque, so that what is formed from it (addresses, the cells' loads) is
    // not taken out of the loop and held through it.
    asm volatile("" : "+v"(t));
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lane = t & 63;
    largest = wave_max(largest);
    if (lane == 0) sh.wave_max[wave] = largest;
    __syncthreads();
    largest = fmaxf(fmaxf(sh.wave_max[0], sh.wave_max[1]), fmaxf(sh.wave_max[2], sh.wave_max[3]));
    int exponent = 0;  // the largest magnitude is f * 2^exponent, f in [1/2, 1)
    frexpf(largest, &exponent);
    int fresh = kSvdRank - found;
    // The cells of P this thread takes into P^T q and the residual: key t % 128
    // of rows 64 (t / 128) .. + 63, read once G's registers are free.
    const int key = t & (kDim - 1);
    const int half = t >> 7;
    const uint32_t offset = 64 * half * kDim + key;
    const float* const source = a.provider + head * kTile + offset;
    float cell[kDim / 2];
    double z0 = 0.0, z1 = 0.0;  // nothing left: the other triplets are zero
    if (largest > 0.0f) {       // uniform
      const int c = lane & 15;
      const int row = 4 * wave + (lane >> 4);
      double m[8][8];
      if (found == 0) {
        gram_matrix<false>(sh, q, m, wave, lane, exponent);
      } else {
        gram_matrix<true>(sh, q, m, wave, lane, exponent);
        __syncthreads();  // every wave has read q and fit
      }
      reflect_block<0>(sh, m, row, c);
      // The first 16 rows of P, none zero, orthogonal to all others to begin with:
      // such heads are rarely more than one Jacobi sweep.  32 unit matrices 210
      // us, 341 with the direct form in full before it, 171 by Jacobi alone; the
      // test costs other heads at most 0.4%.
      if (found == 0 && __ballot(sh.e[c] != 0.0 || sh.d[c] == 0.0) == 0) {  // uniform
        if (t == 0) a.status[head] = kSvdPending;
        return;
      }
      reflect_block<1>(sh, m, row, c);
      reflect_block<2>(sh, m, row, c);
      reflect_block<3>(sh, m, row, c);
      reflect_block<4>(sh, m, row, c);
      reflect_block<5>(sh, m, row, c);
      reflect_block<6>(sh, m, row, c);
      reflect_block<7>(sh, m, row, c);
      if (c == 14 && row == 14) sh.d[126] = m[7][7];
      if (c == 15 && row == 15) sh.d[127] = m[7][7];
      if (c == 14 && row == 15) sh.e[126] = m[7][7];
      __syncthreads();
      const double top = scale_chain(sh, wave, lane);
      const double lambda = section(sh, top, wave, lane);
      twisted_vector(sh, lambda, wave, lane);
      __syncthreads();
      while (fresh > 1 && !(sh.lambda[fresh - 1] > kSmallestRatio * sh.lambda[0])) --fresh;
      // The same in every wave: formed from the same values by the same steps.
      fresh = __builtin_amdgcn_readfirstlane(
          orthogonal_vectors(sh, fresh, wave, lane, z0, z1));
      if (fresh == 0) {  // uniform
        if (t == 0) a.status[head] = kSvdPending;
        return;
      }
#pragma unroll
      for (int i = 0; i < kDim / 2; ++i) cell[i] = source[i * kDim];
      __syncthreads();  // every wave has read all four vectors
      sh.pivot[wave][0][lane] = z0;
      sh.pivot[wave][0][64 + lane] = z1;
      __syncthreads();
      if (wave == 0) {
        double z[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) z[b] = sh.pivot[lane >> 4][0][16 * b + c];
        unreflect_block<7>(sh, z, c);
        unreflect_block<6>(sh, z, c);
        unreflect_block<5>(sh, z, c);
        unreflect_block<4>(sh, z, c);
        unreflect_block<3>(sh, z, c);
        unreflect_block<2>(sh, z, c);
        unreflect_block<1>(sh, z, c);
        unreflect_block<0>(sh, z, c);
        wave_lds_sync();
        const int slot = found + (lane >> 4);
        if (slot < kSvdRank) {
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            q[(16 * b + c) * kSvdRank + slot] = (lane >> 4) < fresh ? z[b] : 0.0;
          }
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < kDim / 2; ++i) cell[i] = source[i * kDim];
      __syncthreads();  // every wave is done with the pivot area
      if (wave >= found) q[lane * kSvdRank + wave] = q[(64 + lane) * kSvdRank + wave] = 0.0;
    }
    __syncthreads();
    if (wave < found) {
      q[lane * kSvdRank + wave] = own0;
      q[(64 + lane) * kSvdRank + wave] = own1;
    }
    __syncthreads();
    if (found > 0 && largest > 0.0f && !clear_earlier(q, found, fresh, wave, lane)) {
      fresh = kSvdRank - found;  // the rest stays zero
    }
    found += fresh;

    // ---- keys P^T q (vectors not found yet are zero) ------------------------
    const double* const vectors = q + 64 * half * kSvdRank;
    double y[kSvdRank] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < kDim / 2; ++i) {
#pragma unroll
      for (int r = 0; r < kSvdRank; ++r) {
        y[r] = fma(static_cast<double>(cell[i]), vectors[i * kSvdRank + r], y[r]);
      }
      if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) sh.partial[half][key][r] = y[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) y[r] = sh.partial[0][key][r] + sh.partial[1][key][r];

    if (found < kSvdRank) {  // uniform: stage P again and go round
      if (wave < found) {
        own0 = q[lane * kSvdRank + wave];
        own1 = q[(64 + lane) * kSvdRank + wave];
      }
      if (half == 0) {
#pragma unroll
        for (int r = 0; r < kSvdRank - 1; ++r) sh.fit[r][key] = y[r];
      }
      __syncthreads();  // the half sums are read
      largest = 0.0f;
#pragma unroll
      for (int i = 0; i < kDim / 2; ++i) {
        double rest = cell[i];
#pragma unroll
        for (int r = 0; r < kSvdRank - 1; ++r) {
          rest = fma(-vectors[i * kSvdRank + r], y[r], rest);
        }
        sh.stage[(64 * half + i) * kStageStride + key] = cell[i];
        largest = fmaxf(largest, fabsf(static_cast<float>(rest)));
        if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
      }
      continue;  // the staged cells and fits are published by the next pass's barrier
    }

    // ---- fp16 compensators, residual --------------------------------------
    float left[kSvdRank];
    uint32_t bits[kSvdRank];
#pragma unroll
    for (int r = 0; r < kSvdRank; ++r) {
      left[r] = static_cast<float>(y[r]);
      bits[r] = float_to_half_bits(half == 0 ? left[r]
                                             : static_cast<float>(q[key * kSvdRank + r]));
    }
    // The first half of the threads writes the keys, the second the values.
    *reinterpret_cast<uint2*>((half == 0 ? a.keys : a.values) + (head * kDim + key) * kSvdRank) =
        make_uint2(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16));
    float* const out = a.residual + head * kTile + offset;
#pragma unroll
    for (int i = 0; i < kDim / 2; ++i) {
      float fit = left[0] * static_cast<float>(vectors[i * kSvdRank]);
#pragma unroll
      for (int r = 1; r < kSvdRank; ++r) {
        fit = fmaf(left[r], static_cast<float>(vectors[i * kSvdRank + r]), fit);
      }
      out[i * kDim] = cell[i] - fit;
      if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
    if (t == 0) a.status[head] = kSvdOk;
    return;
  }
}

}  // namespace
}  // namespace gdn

namespace gdn {
namespace {

int32_t launch_exact_svd(void* stream, const float* provider, float* residual,
                         int8_t* quantized, float* smoothing, float* value_scales,
                         uint16_t* compensator_keys, uint16_t* compensator_values,
                         int32_t* status, uint64_t heads, uint32_t max_sweeps) {
  if (provider == nullptr || residual == nullptr || quantized == nullptr ||
      smoothing == nullptr || value_scales == nullptr || compensator_keys == nullptr ||
      compensator_values == nullptr || status == nullptr || heads == 0 || heads > kMaxGrid ||
      max_sweeps == 0 || max_sweeps > static_cast<uint32_t>(kMaxSweeps) ||
      !aligned16(provider, residual, quantized, smoothing, value_scales, compensator_keys,
                 compensator_values, status)) {
    return kStatusInvalidArgument;
  }
  // The direct form takes the default sweep limit; a caller's own limit means
  // Jacobi sweeps.  Behind the direct form one Jacobi workgroup per CU (as many
  // as run at once) serves the heads it left pending.
  const bool direct = max_sweeps == static_cast<uint32_t>(kMaxSweeps);
  const SvdArgs args{provider, residual, compensator_keys, compensator_values, status, heads,
                     static_cast<int>(max_sweeps), direct};
  void* kernel_args[] = {const_cast<SvdArgs*>(&args)};
  const auto run = [&](const void* kernel, uint64_t grid, int threads, size_t lds) {
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(lds)) == hipSuccess &&
           hipLaunchKernel(kernel, dim3(static_cast<uint32_t>(grid)), dim3(threads), kernel_args,
                           lds, static_cast<hipStream_t>(stream)) == hipSuccess;
  };
  if (direct && !run(reinterpret_cast<const void*>(exact_svd_direct_kernel), heads,
                     kDirectThreads, sizeof(DirectShared))) {
    return kStatusLaunchFailed;
  }
  const uint64_t jacobi_grid = direct && heads > kCus ? kCus : heads;
  if (!run(reinterpret_cast<const void*>(exact_svd_jacobi_kernel), jacobi_grid, kSvdThreads,
           sizeof(SvdShared))) {
    return kStatusLaunchFailed;
  }
  return statecentric_gdn_state_codec_encode_launch_v4(stream, residual, quantized, smoothing,
                                                      value_scales, heads, kValueKey);
}

}  // namespace
}  // namespace gdn

// The exact-SVD initializer for a batch of provider heads.
extern "C" int32_t statecentric_gdn_state_codec_exact_svd_boundary_launch_v1(
    void* stream, const float* provider, float* residual, int8_t* quantized, float* smoothing,
    float* value_scales, uint16_t* compensator_keys, uint16_t* compensator_values,
    int32_t* status, uint64_t heads) {
  return gdn::launch_exact_svd(stream, provider, residual, quantized, smoothing, value_scales,
                               compensator_keys, compensator_values, status, heads,
                               gdn::kMaxSweeps);
}

// The same with a caller-chosen sweep limit.
extern "C" int32_t statecentric_gdn_state_codec_exact_svd_boundary_sweeps_launch_v1(
    void* stream, const float* provider, float* residual, int8_t* quantized, float* smoothing,
    float* value_scales, uint16_t* compensator_keys, uint16_t* compensator_values,
    int32_t* status, uint64_t heads, uint32_t max_sweeps) {
  return gdn::launch_exact_svd(stream, provider, residual, quantized, smoothing, value_scales,
                               compensator_keys, compensator_values, status, heads, max_sweeps);
}
