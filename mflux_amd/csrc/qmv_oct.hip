// Quantized matvec for one to sixteen activation rows on gfx950, eight weight rows
// at a time on the int8 matrix-core instruction:
//   y[0:M, n] = x[0:M] . dequant(W[n]) (+ bias),  8-bit codes, groups of 64.
// The adaLN modulation call of every DiT block
// (src/mflux/models/flux/model/flux_transformer/ada_layer_norm_zero.py:12,
// src/mflux/models/qwen/model/qwen_transformer/qwen_transformer_block.py:36-37).
//
// v_mfma_i32_16x16x64_i8 multiplies A [16 x 64] by B [64 x 16]; lane (j, q) =
// (lane % 16, lane / 16) supplies 16 bytes of A's row j and of B's column j, both
// at k 16 q .. 16 q + 15, and receives D[4 q .. 4 q + 3][j].  Here
//   - B's column j is weight row j / 2 of a block of eight rows, over the 64 k of
//     HALF j % 2 of a 128-byte step: the lane's 16 bytes are piece 4 (j % 2) + q of
//     the row's 128 bytes, so one load instruction fetches eight rows x 128
//     contiguous bytes (eight whole cache lines; 16 rows x 64 bytes, the
//     instruction's natural operand, is half lines and measurably slower);
//   - A's rows 0..7 are x over the first half of the step, rows 8..15 over the
//     second half: activation row m as 15-bit fixed point (xq = rint(x * 2^e)),
//     high bytes in row 2 m, low bytes in row 2 m + 1.  Of D, column j's rows
//     0..7 (j even) or 8..15 (j odd) are the products that belong together; the
//     others pair a half of the weights with the other half of x and are dropped.
//     Up to four activation rows cost what one does.
//   - a code enters as the signed byte code - 128 (one XOR per word); a half step
//     is one group of 64 codes, so per instruction and lane, with Sx the sum of xq
//     over the group's 64 k,
//         d = 256 D_high + D_low + 128 Sx        (int32, exactly sum(xq code))
//         acc += scale * d + bias * Sx           (float32)
//     about 17 vector instructions per KiB of weights and no conversion of a code
//     to floating point.
// One workgroup of eight wavefronts per compute unit takes a contiguous run of
// blocks; wavefront w owns eighth w of K (its part of the image of x stays in
// registers: no wavefront waits for another before the end), with the loads of
// three blocks in flight in three register sets, all unconditional so that every
// wait leaves exactly the younger loads in flight.  The eight partial sums of a
// block meet in LDS at the end of the run, where each thread adds up one output.
// Calls that multiplied x as it is before (oct_wide(): more than four rows, two to four on
// some row lengths) keep three bytes of it, 23 bits: A's rows 4 i .. 4 i + 2 are the bytes
// of one activation row, two rows to an instruction, high and lower bytes are summed apart
// as integers and joined in float32.
// Bound by HBM, and from five rows on by the image of x in front of the first block:
// 3072 -> 18432 takes 11.4 us with one row, 14.7 with eight (24.5 on the kernel that
// dequantises).  Distance from float64 of a float32 output, rows with one element in 128
// at 300 times the others: 2e-7 of the norm with three bytes, 3.4e-4 with two; with the
// rounded weights of the kernels that dequantise 1.6e-3 in bfloat16, 2e-4 in float16.
// Rows whose steps do not come in eights are split over ten wavefronts (K = 2560, 3840).
#include <type_traits>

#include "qmv_oct_common.h"

namespace mfq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kOctRows = 8;       // weight rows per block
constexpr int kOctSets = 3;       // blocks in flight per wavefront
constexpr int kOctMaxBlocks = 12;  // blocks per workgroup (their partial sums wait in LDS)
constexpr int kOctLongRun = 9;    // blocks per workgroup when a compute unit's share exceeds that

constexpr int kDppXor1 = 0xB1;         // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;         // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <- lane 7-i of its half row
constexpr int kDppMirror = 0x140;      // lane i <- lane 15-i of its row

template <int kCtrl>
__device__ inline int oct_dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xf, 0xf, false);
}
// sum over the lane's row of 16 lanes, in every lane of the row
__device__ inline int oct_row16_sum(int v) {
  v += oct_dpp<kDppXor1>(v);
  v += oct_dpp<kDppXor2>(v);
  v += oct_dpp<kDppHalfMirror>(v);
  v += oct_dpp<kDppMirror>(v);
  return v;
}
__device__ inline int oct_wave_max(int v) {
  v = max(v, oct_dpp<kDppXor1>(v));
  v = max(v, oct_dpp<kDppXor2>(v));
  v = max(v, oct_dpp<kDppHalfMirror>(v));
  v = max(v, oct_dpp<kDppMirror>(v));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <int kSteps>
struct ScaleWindow {
  uint32_t d[kSteps];  // dword s: the scales (or biases) of the two halves of step s
};

// K = 128 kWaves kSteps, kSteps 128-byte steps per wavefront and row; kM: activation rows the image is built for
// (1, 2, 4 or 8; other M run as the next of these with their last row repeated, more than kM on several workgroups).
// kWide: three bytes per element of x instead of two.
template <typename T, int kWaves, int kSteps, int kM, bool kWide, bool kSilu>
__global__ __launch_bounds__(64 * kWaves) void qmv_oct_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint16_t* __restrict__ bias, void* __restrict__ y, int y_is_f32, int M,
    int N, int blocks_per_wg) {
  constexpr int K = 128 * kWaves * kSteps;
  constexpr int kSlice = 128 * kSteps;       // bytes (= codes) per row and wavefront
  constexpr int kGroups = K / 64;
  constexpr int kPitch = kSlice + 16;        // image rows in LDS
  constexpr int kBytes = kWide ? 3 : 2;
  constexpr int kPasses = kWide ? kM / 2 : 1;  // instructions per step: two activation rows each, or up to four
  constexpr int kImageRows = kBytes * kM;
  constexpr int kImageBytes = oct_image_bytes(kWide, kM, 8, kPitch, 2 * kSteps);
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int j = lane & 15, q = lane >> 4;
  const int n8 = j >> 1, h = j & 1;
  char* image = lds + wave * kImageBytes;
  int2* sums = reinterpret_cast<int2*>(image + kImageRows * kPitch);  // of xq: high bytes, the rest (narrow: all)
  float* partials = reinterpret_cast<float*>(lds + kWaves * kImageBytes);  // [block][wavefront][oct_partials()]
  constexpr int kPartials = oct_partials(kWide, kM, 8);
  int run = blockIdx.x;
  if constexpr (kWide) {
    const int m0 = oct_run_and_first_row<kM>(M, run);
    x += (size_t)m0 * K;
    y = static_cast<char*>(y) + (size_t)m0 * N * (y_is_f32 ? 4 : 2);
    M = min(kM, M - m0);
  }

  const int n_blocks_all = N / kOctRows;
  const int blk_first = run * blocks_per_wg;
  if (kWide && blk_first >= n_blocks_all) return;  // (runs are dealt out in eights)
  const int n_blocks = min(blocks_per_wg, n_blocks_all - blk_first);
  const int blk_last = blk_first + n_blocks - 1;

  // the output this thread will add up at the end (block, weight row, activation row), and its layer bias:
  // requested now, with everything else, so that nothing is fetched behind the last barrier
  constexpr int kOuts = (kOctMaxBlocks * kOctRows * (kM > 4 ? kM : 4) + 64 * kWaves - 1) / (64 * kWaves);
  uint16_t out_bias[kOuts];
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = (int)threadIdx.x + i * 64 * kWaves;
    const int64_t row = (int64_t)(blk_first + min(o / M / kOctRows, n_blocks - 1)) * kOctRows + (o / M) % kOctRows;
    out_bias[i] = (bias ? bias : scales)[row];
  }

  // ---- requests: x first (it is needed first, and loads return in order), the first block behind it ----
  constexpr int kChunks = (32 * kSteps + 63) / 64;  // chunks of 4 consecutive k per lane and activation row
  uint2 raw[kM][kChunks];
#pragma unroll
  for (int m = 0; m < kM; ++m)
#pragma unroll
    for (int t = 0; t < kChunks; ++t) {
      const int c = min(lane + 64 * t, 32 * kSteps - 1);
      raw[m][t] = *reinterpret_cast<const uint2*>(x + (size_t)min(m, M - 1) * K + wave * kSlice + 4 * c);
    }

  const char* wlane = reinterpret_cast<const char*>(wq) + (size_t)n8 * K + wave * kSlice + 16 * (4 * h + q);
  const char* slane = reinterpret_cast<const char*>(scales) + ((size_t)n8 * kGroups + wave * 2 * kSteps) * 2;
  const char* blane = reinterpret_cast<const char*>(biases) + ((size_t)n8 * kGroups + wave * 2 * kSteps) * 2;
  u32x4 wv[kOctSets][kSteps];
  ScaleWindow<kSteps> sw[kOctSets], bw[kOctSets];
  // every load is unconditional (a block past the run's end is its last block again)
  auto issue = [&](int set, int blk) __attribute__((always_inline)) {
    const size_t b = (size_t)min(blk, blk_last);
    sw[set] = *reinterpret_cast<const ScaleWindow<kSteps>*>(slane + b * (kOctRows * kGroups * 2));
    bw[set] = *reinterpret_cast<const ScaleWindow<kSteps>*>(blane + b * (kOctRows * kGroups * 2));
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
      // (streaming loads: left to the default cache policy the same call takes 1.2 us longer)
      wv[set][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wlane + b * (kOctRows * K) + 128 * s));
  };
  // the first block now, the other two behind the image of x: with two wavefronts on a SIMD the older one's
  // requests are served first, and all three blocks at once would set the younger one back by their whole length
  issue(0, blk_first);

  // ---- the integer image of this wavefront's eighth of x ------------------------------------------------
  // One power of two per activation row and eighth of K: the eighths' sums are scaled back before they meet,
  // so the wavefronts need not agree on it and nobody waits for anybody here.
  float unscale_m[kM];  // narrow: the factor, wide: the exponent
#pragma unroll
  for (int m = 0; m < kM; ++m) {
    int amax = 0;
#pragma unroll
    for (int t = 0; t < kChunks; ++t) {
      if constexpr (kSilu) {
        raw[m][t].x = oct_silu<T, kWide>(raw[m][t].x);
        raw[m][t].y = oct_silu<T, kWide>(raw[m][t].y);
      }
      amax = max(amax, max(mag_bits(raw[m][t].x), mag_bits(raw[m][t].y)));
    }
    amax = oct_wave_max(amax);
    // an infinity or NaN anywhere in a row of x: every output of that row is NaN (through this eighth's sums)
    const int e = kWide ? wide_exponent<T>(amax) : scale_exponent<T>(amax);
    const float mult = kWide ? 0.f : pow2(e);
    unscale_m[m] = not_finite<T>(amax) ? __builtin_nanf("") : kWide ? __builtin_amdgcn_ldexpf(1.f, -e) : pow2(-e);
#pragma unroll
    for (int t = 0; t < kChunks; ++t) {
      const int c = lane + 64 * t;
      const bool in = c < 32 * kSteps;
      uint32_t hi, mid = 0, lo;
      if constexpr (kWide)
        split4_wide<T>(raw[m][t].x, raw[m][t].y, e, hi, mid, lo);
      else
        split4<T>(raw[m][t].x, raw[m][t].y, mult, hi, lo);
      if (in) {
        uint32_t* row = reinterpret_cast<uint32_t*>(image + kBytes * m * kPitch + 4 * c);
        row[0] = hi;
        if constexpr (kWide) row[kPitch / 4] = mid;
        row[(kBytes - 1) * (kPitch / 4)] = lo;
      }
      // the sum of xq over a half step's 64 k: its 16 chunks are the 16 lanes of a row of lanes
      const int dot_hi = __builtin_amdgcn_sdot4((int)hi, 0x01010101, 0, false);
      const int dot_lo = __builtin_amdgcn_sdot4((int)lo, 0x01010101, 0, false);
      const int dot_mid = kWide ? __builtin_amdgcn_sdot4((int)mid, 0x01010101, 0, false) : dot_hi;
      const int rest = oct_row16_sum(in ? dot_mid * 256 + dot_lo : 0);
      const int high = kWide ? oct_row16_sum(in ? dot_hi : 0) : 0;
      if (j == 0 && in) sums[m * 2 * kSteps + (c >> 4)] = make_int2(high, rest);
    }
  }
  // (LDS written and read by this wavefront only: program order holds)
  // this lane's A operands, pass p.  Two bytes: image row j % 8 over half j / 8 of every step (image rows past 2 kM:
  // any row, their results are never read).  Three: activation row 2 p + (j % 8) / 4, byte j % 4 (the fourth: the
  // third again, never read).
  // They stay in registers up to twelve of them (each four); otherwise every block reads them again, four times its
  // weights' bytes, a third of what the LDS delivers in the time the weights take (4096 -> 24576, eight rows: 25.8 us,
  // 29.0 on two workgroups of four).
  constexpr bool kHeld = kPasses * kSteps <= 12;
  const int arow = (kWide ? 3 * ((j >> 2) & 1) + min(j & 3, 2) : j & 7 & (kImageRows - 1)) * kPitch + 64 * (j >> 3) + 16 * q;
  i32x4 xa[kHeld ? kPasses : 1][kHeld ? kSteps : 1];
  const auto a_operand = [&](int p, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const i32x4*>(image + arow + 6 * p * kPitch + 128 * s);
  };
  if constexpr (kHeld) {
#pragma unroll
    for (int p = 0; p < kPasses; ++p)
#pragma unroll
      for (int s = 0; s < kSteps; ++s) xa[p][s] = a_operand(p, s);
  }
  // results: register r of lane (j, q) is A's row 4 q + r against column j.  Of use where q / 2 == j % 2.  Two bytes:
  // activation rows 2 (q % 2) (registers 0, 1: high, low bytes) and 2 (q % 2) + 1 (registers 2, 3); three:
  // activation row 2 p + q % 2 (registers 0, 1, 2).
  constexpr bool kTwo = !kWide && kM > 1;  // one activation row: registers 2 and 3 hold nothing of use
  // the sums of xq over this lane's half steps: as float for the bias term, and 128 times them as integers
  // (a code enters the matrix instruction as code - 128; adding 128 sum(xq) to its result gives sum(xq code))
  float sx_a[kPasses][kSteps], sx_b[kPasses][kSteps], us_a[kPasses], us_b[kPasses];
  int sx128_a[kPasses][kSteps], sx128_b[kPasses][kSteps];  // wide: of the lower bytes, of the high ones
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    if constexpr (kWide) {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int2 sum = sums[(2 * p + (q & 1)) * 2 * kSteps + 2 * s + h];
        sx_a[p][s] = (float)(sum.x * 65536 + sum.y);  // 64 elements below 2^23
        sx128_a[p][s] = 128 * sum.y;
        sx128_b[p][s] = 128 * sum.x;
      }
      us_a[p] = unscale_m[2 * p];
      us_a[p] = (q & 1) ? unscale_m[2 * p + 1] : us_a[p];
    } else {
      const int m_a = (2 * (q & 1)) & (kM - 1), m_b = (2 * (q & 1) + 1) & (kM - 1);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int sum_a = sums[m_a * 2 * kSteps + 2 * s + h].y;
        const int sum_b = kTwo ? sums[m_b * 2 * kSteps + 2 * s + h].y : 0;
        sx_a[p][s] = (float)sum_a;
        sx_b[p][s] = (float)sum_b;
        sx128_a[p][s] = 128 * sum_a;
        sx128_b[p][s] = 128 * sum_b;
      }
      us_a[p] = unscale_m[0];
      us_b[p] = unscale_m[kTwo ? 1 : 0];
      if constexpr (kM > 2) {
        us_a[p] = (q & 1) ? unscale_m[2] : us_a[p];
        us_b[p] = (q & 1) ? unscale_m[3] : us_b[p];
      }
    }
  }

#pragma unroll
  for (int t = 1; t < kOctSets; ++t) issue(t, blk_first + t);
  auto consume = [&](int set, int slot) __attribute__((always_inline)) {
    float acc_a[kPasses], acc_b[kPasses];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) acc_a[p] = 0.f, acc_b[p] = 0.f;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      i32x4 wb;
#pragma unroll
      for (int k = 0; k < 4; ++k) wb[k] = (int)(wv[set][s][k] ^ 0x80808080u);  // code - 128 as signed bytes
      const float sc = T::to_f32((uint16_t)(h ? sw[set].d[s] >> 16 : sw[set].d[s]));
      const float bi = T::to_f32((uint16_t)(h ? bw[set].d[s] >> 16 : bw[set].d[s]));
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        const i32x4 zero = {0, 0, 0, 0};
        i32x4 a;
        if constexpr (kHeld) a = xa[p][s];
        else a = a_operand(p, s);
        const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, wb, zero, 0, 0, 0);
        if constexpr (kWide) {
          // sum(xq code) over the half step's group: high and lower bytes exact, joined in float32
          const int dl = d[1] * 256 + d[2] + sx128_a[p][s], dh = d[0] + sx128_b[p][s];
          acc_a[p] = __builtin_fmaf(sc, __builtin_fmaf(65536.f, (float)dh, (float)dl), acc_a[p]);
          acc_a[p] = __builtin_fmaf(bi, sx_a[p][s], acc_a[p]);
        } else {
          // sum(xq code) over the half step's group, exact: high and low bytes of xq joined as integers
          const int da = d[0] * 256 + d[1] + sx128_a[p][s];
          acc_a[p] = __builtin_fmaf(sc, (float)da, acc_a[p]);
          acc_a[p] = __builtin_fmaf(bi, sx_a[p][s], acc_a[p]);
          if constexpr (kTwo) {
            const int db = d[2] * 256 + d[3] + sx128_b[p][s];
            acc_b[p] = __builtin_fmaf(sc, (float)db, acc_b[p]);
            acc_b[p] = __builtin_fmaf(bi, sx_b[p][s], acc_b[p]);
          }
        }
      }
    }
    float* dst = partials + (slot * kWaves + wave) * kPartials;
    if constexpr (kWide) {
      if ((q >> 1) == h) {  // the useful half of the lanes, one value per pass
#pragma unroll
        for (int p = 0; p < kPasses; ++p) dst[32 * p + 2 * j + (q & 1)] = acc_a[p] * us_a[p];
      }
    } else {
      reinterpret_cast<float2*>(dst)[lane] = make_float2(acc_a[0] * us_a[0], acc_b[0] * us_b[0]);
    }
  };

  // Three blocks per trip, one per register set, and between the arithmetic of two blocks the requests for the
  // block three further on; the last trip requests nothing (loads still in flight at the end would hold their
  // registers, and the adding-up below, until they land).  A block past the run's end is computed again
  // into a slot of its own that nobody reads.
  int b = 0;
  for (; b + kOctSets < n_blocks; b += kOctSets) {
#pragma unroll
    for (int t = 0; t < kOctSets; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      consume(t, b + t);
      __builtin_amdgcn_sched_barrier(0);
      issue(t, blk_first + b + t + kOctSets);
    }
  }
#pragma unroll
  for (int t = 0; t < kOctSets; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    consume(t, min(b + t, n_blocks));
  }
  __syncthreads();

  // ---- one output per thread: block, weight row, activation row; 8 eighths x 2 halves of partial sums --------
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = (int)threadIdx.x + i * 64 * kWaves;
    const int out_m = o % M, out_row8 = (o / M) % kOctRows, out_blk = o / M / kOctRows;
    const bool mine = out_blk < n_blocks;
    const int64_t out_row = (int64_t)(blk_first + out_blk) * kOctRows + out_row8;
    float v = 0.f;
    if (mine) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int src_j = 2 * out_row8 + hh;
          const float* src = partials + (out_blk * kWaves + w) * kPartials;
          if constexpr (kWide) {
            v += src[32 * (out_m >> 1) + 2 * src_j + (out_m & 1)];
          } else {
            const float2 p = reinterpret_cast<const float2*>(src)[src_j + 16 * (2 * hh + (out_m >> 1))];
            v += (out_m & 1) ? p.y : p.x;
          }
        }
    }
    // an infinity in x is an infinity of the weight's sign in y, as the kernels that dequantise give it
    if constexpr (kWide) v = oct_keep_infinities<T, 8, kSilu>(mine, v, x, wq, scales, biases, out_m, out_row, K, lane);
    const float bias_v = T::to_f32(out_bias[i]);
    if (mine && y_is_f32) {
      reinterpret_cast<float*>(y)[(int64_t)out_m * N + out_row] = bias ? v + bias_v : v;
    } else if (mine) {
      const uint16_t h0 = T::from_f32(v);
      const uint16_t h1 = T::from_f32(T::to_f32(h0) + bias_v);  // second rounding, as a separate add would do
      reinterpret_cast<uint16_t*>(y)[(int64_t)out_m * N + out_row] = bias ? h1 : h0;
    }
  }
}

template <typename T, int kWaves, int kSteps, int kM, bool kWide, bool kSilu>
int launch_oct(const void* x, int64_t M, const uint32_t* wq, const void* scales, const void* biases, const void* bias,
               int64_t N, void* y, int y_dtype, hipStream_t stream) {
  auto kernel = qmv_oct_kernel<T, kWaves, kSteps, kM, kWide, kSilu>;
  constexpr int kImageBytes = oct_image_bytes(kWide, kM, 8, 128 * kSteps + 16, 2 * kSteps);
  constexpr int kPerBlock = kWaves * oct_partials(kWide, kM, 8) * 4;
  static PerDeviceInt configured;
  return launch_oct_runs<kWaves, kM>(kernel, configured, kWaves * kImageBytes, kPerBlock, kOctRows, kOctMaxBlocks,
                                     kOctLongRun, x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
}

// Activation rows the image is built for: 1, 2, 4 or kMost (0: four at most), the last two with their last rows repeated.
template <typename T, int kWaves, int kSteps, int kMost, bool kSilu>
int launch_oct_rows(const void* x, int64_t M, const uint32_t* wq, const void* scales, const void* biases,
                    const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  constexpr int K = 128 * kWaves * kSteps;
  if (M == 1) return launch_oct<T, kWaves, kSteps, 1, false, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  constexpr bool kWide = oct_wide(2, K, 8);
  if (M == 2) return launch_oct<T, kWaves, kSteps, 2, kWide, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  if (M <= 4) return launch_oct<T, kWaves, kSteps, 4, kWide, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  if constexpr (!kSilu && kMost > 0)
    return launch_oct<T, kWaves, kSteps, kMost, true, false>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  return MFQ_EUNSUPPORTED;
}

// The split of K: wavefronts times 128-byte steps of each, and the rows a workgroup takes of more than four: eight where
// that fits (10 x 3: 168 registers to a wavefront, 78 us of spills instead of 31, and no less from LDS; 8 x 6: no room in
// LDS for more than two blocks' sums), 0 where oct_takes() ends at four.
template <typename T, bool kSilu>
int launch_oct_steps(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales, const void* biases,
                     const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  switch (K) {
    case 256: return launch_oct_rows<T, 2, 1, 0, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 1024: return launch_oct_rows<T, 8, 1, 0, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 2048: return launch_oct_rows<T, 8, 2, 8, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 2560: return launch_oct_rows<T, 10, 2, 8, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 3072: return launch_oct_rows<T, 8, 3, 8, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 3840: return launch_oct_rows<T, 10, 3, 4, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 4096: return launch_oct_rows<T, 8, 4, 8, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 6144: return launch_oct_rows<T, 8, 6, 4, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    default: return MFQ_EUNSUPPORTED;
  }
}

}  // namespace

// Shapes this kernel takes: 8-bit codes in groups of 64, up to sixteen activation rows, the K that
// launch_oct_steps splits, whole eights of weight rows, x and the weights 16-byte aligned, scales and biases
// 4-byte aligned.
bool qmv_oct_covers(int64_t M, int64_t K, int64_t N, int gs, int bits, const void* x, const void* scales,
                    const void* biases) {
  if (!(bits == 8 && gs == 64 && oct_takes(M, K, bits) && N % kOctRows == 0)) return false;
  return aligned16(x) && ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) == 0;
}

int launch_qmv_oct(const void* x, int dtype, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                   const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype,
                   hipStream_t stream, bool silu) {
  if (!qmv_oct_covers(M, K, N, gs, bits, x, scales, biases)) return MFQ_EUNSUPPORTED;
  if (dtype != MFQ_BF16 && dtype != MFQ_F16) return MFQ_EDTYPE;
  const bool bf = dtype == MFQ_BF16;
  if (silu)
    return bf ? launch_oct_steps<BF16, true>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream)
              : launch_oct_steps<F16, true>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream);
  return bf ? launch_oct_steps<BF16, false>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream)
            : launch_oct_steps<F16, false>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream);
}

}  // namespace mfq
