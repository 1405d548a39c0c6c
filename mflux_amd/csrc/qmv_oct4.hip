// Quantized matvec for one to sixteen activation rows and 4-bit codes on gfx950,
// eight weight rows at a time on the int8 matrix-core instruction: the scheme
// of qmv_oct.hip (which see) for packed nibbles,
//   y[0:M, n] = x[0:M] . dequant(W[n]) (+ bias),  groups of 64.
// The adaLN modulation call of every DiT block of a 4-bit model
// (src/mflux/models/qwen/model/qwen_transformer/qwen_transformer_block.py:36-37,
// src/mflux/models/flux/model/flux_transformer/ada_layer_norm_zero.py:12).
//
// A load instruction again fetches eight rows x 128 contiguous bytes, now 256
// codes of each row: four groups.  Lane (j, q) = (lane % 16, lane / 16) holds
// piece 4 (j % 2) + q of row j / 2, 32 codes; their even nibbles (w & 0x0f..) and
// odd nibbles ((w >> 4) & 0x0f..) are the B operands of two
// v_mfma_i32_16x16x64_i8 that add into the same sums.  Column j's four lanes
// cover TWO groups (pieces 2g, 2g + 1 are group g of the column's half row), so
// the A operand tells them apart: A's row 8 h + 4 g + 2 m + l is activation row
// m (two of them per pair of instructions), high (l = 0) or low byte of its
// 15-bit fixed point, over the k of half h -- and zero in the lanes of the
// other group.  Column j's useful sums are rows 8 (j % 2) .. + 7: lane
// (j, 2 (j % 2) + g) receives group g's for both activation rows, one scale and
// bias per lane and step as in the 8-bit kernel.  Nibbles are non-negative, so
// nothing is offset:
//     d = 256 D_high + D_low      (int32, exactly sum(xq code) over the group)
//     acc += scale * d + bias * sum(xq)
// Rows three and four are another pair of instructions on the same B operands.  Calls
// that multiplied x as it is before (oct_wide()) keep three bytes of it: A's row
// 8 h + 4 g + l is byte l of ONE activation row, and d = 65536 D_high + 256 D_mid + D_low
// is put together in float32.  More than four activation rows take a workgroup to every
// three or four.  3072 -> 18432 takes 7.4 us with one row, 8.4 with four, 17 with eight, where
// the vector instructions of the bytes are as long as the loads (31 on the kernel that
// dequantises).  Work layout, register sets, the meeting of the wavefronts' partial sums
// at the end: qmv_oct.hip's, with K split over kWaves wavefronts.
#include <type_traits>

#include "qmv_oct_common.h"

namespace mfq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows4 = 8;        // weight rows per block
constexpr int kSets4 = 3;        // blocks in flight per wavefront
constexpr int kMaxBlocks4 = 12;  // blocks per workgroup (their partial sums wait in LDS)
constexpr int kLongRun4 = 9;     // blocks per workgroup when a compute unit's share exceeds that

constexpr int kDppXor1 = 0xB1;         // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;         // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <- lane 7-i of its half row
constexpr int kDppMirror = 0x140;      // lane i <- lane 15-i of its row

template <int kCtrl>
__device__ inline int oct4_dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xf, 0xf, false);
}
// sum over the lane's eight (lanes 8 i .. 8 i + 7), in every lane of it
__device__ inline int oct4_sum8(int v) {
  v += oct4_dpp<kDppXor1>(v);
  v += oct4_dpp<kDppXor2>(v);
  v += oct4_dpp<kDppHalfMirror>(v);
  return v;
}
__device__ inline int oct4_wave_max(int v) {
  v = max(v, oct4_dpp<kDppXor1>(v));
  v = max(v, oct4_dpp<kDppXor2>(v));
  v = max(v, oct4_dpp<kDppHalfMirror>(v));
  v = max(v, oct4_dpp<kDppMirror>(v));
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <int kSteps>
struct ScaleWindow4 {
  uint32_t d[2 * kSteps];  // dword 2 s + h: the scales (or biases) of the two groups of half h of step s
};

// kWaves: wavefronts per workgroup, each with kSteps 128-byte steps of every row (K = 256 kWaves kSteps codes);
// kM: activation rows the image is built for (1, 2, 3 or 4; other M run as the next of these with their last row repeated, more than
// kM on several workgroups).  kWide: three bytes per element of x instead of two.
template <typename T, int kWaves, int kSteps, int kM, bool kWide, bool kSilu>
__global__ __launch_bounds__(64 * kWaves) void qmv_oct4_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint16_t* __restrict__ bias, void* __restrict__ y, int y_is_f32, int M,
    int N, int blocks_per_wg) {
  constexpr int K = 256 * kWaves * kSteps;
  constexpr int kRowBytes = K / 2;
  constexpr int kSlice = 128 * kSteps;       // bytes per row and wavefront: 2 kSlice codes
  constexpr int kGroups = K / 64;
  constexpr int kBytes = kWide ? 3 : 2;
  constexpr int kPasses = kWide ? kM : kM > 2 ? kM / 2 : 1;  // pairs of instructions per step: one activation row each, or two
  constexpr int kImageRows = kBytes * kM;    // (activation row, byte from the top)
  constexpr int kPitch = 2 * kSlice + 32;    // an image row: kSlice bytes of even k, kSlice of odd k
  constexpr int kImageBytes = oct_image_bytes(kWide, kM, 4, kPitch, 4 * kSteps);
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int j = lane & 15, q = lane >> 4;
  const int n8 = j >> 1, h = j & 1;
  char* image = lds + wave * kImageBytes;
  float* sums = reinterpret_cast<float*>(image + kImageRows * kPitch);  // [activation row][group of the slice]
  float* partials = reinterpret_cast<float*>(lds + kWaves * kImageBytes);  // [block][wavefront][oct_partials()]
  constexpr int kPartials = oct_partials(kWide, kM, 4);
  int run = blockIdx.x;
  if constexpr (kWide) {
    const int m0 = oct_run_and_first_row<kM>(M, run);
    x += (size_t)m0 * K;
    y = static_cast<char*>(y) + (size_t)m0 * N * (y_is_f32 ? 4 : 2);
    M = min(kM, M - m0);
  }

  const int n_blocks_all = N / kRows4;
  const int blk_first = run * blocks_per_wg;
  if (kWide && blk_first >= n_blocks_all) return;  // (runs are dealt out in eights)
  const int n_blocks = min(blocks_per_wg, n_blocks_all - blk_first);
  const int blk_last = blk_first + n_blocks - 1;

  // the outputs this thread will add up at the end (block, weight row, activation row), and their layer bias:
  // requested now, with everything else, so that nothing is fetched behind the last barrier
  constexpr int kOuts = (kMaxBlocks4 * kRows4 * (kM > 4 ? kM : 4) + 64 * kWaves - 1) / (64 * kWaves);
  uint16_t out_bias[kOuts];
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = (int)threadIdx.x + i * 64 * kWaves;
    const int64_t row = (int64_t)(blk_first + min(o / M / kRows4, n_blocks - 1)) * kRows4 + (o / M) % kRows4;
    out_bias[i] = (bias ? bias : scales)[row];
  }

  // ---- requests: x first (it is needed first, and loads return in order), the first block behind it ----
  // chunk c = 8 consecutive k (16 bytes of x): one word of codes
  constexpr int kChunks = (32 * kSteps + 63) / 64;
  u32x4 raw[kM][kChunks];
#pragma unroll
  for (int m = 0; m < kM; ++m)
#pragma unroll
    for (int t = 0; t < kChunks; ++t) {
      const int c = min(lane + 64 * t, 32 * kSteps - 1);
      raw[m][t] = *reinterpret_cast<const u32x4*>(x + (size_t)min(m, M - 1) * K + wave * 2 * kSlice + 8 * c);
    }

  const char* wlane = reinterpret_cast<const char*>(wq) + (size_t)n8 * kRowBytes + wave * kSlice + 16 * (4 * h + q);
  const char* slane = reinterpret_cast<const char*>(scales) + ((size_t)n8 * kGroups + wave * 4 * kSteps) * 2;
  const char* blane = reinterpret_cast<const char*>(biases) + ((size_t)n8 * kGroups + wave * 4 * kSteps) * 2;
  u32x4 wv[kSets4][kSteps];
  ScaleWindow4<kSteps> sw[kSets4], bw[kSets4];
  // every load is unconditional (a block past the run's end is its last block again)
  auto issue = [&](int set, int blk) __attribute__((always_inline)) {
    const size_t b = (size_t)min(blk, blk_last);
    sw[set] = *reinterpret_cast<const ScaleWindow4<kSteps>*>(slane + b * (kRows4 * kGroups * 2));
    bw[set] = *reinterpret_cast<const ScaleWindow4<kSteps>*>(blane + b * (kRows4 * kGroups * 2));
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
      wv[set][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wlane + b * (kRows4 * kRowBytes) + 128 * s));
  };
  issue(0, blk_first);

  // ---- the integer image of this wavefront's part of x: per activation row and byte (high, low) one LDS row,
  // even k in its first kSlice bytes, odd k behind them --------------------------------------------------
  float unscale_m[kM];
#pragma unroll
  for (int m = 0; m < kM; ++m) {
    int amax = 0;
#pragma unroll
    for (int t = 0; t < kChunks; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (kSilu) raw[m][t][i] = oct_silu<T, kWide>(raw[m][t][i]);
        amax = max(amax, mag_bits(raw[m][t][i]));
      }
    amax = oct4_wave_max(amax);
    // an infinity or NaN anywhere in a row of x: every output of that row is NaN (through this part's sums)
    const int e = kWide ? wide_exponent<T>(amax) : scale_exponent<T>(amax);
    const float mult = kWide ? 0.f : pow2(e);
    unscale_m[m] = not_finite<T>(amax) ? __builtin_nanf("") : kWide ? __builtin_amdgcn_ldexpf(1.f, -e) : pow2(-e);
#pragma unroll
    for (int t = 0; t < kChunks; ++t) {
      const int c = lane + 64 * t;
      const bool in = c < 32 * kSteps;
      // raw[..][i] = (x[2 i], x[2 i + 1]): even k in the low halves
      const u32x4 r = raw[m][t];
      const uint32_t ev0 = (r[0] & 0xffffu) | (r[1] << 16), ev1 = (r[2] & 0xffffu) | (r[3] << 16);
      const uint32_t od0 = (r[0] >> 16) | (r[1] & 0xffff0000u), od1 = (r[2] >> 16) | (r[3] & 0xffff0000u);
      uint32_t hi_e, mid_e = 0, lo_e, hi_o, mid_o = 0, lo_o;
      if constexpr (kWide) {
        split4_wide<T>(ev0, ev1, e, hi_e, mid_e, lo_e);
        split4_wide<T>(od0, od1, e, hi_o, mid_o, lo_o);
      } else {
        split4<T>(ev0, ev1, mult, hi_e, lo_e);
        split4<T>(od0, od1, mult, hi_o, lo_o);
      }
      if (in) {
        char* even = image + kBytes * m * kPitch + 4 * c;
        char* odd = even + kSlice + 16;
        *reinterpret_cast<uint32_t*>(even) = hi_e;
        *reinterpret_cast<uint32_t*>(odd) = hi_o;
        if constexpr (kWide) {
          *reinterpret_cast<uint32_t*>(even + kPitch) = mid_e;
          *reinterpret_cast<uint32_t*>(odd + kPitch) = mid_o;
        }
        *reinterpret_cast<uint32_t*>(even + (kBytes - 1) * kPitch) = lo_e;
        *reinterpret_cast<uint32_t*>(odd + (kBytes - 1) * kPitch) = lo_o;
      }
      // the sum of xq over a group's 64 k (below 2^29): its 8 chunks are 8 neighbouring lanes
      const auto sum4 = [](uint32_t a, uint32_t b) __attribute__((always_inline)) {
        return __builtin_amdgcn_sdot4((int)a, 0x01010101, 0, false) + __builtin_amdgcn_sdot4((int)b, 0x01010101, 0, false);
      };
      int part = sum4(hi_e, hi_o) * 256;
      if constexpr (kWide) part = (part + sum4(mid_e, mid_o)) * 256;
      part += sum4(lo_e, lo_o);
      const int total = oct4_sum8(in ? part : 0);
      if ((lane & 7) == 0 && in) sums[m * 4 * kSteps + (c >> 3)] = (float)total;
    }
  }
  // (LDS written and read by this wavefront only: program order holds)
  // this lane's A operands, pass p: A's row j = 8 h' + 4 g + r over half h' = j / 8 of every step, zero unless this
  // lane's k (pieces 2 g, 2 g + 1 of the half: q / 2 == g) belong to group g = (j / 4) % 2.  Two bytes: r = 2 (m % 2) + l
  // is byte l of activation row m = 2 p + r / 2; three: byte r of activation row p (r = 3: byte 2 again, never read)
  i32x4 xa_e[kPasses][kSteps], xa_o[kPasses][kSteps];
  {
    const bool mine = (q >> 1) == ((j >> 2) & 1);
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int row = kWide ? 3 * p + min(j & 3, 2) : 2 * ((2 * p + ((j >> 1) & 1)) & (kM - 1)) + (j & 1);
      const char* arow = image + row * kPitch + 64 * (j >> 3) + 16 * q;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const i32x4 zero = {0, 0, 0, 0};
        xa_e[p][s] = mine ? *reinterpret_cast<const i32x4*>(arow + 128 * s) : zero;
        xa_o[p][s] = mine ? *reinterpret_cast<const i32x4*>(arow + kSlice + 16 + 128 * s) : zero;
      }
    }
  }
  // results: register r of lane (j, q) is A's row 4 q + r against column j.  Of use where q / 2 == j % 2: group
  // g = q % 2 of the column's half.  Two bytes: activation rows 2 p (registers 0, 1: high, low bytes) and 2 p + 1
  // (2, 3); three: activation row p (0, 1, 2)
  constexpr bool kTwo = !kWide && kM > 1;  // one activation row: registers 2 and 3 hold nothing of use
  const int g = q & 1;
  float sx_a[kPasses][kSteps], sx_b[kPasses][kSteps], us_a[kPasses], us_b[kPasses];
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int m_a = kWide ? p : (2 * p) & (kM - 1), m_b = (2 * p + 1) & (kM - 1);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      sx_a[p][s] = sums[m_a * 4 * kSteps + 4 * s + 2 * h + g];
      sx_b[p][s] = kTwo ? sums[m_b * 4 * kSteps + 4 * s + 2 * h + g] : 0.f;
    }
    us_a[p] = unscale_m[m_a];
    us_b[p] = unscale_m[m_b];
  }

#pragma unroll
  for (int t = 1; t < kSets4; ++t) issue(t, blk_first + t);
  auto consume = [&](int set, int slot) __attribute__((always_inline)) {
    float acc_a[kPasses], acc_b[kPasses];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) acc_a[p] = 0.f, acc_b[p] = 0.f;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      i32x4 ev, od;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        ev[k] = (int)(wv[set][s][k] & 0x0f0f0f0fu);
        od[k] = (int)((wv[set][s][k] >> 4) & 0x0f0f0f0fu);
      }
      // (selects between registers named at compile time: an index that depends on the lane would put the windows in memory)
      const uint32_t sd = h ? sw[set].d[2 * s + 1] : sw[set].d[2 * s];
      const uint32_t bd = h ? bw[set].d[2 * s + 1] : bw[set].d[2 * s];
      const float sc = T::to_f32((uint16_t)(g ? sd >> 16 : sd));
      const float bi = T::to_f32((uint16_t)(g ? bd >> 16 : bd));
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        const i32x4 zero = {0, 0, 0, 0};
        i32x4 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa_e[p][s], ev, zero, 0, 0, 0);
        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa_o[p][s], od, d, 0, 0, 0);
        if constexpr (kWide) {
          // sum(xq code) over the group: high and lower bytes exact, joined in float32
          acc_a[p] = __builtin_fmaf(sc, __builtin_fmaf(65536.f, (float)d[0], (float)(d[1] * 256 + d[2])), acc_a[p]);
          acc_a[p] = __builtin_fmaf(bi, sx_a[p][s], acc_a[p]);
        } else {
          // sum(xq code) over the group, exact: high and low bytes of xq joined as integers
          acc_a[p] = __builtin_fmaf(sc, (float)(d[0] * 256 + d[1]), acc_a[p]);
          acc_a[p] = __builtin_fmaf(bi, sx_a[p][s], acc_a[p]);
          if constexpr (kTwo) {
            acc_b[p] = __builtin_fmaf(sc, (float)(d[2] * 256 + d[3]), acc_b[p]);
            acc_b[p] = __builtin_fmaf(bi, sx_b[p][s], acc_b[p]);
          }
        }
      }
    }
    float* dst = partials + (slot * kWaves + wave) * kPartials;
    if constexpr (kWide) {
      if ((q >> 1) == h) {  // the useful half of the lanes
#pragma unroll
        for (int p = 0; p < kPasses; ++p) dst[32 * p + 2 * j + g] = acc_a[p] * us_a[p];
      }
    } else {
#pragma unroll
      for (int p = 0; p < kPasses; ++p)
        reinterpret_cast<float2*>(dst)[64 * p + lane] = make_float2(acc_a[p] * us_a[p], acc_b[p] * us_b[p]);
    }
  };

  // Three blocks per trip, one per register set, and between the arithmetic of two blocks the requests for the
  // block three further on; the last trip requests nothing.  A block past the run's end is computed again
  // into a slot of its own that nobody reads.
  int b = 0;
  for (; b + kSets4 < n_blocks; b += kSets4) {
#pragma unroll
    for (int t = 0; t < kSets4; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      consume(t, b + t);
      __builtin_amdgcn_sched_barrier(0);
      issue(t, blk_first + b + t + kSets4);
    }
  }
#pragma unroll
  for (int t = 0; t < kSets4; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    consume(t, min(b + t, n_blocks));
  }
  __syncthreads();

  // ---- one output per thread: block, weight row, activation row; per wavefront the two halves' two groups -----
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = (int)threadIdx.x + i * 64 * kWaves;
    const int out_m = o % M, out_row8 = (o / M) % kRows4, out_blk = o / M / kRows4;
    const bool mine = out_blk < n_blocks;
    const int64_t out_row = (int64_t)(blk_first + out_blk) * kRows4 + out_row8;
    float v = 0.f;
    if (mine) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int hg = 0; hg < 4; ++hg) {  // half hg / 2, group hg % 2: lane (2 row + half, 2 half + group)
          const int src_j = 2 * out_row8 + (hg >> 1);
          const float* src = partials + (out_blk * kWaves + w) * kPartials;
          if constexpr (kWide) {
            v += src[32 * out_m + 2 * src_j + (hg & 1)];
          } else {
            const float2 p = reinterpret_cast<const float2*>(src)[64 * (out_m >> 1) + src_j + 16 * hg];
            v += (out_m & 1) ? p.y : p.x;
          }
        }
    }
    // an infinity in x is an infinity of the weight's sign in y, as the kernels that dequantise give it
    if constexpr (kWide) v = oct_keep_infinities<T, 4, kSilu>(mine, v, x, wq, scales, biases, out_m, out_row, K, lane);
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
int launch_oct4(const void* x, int64_t M, const uint32_t* wq, const void* scales, const void* biases, const void* bias,
                int64_t N, void* y, int y_dtype, hipStream_t stream) {
  auto kernel = qmv_oct4_kernel<T, kWaves, kSteps, kM, kWide, kSilu>;
  constexpr int kImageBytes = oct_image_bytes(kWide, kM, 4, 256 * kSteps + 32, 4 * kSteps);
  constexpr int kPerBlock = kWaves * oct_partials(kWide, kM, 4) * 4;
  static PerDeviceInt configured;
  return launch_oct_runs<kWaves, kM>(kernel, configured, kWaves * kImageBytes, kPerBlock, kRows4, kMaxBlocks4, kLongRun4,
                                     x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
}

// Activation rows the image is built for: 1, 2 or 4, fours with their last row repeated.  More than four rows: a
// workgroup to every four, or to every three where that makes no more of them (five rows of 3072 -> 18432: 14.8 us, 17.7
// in fours).  Eight to one, with a register image twice as large, measured behind on every row length: 256 -> 15360 14.0
// against 6.6 us, 3072 -> 18432, where it spills, 35 against 17.
template <typename T, int kWaves, int kSteps, bool kSilu>
int launch_oct4_rows(const void* x, int64_t M, const uint32_t* wq, const void* scales, const void* biases,
                     const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  constexpr int K = 256 * kWaves * kSteps;
  if (M == 1) return launch_oct4<T, kWaves, kSteps, 1, false, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  constexpr bool kWide = oct_wide(2, K, 4);
  if (M == 2) return launch_oct4<T, kWaves, kSteps, 2, kWide, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  if (M <= 4) return launch_oct4<T, kWaves, kSteps, 4, kWide, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  if constexpr (!kSilu)
    return (M + 2) / 3 == (M + 3) / 4
               ? launch_oct4<T, kWaves, kSteps, 3, true, false>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream)
               : launch_oct4<T, kWaves, kSteps, 4, true, false>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
  return MFQ_EUNSUPPORTED;
}

template <typename T, bool kSilu>
int launch_oct4_k(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales, const void* biases,
                  const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  // (K = 3072, twelve steps to a row: six wavefronts of two measured ahead of four of three and twelve of one)
  switch (K) {
    case 256: return launch_oct4_rows<T, 1, 1, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 1024: return launch_oct4_rows<T, 4, 1, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 2048: return launch_oct4_rows<T, 8, 1, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 2560: return launch_oct4_rows<T, 5, 2, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 3072: return launch_oct4_rows<T, 6, 2, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 3840: return launch_oct4_rows<T, 5, 3, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 4096: return launch_oct4_rows<T, 8, 2, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    case 6144: return launch_oct4_rows<T, 8, 3, kSilu>(x, M, wq, scales, biases, bias, N, y, y_dtype, stream);
    default: return MFQ_EUNSUPPORTED;
  }
}

}  // namespace

// Shapes this kernel takes: 4-bit codes in groups of 64, up to sixteen activation rows, the K that
// launch_oct4_k splits, whole eights of weight rows, x and the weights 16-byte aligned, scales and biases
// 4-byte aligned.
bool qmv_oct4_covers(int64_t M, int64_t K, int64_t N, int gs, int bits, const void* x, const void* scales,
                     const void* biases) {
  if (!(bits == 4 && gs == 64 && oct_takes(M, K, bits) && N % kRows4 == 0))
    return false;
  return aligned16(x) && ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) == 0;
}

int launch_qmv_oct4(const void* x, int dtype, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                    const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype,
                    hipStream_t stream, bool silu) {
  if (!qmv_oct4_covers(M, K, N, gs, bits, x, scales, biases)) return MFQ_EUNSUPPORTED;
  if (dtype != MFQ_BF16 && dtype != MFQ_F16) return MFQ_EDTYPE;
  const bool bf = dtype == MFQ_BF16;
  if (silu)
    return bf ? launch_oct4_k<BF16, true>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream)
              : launch_oct4_k<F16, true>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream);
  return bf ? launch_oct4_k<BF16, false>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream)
            : launch_oct4_k<F16, false>(x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream);
}

}  // namespace mfq
