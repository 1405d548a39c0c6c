// What the two eight-rows matvec kernels (qmv_oct.hip, qmv_oct4.hip) share on the host and off their main path.
#pragma once
#include "common.h"

namespace mfq {

// The calls the kernels take: row lengths they are built for, up to sixteen activation rows.  Measured against the
// kernels that take these calls otherwise (us, stream of launches on cold weights):
//   one row: K = 1024 .. 4096 in steps of 1024 (11.4 on 3072 -> 18432 at 8 bits); on the other row lengths the
//     one-row kernel of qmv_dot.hip is level or ahead (2560 -> 15360 at 8 bits 9.1 against 9.7, 3840 -> 23040 at 4 bits
//     10.1 against 10.9) unless a quarter or more of its KiB-sized loads lies past the row's end (256 -> 15360 at 8 bits
//     4.6 against 3.5 here, 2560 -> 15360 at 4 bits 7.3 against 6.2);
//   two to four: everywhere (6144 -> 36864 at 8 bits 67 -> 40, 256 -> 15360 at 4 bits 11.4 -> 5.9);
//   five and more, against the kernel that dequantises (qmv.hip): 3072 -> 18432 at 8 bits, five rows 19.7 -> 14.4,
//     sixteen 36.5 -> 25.8; at 4 bits 23.6 -> 14.8 and 59.9 -> 27.7.  8-bit rows of up to 1024 codes stay there: the
//     image of x in front of the first block is most of so short a call (1024 -> 6144, five rows 5.4 there, 6.5 here).
inline bool oct_takes(int64_t M, int64_t K, int bits) {
  if (M < 1 || M > 16) return false;
  const bool even = K == 1024 || K == 2048 || K == 3072 || K == 4096;
  if (!even && K != 256 && K != 2560 && K != 3840 && K != 6144) return false;
  if (M == 1) {
    const int64_t bytes = K * bits / 8, loads = (bytes + 1023) / 1024;
    return even || 4 * bytes <= 3 * 1024 * loads;
  }
  return M <= 4 || bits == 4 || K > 1024;
}

// Whether a call of m rows keeps three bytes of an element of x: the calls that came from kernels on dequantised
// weights (more than four rows; two to four on row lengths the four-rows kernel does not take), which multiplied x as
// it is.  With two bytes, float16 rows with one element in 128 at 300 times the others were 3.4e-4 of the norm from
// float64, 2.0e-4 in those kernels and 2e-7 with three.  The other calls keep the two bytes (15-bit fixed point) of
// the integer kernels they came from.
constexpr bool oct_wide(int64_t m, int64_t K, int bits) {
  return m > 4 || (m > 1 && (K % 1024 != 0 || K > 4096) && !(bits == 8 && K == 256));
}

// LDS of a wavefront's image of x: its rows and, for every `sums_per_row` groups of 64 k of each, the sum of xq.
constexpr int oct_image_bytes(bool wide, int m, int bits, int pitch, int sums_per_row) {
  return ((wide ? 3 : 2) * m * pitch + m * sums_per_row * (bits == 8 ? 8 : 4) + 255) & ~255;
}

// SiLU of a pair: where x keeps three bytes the values are those of the separate activation that these calls had.  Two
// rows take 0.3 to 5 us longer than with silu_pair's sigmoid, four 0.9 to 12 (6144 -> 36864 at 4 bits, 27.4 to 39.6); as
// a launch of its own the activation is 2.7.
template <typename T, bool kWide>
__device__ inline uint32_t oct_silu(uint32_t pair) {
  return kWide ? silu_exact_pair<T>(pair) : silu_pair<T>(pair);
}

// Floats of partial sums per block and wavefront.  Two bytes: a pair per lane and instruction (8 bits: up to four rows
// an instruction, 4 bits: two).  Three: one per lane of the useful half (8 bits: two rows an instruction, 4 bits: one).
constexpr int oct_partials(bool wide, int m, int bits) {
  if (wide) return 32 * (bits == 8 ? m / 2 : m);
  return bits == 4 && m > 2 ? 256 : 128;
}

// Workgroup -> run of weight rows and first activation row.  With more than kM activation rows the workgroups of a run
// are eight apart in the grid, on one XCD and at one time, so that all but the first find the weights in a cache.
template <int kM>
__device__ inline int oct_run_and_first_row(int M, int& run) {
  if (M <= kM) return 0;
  const int groups = (M + kM - 1) / kM, eight = run >> 3;
  run = (eight / groups << 3) + (run & 7);
  return eight % groups * kM;
}

// x . dequant(W[row]) on the weights rounded to the 16-bit type: what an output is whose row of x holds an infinity or
// a NaN, which the integer image cannot.  Called by whole wavefronts: a lane takes every 64th word of codes.
template <typename T, int BITS, bool kSilu>
__device__ __attribute__((noinline)) float oct_plain_dot(const uint16_t* x, const uint32_t* wq, const uint16_t* scales,
                                                         const uint16_t* biases, int64_t row, int K, int lane) {
  constexpr int kPerWord = 32 / BITS;
  typedef uint32_t xwords __attribute__((ext_vector_type(kPerWord / 2)));
  float v = 0.f;
#pragma unroll 4
  for (int k = kPerWord * lane; k < K; k += kPerWord * kWave) {
    const uint32_t codes = wq[(row * K + k) / kPerWord];
    const float sc = T::to_f32(scales[(row * K + k) / 64]), bi = T::to_f32(biases[(row * K + k) / 64]);
    const xwords xv = *reinterpret_cast<const xwords*>(x + k);
#pragma unroll
    for (int i = 0; i < kPerWord; ++i) {
      const float wv = __builtin_fmaf((float)((codes >> (BITS * i)) & ((1u << BITS) - 1)), sc, bi);
      const uint32_t pair = kSilu ? silu_exact_pair<T>(xv[i / 2]) : xv[i / 2];
      v = __builtin_fmaf(T::to_f32((uint16_t)(i & 1 ? pair >> 16 : pair)), T::to_f32(T::from_f32(wv)), v);
    }
  }
#pragma unroll
  for (int i = kWave / 2; i > 0; i /= 2) v += __shfl_xor(v, i);
  return v;
}
// v, or where it is NaN on a lane whose output is `mine` the above.  The wavefront walks such rows one after the other:
// with a lane to each, 3072 -> 18432 at 8 bits with an infinity in one row of eight took 778 us (24 without).
template <typename T, int BITS, bool kSilu>
__device__ inline float oct_keep_infinities(bool mine, float v, const uint16_t* x, const uint32_t* wq,
                                            const uint16_t* scales, const uint16_t* biases, int out_m, int64_t out_row,
                                            int K, int lane) {
  uint64_t left = __ballot(mine && v != v);
  while (left) {
    const int of = __builtin_ctzll(left);
    left &= left - 1;
    const int m = __builtin_amdgcn_readlane(out_m, of), row = __builtin_amdgcn_readlane((int)out_row, of);
    const float dot = oct_plain_dot<T, BITS, kSilu>(x + (size_t)m * K, wq, scales, biases, row, K, lane);
    if (lane == of) v = dot;
  }
  return v;
}

// Launches either kernel on contiguous runs of blocks of weight rows.  kM: activation rows of the instantiation.
template <int kWaves, int kM, typename Kernel>
int launch_oct_runs(Kernel kernel, PerDeviceInt& configured, int image_bytes, int per_block, int rows, int max_blocks,
                    int long_run, const void* x, int64_t M, const uint32_t* wq, const void* scales, const void* biases,
                    const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  const int wanted = image_bytes + (max_blocks + 1) * per_block;
  const int lds_max = wanted < 160 * 1024 ? wanted : 160 * 1024;
  if (!raise_lds_limit(configured, reinterpret_cast<const void*>(kernel), lds_max)) return MFQ_ELAUNCH;
  const int64_t blocks = N / rows;
  // workgroups resident at once: one per compute unit, several where a workgroup is only one or two wavefronts
  const int64_t places = (int64_t)compute_units() * (kWaves <= 2 ? 8 / kWaves : 1);
  const int64_t groups = (M + kM - 1) / kM;
  const int64_t fit = (lds_max - image_bytes) / per_block - 1;
  int64_t per_wg = (blocks * groups + places - 1) / places;
  if (kM > 4 || groups > 1) {
    // as many equal rounds of workgroups as the room for partial sums asks for
    const int64_t most = fit < max_blocks ? fit : max_blocks;
    const int64_t rounds = (per_wg + most - 1) / most;
    per_wg = (blocks * groups + places * rounds - 1) / (places * rounds);
  } else {
    // One workgroup per compute unit while that is at most max_blocks blocks each; longer weights in runs of
    // long_run blocks to as many workgroups as that takes (several resident per unit: a run's last loads and
    // its adding-up overlap the next run's first requests).
    if (per_wg > max_blocks) per_wg = long_run;
    if (per_wg > fit) per_wg = fit;
  }
  int64_t n_wg = (blocks + per_wg - 1) / per_wg;
  if (groups > 1) n_wg = (n_wg + 7) / 8 * 8 * groups;  // the groups of eight runs at a time
  const int lds = image_bytes + ((int)per_wg + 1) * per_block;
  hipLaunchKernelGGL(kernel, dim3((unsigned)n_wg), dim3(64 * kWaves), lds, stream, (const uint16_t*)x,
                     wq, (const uint16_t*)scales, (const uint16_t*)biases, (const uint16_t*)bias, y,
                     (int)(y_dtype == MFQ_F32), (int)M, (int)N, (int)per_wg);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

}  // namespace mfq
