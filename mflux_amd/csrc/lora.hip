// Low-rank update of a finished product for gfx950: y[M, N] += t[M, R] @ bs[N, R]^T.
//
// This is the LoRA branch of a wrapped linear layer,
//   base(x) + scale * (x @ A) @ B
// (src/mflux/models/common/lora/layer/linear_lora_layer.py:50-53, and the sum
// over several adapters in fused_linear_lora_layer.py:13-20), with
// t = x @ [A_1 | A_2 | ...] and bs = [scale_1 * B_1^T | scale_2 * B_2^T | ...].
// The GEMM kernels accumulate the update with the product themselves; this
// kernel serves the products that come from elsewhere (one to sixteen
// activation rows, odd bit widths dequantised for a library GEMM).
//
// A workgroup of four wavefronts owns 64 rows x 128 columns of y; wavefront w
// takes columns [32w, 32w+32) as two 32x32x16 matrix-core accumulators.  R is
// small (a LoRA rank, or the sum of a few), so both operands are read straight
// from memory as matrix fragments: a lane's 8 consecutive k of one row of bs or
// t are one 16-byte load.  y is read, updated in float32 and rounded back.
#include <type_traits>

#include "common.h"

namespace mfq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 64;
constexpr int kCols = 128;

template <typename T>
__global__ __launch_bounds__(256) void low_rank_add_kernel(const uint16_t* __restrict__ t,
                                                           const uint16_t* __restrict__ bs, int R, int M, int N,
                                                           void* __restrict__ y, int y_is_f32, int vec_ok) {
  using vec8 = typename T::vec8;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 31;
  const int h = lane >> 5;
  const int n0 = blockIdx.x * kCols + 32 * wave;
  const int m0 = blockIdx.y * kRows;

  // rows past M / N are clamped for loads and never stored
  const uint16_t* brow = bs + (int64_t)min(n0 + r, N - 1) * R + 8 * h;
  const uint16_t* trow[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) trow[i] = t + (int64_t)min(m0 + 32 * i + r, M - 1) * R + 8 * h;

  f32x16 acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  for (int k = 0; k < R; k += 16) {
    const vec8 bf = *reinterpret_cast<const vec8*>(brow + k);
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[i] = mfma32(bf, *reinterpret_cast<const vec8*>(trow[i] + k), acc[i]);
  }

  // register e of accumulator i: row m0 + 32 i + r, column n0 + 8 (e / 4) + 4 h + e % 4
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = m0 + 32 * i + r;
    if (row >= M) continue;
#pragma unroll
    for (int eb = 0; eb < 4; ++eb) {
      const int col = n0 + 8 * eb + 4 * h;
      if (col >= N) continue;
      const int64_t o = (int64_t)row * N + col;
      if (y_is_f32) {
        float* dst = reinterpret_cast<float*>(y) + o;
        if (vec_ok) {
          float4 v = *reinterpret_cast<const float4*>(dst);
          v.x += acc[i][4 * eb];
          v.y += acc[i][4 * eb + 1];
          v.z += acc[i][4 * eb + 2];
          v.w += acc[i][4 * eb + 3];
          *reinterpret_cast<float4*>(dst) = v;
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (col + c < N) dst[c] += acc[i][4 * eb + c];
        }
      } else {
        uint16_t* dst = reinterpret_cast<uint16_t*>(y) + o;
        if (vec_ok) {
          uint2 v = *reinterpret_cast<const uint2*>(dst);
          v.x = T::pack2(lo_f32<T>(v.x) + acc[i][4 * eb], hi_f32<T>(v.x) + acc[i][4 * eb + 1]);
          v.y = T::pack2(lo_f32<T>(v.y) + acc[i][4 * eb + 2], hi_f32<T>(v.y) + acc[i][4 * eb + 3]);
          *reinterpret_cast<uint2*>(dst) = v;
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (col + c < N) dst[c] = T::from_f32(T::to_f32(dst[c]) + acc[i][4 * eb + c]);
        }
      }
    }
  }
}

template <typename T>
int launch(LowRank lr, int64_t M, int64_t N, void* y, int y_dtype, hipStream_t stream) {
  const dim3 grid((unsigned)((N + kCols - 1) / kCols), (unsigned)((M + kRows - 1) / kRows));
  // four consecutive outputs move as one piece when no piece can straddle a row or be misaligned
  const int vec_ok = (N & 3) == 0 && aligned16(y);
  hipLaunchKernelGGL((low_rank_add_kernel<T>), grid, dim3(256), 0, stream, (const uint16_t*)lr.t,
                     (const uint16_t*)lr.bs, lr.R, (int)M, (int)N, y, (int)(y_dtype == MFQ_F32), vec_ok);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

// ---- the down-projection in front of it: t[M, R] = x[M, K] @ A[K, R].
//
// x is read once (2 M K bytes: the kernel is bound by that read, and the whole of it is only a few times what
// must be in flight to cover the memory latency), so the work is cut for memory parallelism, not for the matrix
// cores: a workgroup of 8 wavefronts owns 16 rows of x, the trips (four pairs of 32-k steps: 512 bytes of each row,
// 8 KiB of x) are dealt to its wavefronts in turn, so that the workgroup reads one 4 KiB window of every row at a
// time, and a wavefront requests a whole trip before it uses any of it and the next one while it computes.
//   - the vector memory path takes about as long per cache line touched as per 128 bytes moved, so every load
//     covers whole lines: x goes row-segment-wise (8 lanes = one 128-byte line of a row) through a private LDS
//     region of the wavefront (no barrier), XOR-swizzled so that the fragment reads are conflict free;
//   - A is packed once per adapter set, so it is handed over in the order the matrix instruction consumes
//     (af [R/16][K/32][64 lanes][8]: lane 16 q + c of step s holds A[32 s + 8 q .. + 7][16 f + c]) and a
//     wavefront's fragment is 1 KiB of contiguous memory; it is small and stays in L2;
//   - the partial tiles meet in LDS and are added in the order of the wavefronts; A is the matrix
//     instruction's A operand so that a lane ends up with four consecutive columns of one row of t.
// F fragments of 16 columns of t per workgroup (blockIdx.y takes the next 16 F).
constexpr int kDownWaves = 8;
constexpr int kDownPairs = 4;                          // pairs of steps per trip
constexpr int kDownStage = kDownPairs * 16 * 128;      // bytes of x a wavefront stages per trip

// kTrain: t times `scale` ahead of the rounding, zeros from column `rank` on (an infinity of x makes NaN of the zeros there),
// and once more in tf, in the order of a matrix instruction whose k are the rows (see low_rank_up), with zeros for the rows
// past M of the last 32.
template <typename T, int F, bool kTrain, int kM>
__device__ __forceinline__ void low_rank_down(char* lds, const uint16_t* __restrict__ x, const uint16_t* __restrict__ af, int M,
                                              int K, int R, int m0, int f0, float scale, int rank,
                                              uint16_t* __restrict__ t, uint16_t* __restrict__ tf) {
  using vec8 = typename T::vec8;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c16 = lane & 15, q = lane >> 4;
  char* stage = lds + wave * kDownStage;

  const int steps = K / 32, pairs = (steps + 1) / 2;
  // trips are dealt round-robin: trip t of wavefront w is pairs (t * 8 + w) * 4 .. + 3, so that at any time the
  // workgroup reads one window of 4 KiB per row (16 pages in flight instead of 128)
  const int p_begin = wave * kDownPairs, p_end = pairs, p_stride = kDownWaves * kDownPairs;
  // staging: piece h (0, 1) of a pair is rows 8 h + lane / 8, 16-byte column lane % 8 of the pair's 128 bytes;
  // in LDS the column is XORed with row % 8.  A pair's second step may lie past K (K % 64 == 32): its columns
  // re-read the first step's and are not used.
  const int srow = lane >> 3, scol = lane & 7;
  constexpr int kPieces = kM / 8;
  const uint16_t* xsrc[kPieces];
  int sput[kPieces];
#pragma unroll
  for (int h = 0; h < kPieces; ++h) {
    xsrc[h] = x + (int64_t)min(m0 + 8 * h + srow, M - 1) * K;  // rows past M re-read the last one
    sput[h] = (8 * h + srow) * 128 + ((scol ^ srow) << 4);
  }
  int sget[2];  // step j of a pair: row c16, column 4 j + q
#pragma unroll
  for (int j = 0; j < 2; ++j) sget[j] = (c16 & (kM - 1)) * 128 + (((4 * j + q) ^ (c16 & 7)) << 4);
  const uint16_t* asrc = af + ((int64_t)f0 * steps * kWave + lane) * 8;

  f32x4 acc[F];
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the fragments of A are requested with the x they meet, as far as there are registers for them
  constexpr bool kAhead = F <= 2;
  auto load_a = [&](int f, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const vec8*>(asrc + ((int64_t)f * steps + s) * (kWave * 8));
  };
  auto request = [&](u32x4 (&xr)[kDownPairs][kPieces], vec8 (&ar)[kDownPairs][2][F], int p0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kDownPairs; ++u) {
      const int p = min(p0 + u, p_end - 1);  // pairs past the end repeat the last one and are not used
      const int col = min(64 * p + 8 * scol, K - 8);
#pragma unroll
      for (int h = 0; h < kPieces; ++h) {
        const u32x4* piece = reinterpret_cast<const u32x4*>(xsrc[h] + col);
        if constexpr (kTrain) xr[u][h] = *piece;  // (the same rows are read again, by columns and by the large product)
        else xr[u][h] = __builtin_nontemporal_load(piece);
      }
      if constexpr (kAhead) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int f = 0; f < F; ++f) ar[u][j][f] = load_a(f, min(2 * p + j, steps - 1));
      }
    }
  };
  u32x4 xr[kDownPairs][kPieces];
  vec8 a_now[kDownPairs][2][F], a_next[kDownPairs][2][F];
  if (p_begin < p_end) request(xr, a_now, p_begin);
  for (int p0 = p_begin; p0 < p_end; p0 += p_stride) {
#pragma unroll
    for (int u = 0; u < kDownPairs; ++u)
#pragma unroll
      for (int h = 0; h < kPieces; ++h) *reinterpret_cast<u32x4*>(stage + u * 2048 + sput[h]) = xr[u][h];
    // the next trip's x is on its way while this one meets its fragments of A
    if (p0 + p_stride < p_end) request(xr, a_next, p0 + p_stride);
    // (the region is private to the wavefront, whose LDS operations complete in order: no barrier)
#pragma unroll
    for (int u = 0; u < kDownPairs; ++u) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int s = 2 * (p0 + u) + j;
        if (p0 + u < p_end && s < steps) {
          const vec8 xf = *reinterpret_cast<const vec8*>(stage + u * 2048 + sget[j]);
#pragma unroll
          for (int f = 0; f < F; ++f) acc[f] = mfma16(kAhead ? a_now[u][j][f] : load_a(f, s), xf, acc[f]);
        }
      }
    }
    if constexpr (kAhead) {
#pragma unroll
      for (int u = 0; u < kDownPairs; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int f = 0; f < F; ++f) a_now[u][j][f] = a_next[u][j][f];
    }
  }
  __syncthreads();  // every wavefront is done with its staging region: the partial tiles go over it
  f32x4* parts = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int f = 0; f < F; ++f) parts[(wave * F + f) * kWave + lane] = acc[f];
  __syncthreads();
  if (wave < F) {  // wavefront f finishes fragment f: row m0 + c16, columns 16 (f0 + f) + 4 q .. + 3
    f32x4 v = parts[wave * kWave + lane];
#pragma unroll
    for (int w = 1; w < kDownWaves; ++w) {
      const f32x4 p = parts[(w * F + wave) * kWave + lane];
      v[0] += p[0]; v[1] += p[1]; v[2] += p[2]; v[3] += p[3];
    }
    const int row = m0 + c16;
    if (kM < 16 && c16 >= kM) return;  // (those lanes' rows are the others' again)
    if constexpr (kTrain) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = 16 * (f0 + wave) + 4 * q + e < rank ? v[e] * scale : 0.f;
      uint16_t* out = tf + (((int64_t)(f0 + wave) * ((M + 31) / 32) + row / 32) * 4 + (row & 31) / 8) * 128 + 32 * q + (row & 7);
#pragma unroll
      for (int e = 0; e < 4; ++e) out[8 * e] = row < M ? T::from_f32(v[e]) : (uint16_t)0;
    }
    if (row < M)
      *reinterpret_cast<uint2*>(t + (int64_t)row * R + 16 * (f0 + wave) + 4 * q) =
          make_uint2(T::pack2(v[0], v[1]), T::pack2(v[2], v[3]));
  }
}

template <typename T, int F>
__global__ __launch_bounds__(kDownWaves* kWave, 2) void low_rank_down_kernel(const uint16_t* __restrict__ x,
                                                                             const uint16_t* __restrict__ af, int M,
                                                                             int K, int R, uint16_t* __restrict__ t) {
  __shared__ __attribute__((aligned(16))) char lds[kDownWaves * kDownStage];
  low_rank_down<T, F, false, 16>(lds, x, af, M, K, R, blockIdx.x * 16, blockIdx.y * F, 1.f, R, t, nullptr);
}

// ---- training: the gradients of the two factors.
//
//   gt = scale (g @ lora_B^T) [M, R],   dB = scale (t^T @ g) [R, N],   dA = x^T @ gt [K, R]
//
// The first is the kernel above on g.  The others sum over the rows of what they read (g, x), while a lane of a matrix
// instruction holds eight consecutive k of one column, here eight rows:
//   - a workgroup owns 16 C columns (C = 4: 128 bytes of a row) and all rows, 32 at a time dealt to its eight wavefronts in
//     turn; lane (q, c) takes C columns of the rows 8 q .. + 7, so that 16 lanes read a whole line, and pairs of rows become
//     operands with one byte permutation per two values;
//   - the other factor (t, gt) comes in fragments of 1 KiB, which the kernel that computed it wrote in that order;
//   - the eight partial sums meet in LDS, added in the order of the wavefronts: no planes, no atomics, one rounding.
// gt and dB read the same g and do not need each other: one launch, the rows' workgroups first, the columns' behind them.
// 1536 rows, 3072 -> 12288, rank 16, with cold activations: the factors packed 3.1 us, t 4.2, gt and dB 18.7 (12.3 and 11.0 by
// themselves; bound by the bytes of g, read twice, and of the fragments), dA 6.6; lora_B transposed by torch and the BLAS
// library's four products 3.3, 10.4, 15.8, 11.9 and 10.1.
template <typename T, int F, int C>
__device__ __forceinline__ void low_rank_up(char* lds, const uint16_t* __restrict__ tf, const uint16_t* __restrict__ g, int M,
                                            int N, int n0, float scale, int rank, bool columns_first,
                                            uint16_t* __restrict__ out) {
  using vec8 = typename T::vec8;
  constexpr int W = C / 2;  // words of a lane and row
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c16 = lane & 15, q = lane >> 4;
  const int chunks = (M + 31) / 32;
  const uint16_t* src = g + min(n0 + C * c16, N - C);  // columns past N repeat the last ones and are not stored

  f32x4 acc[F][C];
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int i = 0; i < C; ++i) acc[f][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Chunk {
    uint32_t v[8][W];
    vec8 t[F];
  };
  auto request = [&](Chunk& c, int s) __attribute__((always_inline)) {
    auto& v = c.v;
#pragma unroll
    for (int f = 0; f < F; ++f) c.t[f] = *reinterpret_cast<const vec8*>(tf + (((int64_t)f * chunks + s) * kWave + lane) * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint16_t* p = src + (int64_t)min(32 * s + 8 * q + j, M - 1) * N;
      if constexpr (W == 2) {
        const uint2 d = *reinterpret_cast<const uint2*>(p);
        v[j][0] = d.x;
        v[j][1] = d.y;
      } else {
        v[j][0] = *reinterpret_cast<const uint32_t*>(p);
      }
    }
  };
  auto multiply = [&](Chunk& c, int s) __attribute__((always_inline)) {
    auto& v = c.v;
    if (32 * s + 32 > M) {  // what was read in the place of rows past M may not be finite
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (32 * s + 8 * q + j >= M) {
#pragma unroll
          for (int w = 0; w < W; ++w) v[j][w] = 0;
        }
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      u32x4 b;  // column C c16 + i, rows 8 q ..
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[j] = __builtin_amdgcn_perm(v[2 * j + 1][i / 2], v[2 * j][i / 2], i % 2 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int f = 0; f < F; ++f) acc[f][i] = mfma16(c.t[f], __builtin_bit_cast(vec8, b), acc[f][i]);
    }
  };
  // two chunks are on their way while two are multiplied; chunks past the end repeat the last one and are not multiplied
  Chunk a0, a1, b0, b1;
  const int step = 2 * kDownWaves;
  auto ask = [&](Chunk& u, Chunk& v, int s) __attribute__((always_inline)) {
    request(u, min(s, chunks - 1));
    request(v, min(s + kDownWaves, chunks - 1));
  };
  auto use = [&](Chunk& u, Chunk& v, int s) __attribute__((always_inline)) {
    if (s < chunks) multiply(u, s);
    if (s + kDownWaves < chunks) multiply(v, s + kDownWaves);
  };
  ask(a0, a1, wave);
  for (int s = wave; s < chunks; s += 2 * step) {
    ask(b0, b1, s + step);
    use(a0, a1, s);
    ask(a0, a1, s + 2 * step);
    use(b0, b1, s + step);
  }

  f32x4* parts = reinterpret_cast<f32x4*>(lds);
  const float* sums = reinterpret_cast<const float*>(lds);
#pragma unroll
  for (int f = 0; f < F; ++f) {  // lane (q, c16) of column set i: rows 16 f + 4 q .. + 3 of column C c16 + i
    __syncthreads();
#pragma unroll
    for (int i = 0; i < C; ++i) parts[(wave * C + i) * kWave + lane] = acc[f][i];
    __syncthreads();
    if (wave >= (columns_first ? C : 4)) continue;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (columns_first) {  // [N, rank]: wavefront i finishes column set i
#pragma unroll
      for (int w = 0; w < kDownWaves; ++w) {
        const f32x4 p = parts[(w * C + wave) * kWave + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p[e];
      }
      const int n = n0 + C * c16 + wave, r = 16 * f + 4 * q;
      if (n >= N || r >= rank) continue;
      uint16_t* dst = out + (int64_t)n * rank + r;
      if (rank % 4 == 0) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(T::pack2(v[0] * scale, v[1] * scale), T::pack2(v[2] * scale, v[3] * scale));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (r + e < rank) dst[e] = T::from_f32(v[e] * scale);
      }
    } else {  // [rank, N]: wavefront e finishes the rows 4 q + e
#pragma unroll
      for (int w = 0; w < kDownWaves; ++w)
#pragma unroll
        for (int i = 0; i < C; ++i) v[i] += sums[((w * C + i) * kWave + lane) * 4 + wave];
      const int n = n0 + C * c16, r = 16 * f + 4 * q + wave;
      if (n >= N || r >= rank) continue;
      uint32_t* dst = reinterpret_cast<uint32_t*>(out + (int64_t)r * N + n);
#pragma unroll
      for (int w = 0; w < W; ++w) dst[w] = T::pack2(v[2 * w] * scale, v[2 * w + 1] * scale);
    }
  }
}

// gt (and its fragments gtf) in the first `row_groups` workgroups, dB in the others
template <typename T, int F, int C, int kM>
__global__ __launch_bounds__(kDownWaves* kWave, 2) void low_rank_gradient_kernel(
    const uint16_t* __restrict__ g, const uint16_t* __restrict__ bf, const uint16_t* __restrict__ tf, int M, int N, int rank,
    int row_groups, float scale, uint16_t* __restrict__ gt, uint16_t* __restrict__ gtf, uint16_t* __restrict__ db) {
  __shared__ __attribute__((aligned(16))) char lds[kDownWaves * kDownStage];
  const int b = blockIdx.x;
  if (b < row_groups) low_rank_down<T, F, true, kM>(lds, g, bf, M, N, 16 * F, b * kM, 0, scale, rank, gt, gtf);
  else low_rank_up<T, F, C>(lds, tf, g, M, N, (b - row_groups) * 16 * C, scale, rank, false, db);
}

// t and its fragments
template <typename T, int F, int kM>
__global__ __launch_bounds__(kDownWaves* kWave, 2) void low_rank_forward_kernel(const uint16_t* __restrict__ x,
                                                                                const uint16_t* __restrict__ af, int M, int K,
                                                                                int rank, uint16_t* __restrict__ t,
                                                                                uint16_t* __restrict__ tf) {
  __shared__ __attribute__((aligned(16))) char lds[kDownWaves * kDownStage];
  low_rank_down<T, F, true, kM>(lds, x, af, M, K, 16 * F, blockIdx.x * kM, 0, 1.f, rank, t, tf);
}

// dA
template <typename T, int F, int C>
__global__ __launch_bounds__(kDownWaves* kWave, 2) void low_rank_up_kernel(const uint16_t* __restrict__ tf,
                                                                           const uint16_t* __restrict__ x, int M, int K, int rank,
                                                                           uint16_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) char lds[kDownWaves * kDownStage];
  low_rank_up<T, F, C>(lds, tf, x, M, K, blockIdx.x * 16 * C, 1.f, rank, true, out);
}

// The factors as the kernels take them, zeros from column `rank` to R, eight values to a thread:
//   af [R/16][K/32][4][16][8]   lora_A in fragment order (t)       ap [K, R]   lora_A, padded (the input gradient's update)
//   bf [R/16][N/32][4][16][8]   lora_B^T in fragment order (gt)    bs [N, R]   scale lora_B^T (the forward product's update)
// One launch, once per step; with torch's operations (two transposed copies, the scaling, the padding) it was up to six.
template <typename T>
__global__ __launch_bounds__(256) void low_rank_pack_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, int K,
                                                            int N, int rank, int R, float scale, uint16_t* __restrict__ af,
                                                            uint16_t* __restrict__ bf, uint16_t* __restrict__ bs,
                                                            uint16_t* __restrict__ ap) {
  const int pieces_a = K * (R / 8), pieces_b = N * (R / 8);
  int p = blockIdx.x * 256 + threadIdx.x;
  uint16_t* out;
  const uint16_t* src;
  int64_t at[8];   // element of src; < 0: zero
  float factor = 1.f;
  if (p < pieces_a || (p >= pieces_a && p < pieces_a + pieces_b)) {  // fragments
    const bool is_a = p < pieces_a;
    if (!is_a) p -= pieces_a;
    const int len = is_a ? K : N, c = p & 15, k = (p >> 4) % (len / 8) * 8, f = (p >> 4) / (len / 8), r = 16 * f + c;
    src = is_a ? a : b;
    out = (is_a ? af : bf) + (int64_t)p * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) at[e] = r >= rank ? -1 : is_a ? (int64_t)(k + e) * rank + r : (int64_t)r * N + k + e;
  } else {
    p -= pieces_a + pieces_b;
    if (p < pieces_b) {  // bs: neighbouring threads take neighbouring columns of lora_B
      const int n = p % N, r = p / N * 8;
      src = b;
      out = bs + (int64_t)n * R + r;
      factor = scale;
#pragma unroll
      for (int e = 0; e < 8; ++e) at[e] = r + e >= rank ? -1 : (int64_t)(r + e) * N + n;
    } else {
      p -= pieces_b;
      if (p >= pieces_a || !ap) return;
      const int k = p / (R / 8), r = p % (R / 8) * 8;
      src = a;
      out = ap + (int64_t)p * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) at[e] = r + e >= rank ? -1 : (int64_t)k * rank + r + e;
    }
  }
  uint16_t v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = at[e] < 0 ? (uint16_t)0 : src[at[e]];
  if (factor != 1.f) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (at[e] >= 0) v[e] = T::from_f32(T::to_f32(v[e]) * factor);  // (zero times an infinite scale is no zero)
  }
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (uint32_t)v[2 * e] | (uint32_t)v[2 * e + 1] << 16;
  *reinterpret_cast<u32x4*>(out) = o;
}

// Rows to a workgroup of low_rank_down: eight (half of a matrix instruction's) as long as that fills the chip once.  What a
// workgroup reads of x and of the fragments comes at some 55 bytes/ns: 1536 rows of 12288 15.6 us with 16, 12.3 with 8; 2304 of
// 3840, rank 32, 7.0 and 10.6.
inline int down_rows(int64_t M) { return M <= 8 * (int64_t)compute_units() ? 8 : 16; }
// Columns to a workgroup of low_rank_up: 32 (lines in halves) as long as they, and the workgroups in front of them, fill the chip
// once, else 64: 1536 rows of 3072 6.6 us with 32, 7.5 with 64; of 12288 17.0 and 10.7.
inline int up_columns(int64_t n, int64_t in_front) { return in_front + (n + 31) / 32 <= compute_units() ? 32 : 64; }

template <typename T>
int launch_down(const void* x, int64_t M, int64_t K, const void* at, int64_t R, void* t, hipStream_t stream) {  // at: fragment order
  const int frags = R % 64 == 0 ? 4 : (R % 32 == 0 ? 2 : 1);
  const dim3 grid((unsigned)((M + 15) / 16), (unsigned)(R / (16 * frags)));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kDownWaves * kWave), 0, stream, (const uint16_t*)x, (const uint16_t*)at,
                       (int)M, (int)K, (int)R, (uint16_t*)t);
  };
  if (frags == 4) go(low_rank_down_kernel<T, 4>);
  else if (frags == 2) go(low_rank_down_kernel<T, 2>);
  else go(low_rank_down_kernel<T, 1>);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

template <typename T, int F>
int launch_gradient(const void* g, int64_t M, int64_t N, const void* bf, const void* tf, int rank, float scale, void* gt, void* gtf,
                    void* db, hipStream_t stream) {
  const int rows = down_rows(M), row_groups = gt ? (int)((M + 31) / 32 * (32 / rows)) : 0;
  auto go = [&](auto kernel, int columns) {
    const int64_t groups = row_groups + (db ? (N + columns - 1) / columns : 0);
    hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3(kDownWaves * kWave), 0, stream, (const uint16_t*)g, (const uint16_t*)bf,
                       (const uint16_t*)tf, (int)M, (int)N, rank, row_groups, scale, (uint16_t*)gt, (uint16_t*)gtf, (uint16_t*)db);
  };
  if (up_columns(N, row_groups) == 64) rows == 8 ? go(low_rank_gradient_kernel<T, F, 4, 8>, 64) : go(low_rank_gradient_kernel<T, F, 4, 16>, 64);
  else rows == 8 ? go(low_rank_gradient_kernel<T, F, 2, 8>, 32) : go(low_rank_gradient_kernel<T, F, 2, 16>, 32);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

template <typename T, int F>
int launch_up(const void* x, int64_t M, int64_t K, const void* tf, int rank, void* out, hipStream_t stream) {
  auto go = [&](auto kernel, int columns) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((K + columns - 1) / columns)), dim3(kDownWaves * kWave), 0, stream,
                       (const uint16_t*)tf, (const uint16_t*)x, (int)M, (int)K, rank, (uint16_t*)out);
  };
  if (up_columns(K, 0) == 64) go(low_rank_up_kernel<T, F, 4>, 64);
  else go(low_rank_up_kernel<T, F, 2>, 32);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

template <typename T, int F>
int launch_forward(const void* x, int64_t M, int64_t K, const void* af, int rank, void* t, void* tf, hipStream_t stream) {
  auto go = [&](auto kernel, int rows) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((M + 31) / 32 * (32 / rows))), dim3(kDownWaves * kWave), 0, stream,
                       (const uint16_t*)x, (const uint16_t*)af, (int)M, (int)K, rank, (uint16_t*)t, (uint16_t*)tf);
  };
  if (down_rows(M) == 8) go(low_rank_forward_kernel<T, F, 8>, 8);
  else go(low_rank_forward_kernel<T, F, 16>, 16);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

// calls f(type, fragments of 16 columns)
template <typename Fn>
int with_type_and_fragments(int dtype, int R, Fn f) {
  const auto frags = [&](auto type) {
    return R == 16 ? f(type, std::integral_constant<int, 1>{}) : f(type, std::integral_constant<int, 2>{});
  };
  return dtype == MFQ_BF16 ? frags(BF16{}) : frags(F16{});
}

}  // namespace

int launch_low_rank_pack(const void* a, const void* b, int dtype, int64_t K, int64_t N, int rank, int R, float scale, void* af,
                         void* bf, void* bs, void* ap, hipStream_t stream) {
  const int64_t pieces = (K + N) * (R / 8) * 2 - (ap ? 0 : K * (R / 8));
  return with_type_and_fragments(dtype, R, [&](auto type, auto) {
    hipLaunchKernelGGL((low_rank_pack_kernel<decltype(type)>), dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream,
                       (const uint16_t*)a, (const uint16_t*)b, (int)K, (int)N, rank, R, scale, (uint16_t*)af, (uint16_t*)bf,
                       (uint16_t*)bs, (uint16_t*)ap);
    return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
  });
}

int launch_low_rank_forward(const void* x, int dtype, int64_t M, int64_t K, const void* af, int rank, int R, void* t, void* tf,
                            hipStream_t stream) {
  return with_type_and_fragments(dtype, R, [&](auto type, auto frags) {
    return launch_forward<decltype(type), decltype(frags)::value>(x, M, K, af, rank, t, tf, stream);
  });
}

int launch_low_rank_gradient(const void* g, int dtype, int64_t M, int64_t N, const void* bf, const void* tf, int rank, int R,
                             float scale, void* gt, void* gtf, void* db, hipStream_t stream) {
  return with_type_and_fragments(dtype, R, [&](auto type, auto frags) {
    return launch_gradient<decltype(type), decltype(frags)::value>(g, M, N, bf, tf, rank, scale, gt, gtf, db, stream);
  });
}

int launch_low_rank_up(const void* x, int dtype, int64_t M, int64_t K, const void* tf, int rank, int R, void* out,
                       hipStream_t stream) {
  return with_type_and_fragments(dtype, R, [&](auto type, auto frags) {
    return launch_up<decltype(type), decltype(frags)::value>(x, M, K, tf, rank, out, stream);
  });
}

int launch_low_rank_down(const void* x, int dtype, int64_t M, int64_t K, const void* at, int64_t R, void* t,
                         hipStream_t stream) {
  if (dtype == MFQ_BF16) return launch_down<BF16>(x, M, K, at, R, t, stream);
  if (dtype == MFQ_F16) return launch_down<F16>(x, M, K, at, R, t, stream);
  return MFQ_EDTYPE;
}

int launch_low_rank_add(int dtype, LowRank low_rank, int64_t M, int64_t N, void* y, int y_dtype,
                        hipStream_t stream) {
  if (low_rank.R == 0) return MFQ_OK;
  if ((M + kRows - 1) / kRows > 65535) return MFQ_EUNSUPPORTED;
  if (dtype == MFQ_BF16) return launch<BF16>(low_rank, M, N, y, y_dtype, stream);
  if (dtype == MFQ_F16) return launch<F16>(low_rank, M, N, y, y_dtype, stream);
  return MFQ_EDTYPE;
}

}  // namespace mfq
