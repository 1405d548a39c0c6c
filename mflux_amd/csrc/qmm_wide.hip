// W4/W8 x A16 quantized matmul for gfx950, some hundred activation rows against many columns or a long K (the encoders' and
// the text streams' MLPs):
//   y[M, N] = x[M, K] @ dequant(wq[N, K])^T (+ bias)
//
// A workgroup of four wavefronts computes a tile of 128 rows x 256 columns, two workgroups to a compute unit.  Each
// wavefront owns all of its rows and 64 of its columns, so a code is dequantised once per workgroup, by the wavefront that
// multiplies it, into the registers the matrix instruction reads: no weight goes through LDS.  That is what bounds the
// 128-column tiles of qmm_mid.hip, where a tile half as large writes and reads 96 KiB of LDS per step of 64 k (here 80 KiB,
// all of it x) and dequantises as many codes per 128 rows.
//   - x: 128 rows x 64 k in LDS, double buffered, rows of 128 bytes with the 16-byte column XORed with (row / 2) % 8; copied
//     through registers, each piece requested as soon as the one before it has been stored;
//   - weights: lane (r, h) takes the 32 codes k = 32 h .. of a step of its columns r and 32 + r, requested two steps ahead;
//     sub-step s multiplies its codes 8 s .., and the lane's x fragment is taken from the same k;
//   - eight codes of each column are dequantised (one float32 fma each, one rounding) while the eight before them are
//     multiplied; x fragments are read three ahead, over the barrier that ends a step.
// With 240 (4 bits) to 252 registers two wavefronts fit a SIMD.  384 rows x 3584 -> 37888 at 4 bits: 105 to 110 us, 0.95 to
// 0.99 PFLOP/s, 320 rows, whose last tile leaves half of its matrix work out, 104 (126 on 888 tiles of 128 x 128); before it did,
// 109, and with x all zeros, which costs less power, 95.  Weight loads
// in whole cache lines (their share of every line is 32 bytes now) would give some 8 % more, but their way through LDS has no
// registers left (half lines through a private region: 115); 96-row tiles took 135 us, 64-row tiles, which dequantise twice as
// often, 120.
#include <type_traits>

#include "common.h"
#include "tile_epilogue.h"

namespace mfq {
namespace {

constexpr int TM = 128, TN = 256, TK = 64;
constexpr int kThreads = 256;
constexpr int kI = TM / 32;              // blocks of 32 rows
constexpr int kBuf = TM * TK * 2;        // a step's x
constexpr int kStage = 4 * 64 * 144;     // what store_block_64x64 needs of four wavefronts
constexpr int kLds = 2 * kBuf > kStage ? 2 * kBuf : kStage;

// 16-byte column `chunk` of row `row`: 16 consecutive lanes (two rows) cover all banks
__device__ inline int swz(int row, int chunk) { return row * (TK * 2) + ((chunk ^ ((row >> 1) & 7)) << 4); }

// K % 256 == 0: the loop runs over quads of four steps, whose scales of a column are one piece of 512 / GS bytes.
// kShort: the last tile of every column has at most 64 rows, and its workgroups run a loop of their own over those.
template <typename T, int GS, int BITS, bool kShort>
__global__ __launch_bounds__(kThreads, 2) void qmm_wide_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint16_t* __restrict__ bias, void* __restrict__ y, int y_is_f32, int M,
    int N, int K, int tiles_m, int tiles_n, int base_quads, int n_long, const uint16_t* __restrict__ lr_t,
    const uint16_t* __restrict__ lr_bs, int lr_rank, Epilogue epi) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  using vec8 = typename T::vec8;
  constexpr int kRing = 4, kAhead = kRing - 1;                   // x fragments in flight
  constexpr int kWords = BITS;                                   // of a lane's 32 codes of a step and column
  constexpr int kSWords = 128 / GS;                              // 32-bit words of a column's scales of a quad
  static_assert(BITS == 4 || BITS == 8, "");
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const int r = lane & 31, h = lane >> 5;

  // Work item = (k range, tile); an XCD walks a contiguous run of the tiles (tile row fastest)
  const int n_tiles = tiles_m * tiles_n;
  const int split = __builtin_amdgcn_readfirstlane((int)blockIdx.x / n_tiles);
  int tile = blockIdx.x - split * n_tiles;
  {
    const int per_xcd = n_tiles / 8;
    if (tile < per_xcd * 8) tile = (tile & 7) * per_xcd + (tile >> 3);
  }
  const int m0 = (tile % tiles_m) * TM, n0 = (tile / tiles_m) * TN;
  // the first n_long k ranges are one quad longer than the others
  const int steps = 4 * (base_quads + (split < n_long ? 1 : 0));
  // first k of the item (by itself the compiler keeps it in a vector register, and the loads' addresses with it)
  const int kb = __builtin_amdgcn_readfirstlane((split * base_quads + min(split, n_long)) * 4 * TK);
  char* y_item = static_cast<char*>(y) + (size_t)split * M * N * 4;   // split > 0 only with float32 planes

  // byte offsets (32 bits, checked by the launcher)
  uint32_t xoff[kI];
#pragma unroll
  for (int i = 0; i < kI; ++i) xoff[i] = ((uint32_t)min(m0 + (t >> 3) + 32 * i, M - 1) * (uint32_t)K + 8u * (t & 7)) * 2u;
  uint32_t woff[2], soff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t row = (uint32_t)min(n0 + 64 * wave + 32 * j + r, N - 1);
    woff[j] = row * (uint32_t)(K * BITS / 8) + (uint32_t)(4 * BITS * h);
    soff[j] = row * (uint32_t)(K / GS) * 2u;
  }
  const char* xb = reinterpret_cast<const char*>(x);
  const char* wb = reinterpret_cast<const char*>(wq);
  const char* sb = reinterpret_cast<const char*>(scales);
  const char* bb = reinterpret_cast<const char*>(biases);
  const int wr_x = swz(t >> 3, t & 7);
  int rd[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) rd[s] = swz(r, 4 * h + s);

  u32x4 xr[kI];               // x of the step after the next
  uint32_t w[2][2][kWords];  // [step & 1][column]
  struct Scales { uint32_t s[2][kSWords], b[2][kSWords]; };
  Scales cur, nxt;
  // q: step of the item; steps past its end repeat the last one (the last quad) and are never multiplied
  auto load_x = [&](int q, int i) __attribute__((always_inline)) {
    const uint32_t k0 = kb + min(q, steps - 1) * TK;
    xr[i] = *reinterpret_cast<const u32x4*>(xb + (size_t)(k0 * 2u) + xoff[i]);
  };
  auto load_w = [&](int set, int q, int j) __attribute__((always_inline)) {
    const uint32_t k0 = kb + min(q, steps - 1) * TK;
    const char* p = wb + (size_t)(k0 / 8u * BITS) + woff[j];
#pragma unroll
    for (int l = 0; l < kWords / 4; ++l) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(p + 16 * l);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[set][j][4 * l + e] = v[e];
    }
  };
  auto load_s = [&](Scales& o, int q, int j) __attribute__((always_inline)) {  // the four steps from q on
    const uint32_t at = (uint32_t)(kb + min(q, steps - 4) * TK) / GS * 2u;
    uint32_t off = soff[j];
    asm volatile("" : "+v"(off));  // (or the 64-bit addresses of all columns' scales live through the loop, and are spilled)
#pragma unroll
    for (int l = 0; l < kSWords; ++l) {
      o.s[j][l] = reinterpret_cast<const uint32_t*>(sb + (size_t)at + off)[l];
      o.b[j][l] = reinterpret_cast<const uint32_t*>(bb + (size_t)at + off)[l];
    }
  };
  float sc[2][2], bi[2][2];  // [step & 1][column]
  auto scale_of = [&](const Scales& o, auto e_c, int j) __attribute__((always_inline)) {
    constexpr int e = decltype(e_c)::value;
    uint32_t s, b;
    if constexpr (GS == 32) {
      s = h ? o.s[j][e] >> 16 : o.s[j][e];
      b = h ? o.b[j][e] >> 16 : o.b[j][e];
    } else {
      constexpr int g = e * 64 / GS;
      s = o.s[j][g / 2] >> (16 * (g & 1));
      b = o.b[j][g / 2] >> (16 * (g & 1));
    }
    sc[e & 1][j] = T::to_f32((uint16_t)s);
    bi[e & 1][j] = T::to_f32((uint16_t)b);
  };

  f32x16 acc[kI][2];
#pragma unroll
  for (int i = 0; i < kI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  u32x4 wf[2][2];  // weight fragments [sub-step & 1][column]
  vec8 xf[kRing];
  uint32_t even, odd;
  f32x2 ev, ov;
  // codes 8 s + 2 p, + 1 of a lane's column (called for p = 0 .. 3 in order)
  auto pair = [&](const uint32_t (&c)[kWords], int s, int p, float sv, float bv) __attribute__((always_inline)) -> uint32_t {
    if constexpr (BITS == 4) {
      if (p == 0) {
        even = c[s] & 0x0f0f0f0fu;
        odd = (c[s] >> 4) & 0x0f0f0f0fu;
        ev = nibble_pair_f32<false>(even);
        ov = nibble_pair_f32<false>(odd);
      } else if (p == 2) {
        ev = nibble_pair_f32<true>(even);
        ov = nibble_pair_f32<true>(odd);
      }
      return T::pack2(__builtin_fmaf(ev[p & 1], sv, bv), __builtin_fmaf(ov[p & 1], sv, bv));
    } else {
      const uint32_t v = c[2 * s + (p >> 1)];
      return T::pack2(__builtin_fmaf(ubyte_f32(v, 2 * (p & 1)), sv, bv), __builtin_fmaf(ubyte_f32(v, 2 * (p & 1) + 1), sv, bv));
    }
  };
  auto read_x = [&](auto rows_c, int buf, int f) __attribute__((always_inline)) {
    constexpr int kR = decltype(rows_c)::value;
    return *reinterpret_cast<const vec8*>(lds + buf * kBuf + f % kR * 4096 + rd[f / kR]);
  };

  // step e of a quad, p of the item, on the tile's first kR blocks of 32 rows
  auto step = [&](auto rows_c, auto e_c, int p) __attribute__((always_inline)) {
    constexpr int kR = decltype(rows_c)::value, e = decltype(e_c)::value, buf = e & 1;
    constexpr int kFrags = 4 * kR;         // x fragments of a step
    constexpr int kGate = kFrags - kAhead;  // in front of this one's instructions the next step's x opens
    constexpr std::integral_constant<int, (e + 1) & 3> e_next{};
#pragma unroll
    for (int f = 0; f < kFrags; ++f) {
      const int s = f / kR, i = f % kR;
      if (f == kGate) __syncthreads();  // all of step p's x has been read, step p + 1's is there
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(__builtin_bit_cast(vec8, wf[s & 1][j]), xf[f % kRing], acc[i][j]);
      xf[(f + kAhead) % kRing] = f + kAhead < kFrags ? read_x(rows_c, buf, f + kAhead) : read_x(rows_c, buf ^ 1, f + kAhead - kFrags);
      if (f % 2 == 0 && f / 2 < kR) {
        *reinterpret_cast<u32x4*>(lds + (buf ^ 1) * kBuf + wr_x + 4096 * (f / 2)) = xr[f / 2];
        load_x(p + 2, f / 2);
      }
      if (f == 2 * kR) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (e == 3) scale_of(nxt, e_next, j);
          else scale_of(cur, e_next, j);
        }
        if constexpr (e == 3) cur = nxt;
      }
#pragma unroll
      for (int q = 8 * i / kR; q < 8 * (i + 1) / kR; ++q) {
        const int j = q >> 2;
        wf[(s + 1) & 1][j][q & 3] = s < 3 ? pair(w[buf][j], s + 1, q & 3, sc[buf][j], bi[buf][j])
                                          : pair(w[buf ^ 1][j], 0, q & 3, sc[buf ^ 1][j], bi[buf ^ 1][j]);
      }
      if (f == 3 * kR) {
#pragma unroll
        for (int j = 0; j < 2; ++j) load_w(buf, p + 2, j);
        if constexpr (e == 0) {
#pragma unroll
          for (int j = 0; j < 2; ++j) load_s(nxt, p + 4, j);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  auto run = [&](auto rows_c) __attribute__((always_inline)) {
    constexpr int kR = decltype(rows_c)::value;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      load_s(cur, 0, j);
      load_w(0, 0, j);
    }
#pragma unroll
    for (int i = 0; i < kR; ++i) load_x(0, i);
#pragma unroll
    for (int j = 0; j < 2; ++j) load_w(1, 1, j);
#pragma unroll
    for (int i = 0; i < kR; ++i) {
      *reinterpret_cast<u32x4*>(lds + wr_x + 4096 * i) = xr[i];
      load_x(1, i);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      scale_of(cur, std::integral_constant<int, 0>{}, j);
#pragma unroll
      for (int q = 0; q < 4; ++q) wf[0][j][q] = pair(w[0][j], 0, q, sc[0][j], bi[0][j]);
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < kAhead; ++f) xf[f] = read_x(rows_c, 0, f);
    for (int p = 0; p < steps; p += 4) {
      step(rows_c, std::integral_constant<int, 0>{}, p);
      step(rows_c, std::integral_constant<int, 1>{}, p + 1);
      step(rows_c, std::integral_constant<int, 2>{}, p + 2);
      step(rows_c, std::integral_constant<int, 3>{}, p + 3);
    }
  };
  // A tile of at most 64 rows leaves the matrix work of the other half out (its weights are dequantised all the same): 320
  // rows x 3584 -> 37888 113 -> 107 us, x 18944 -> 3584 67.6 -> 64.8, at 8 bits 124 -> 117 and level.  A kernel of its own,
  // because both loops in one cost the whole tiles' up to 1 % (registers).
  if (kShort && M - m0 <= TM / 2) run(std::integral_constant<int, kI / 2>{});
  else run(std::integral_constant<int, kI>{});

  // low-rank update: lr_rank more k, 16-bit and unquantised, straight from memory; of a tile's k ranges the first adds it
  if (split == 0) {
#pragma unroll 1
    for (int k = 0; k < lr_rank; k += 16) {
      vec8 wl[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        wl[j] = *reinterpret_cast<const vec8*>(lr_bs + (int64_t)min(n0 + 64 * wave + 32 * j + r, N - 1) * lr_rank + k + 8 * h);
#pragma unroll
      for (int i = 0; i < kI; ++i) {
        const vec8 xl = *reinterpret_cast<const vec8*>(lr_t + (int64_t)min(m0 + 32 * i + r, M - 1) * lr_rank + k + 8 * h);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(wl[j], xl, acc[i][j]);
      }
    }
  }

  __syncthreads();  // the last step's reads ahead are done: LDS is free
#pragma unroll
  for (int i = 0; i < kI; i += 2) {
    const f32x16 half[2][2] = {{acc[i][0], acc[i][1]}, {acc[i + 1][0], acc[i + 1][1]}};
    store_block_64x64<T>(half, lds, wave, lane, m0 + 32 * i, n0 + 64 * wave, M, N, bias, y_item, y_is_f32, epi);
  }
}

// whether the last row of tiles has at most half of its rows
inline bool short_tiles(int64_t M) { return (M - 1) % TM < TM / 2; }

struct WidePlan {
  int splits;  // 0: not this kernel
  int quads;   // of four steps per range
  int n_long;  // the first n_long ranges are one quad longer
  float us;    // what the call is estimated to take
};

// Measured at 4 bits in groups of 64 (600 drawn shapes of 100 to 1040 rows, a stream of launches on cold weights, fit to 7 %):
// a step of 64 k takes 1.6 us with two workgroups to a compute unit and 0.67 (one workgroup on the chip) to 0.93 (one to
// every unit) with one; 8 bits a seventh more.  A cut costs a launch, 2.9 us, and its float32 planes, written at 5 and read
// at 6 bytes/ps; with more ranges than one to a unit the planes (up to 64 MiB) cost what the second workgroup gives.
inline WidePlan plan_wide(int64_t M, int64_t N, int64_t K, int bits, bool may_cut) {
  const int64_t cus = compute_units();
  const int64_t tiles = ((M + TM - 1) / TM) * ((N + TN - 1) / TN);
  const int quads = (int)(K / (4 * TK));
  const float width = bits == 4 ? 1.f : 1.15f;
  const float plane_us = (float)M * (float)N * 4.f * 0.36e-6f;
  WidePlan best{0, 0, 0, 0.f};
  for (int s = 1; s == 1 || (may_cut && tiles * s <= cus && quads / s >= 2); ++s) {
    const int64_t items = tiles * s, rest = items % (2 * cus);
    const float last = rest == 0 ? 0.f : rest > cus ? 1.6f : 0.665f + 0.26f * (float)rest / (float)cus;
    float us = 4.8f + width * (float)(4 * ((quads + s - 1) / s)) * (1.6f * (float)(items / (2 * cus)) + last);
    if (s > 1) us += 2.9f + (float)s * plane_us;
    if (best.splits == 0 || us < 0.98f * best.us) best = WidePlan{s, quads / s, quads % s, us};
  }
  return best;
}

// Taken where its estimate is a tenth below that of the kernel that would run, up to 128 rows a fifth and from 769 rows on a
// sixth.  Of 2180 drawn calls of 17 to 1023 rows at 4 and 8 bits with such a K 105 are, in 0.905 of the time (geometric mean),
// 3 of them 3 to 6 % behind.  Up to 128 rows there is one row of tiles: every code is used once, and weights fetched a quarter
// line at a time are what the call takes; of 45 calls between a tenth and a fifth 17 were behind (67 rows x 2560 -> 19456 29.1 ->
// 33.1 us).  From 769 rows on 256-row tiles are well filled, 3 of 10 between a tenth and a sixth were behind (1019 x 12288 -> 3072
// 89 -> 98 us).  In between the band is worth having (627 x 18944 -> 3072 101 -> 87 us, 135 x 3840 -> 12288 46 -> 42).  Calls of
// 100 us and more, which the power limit slows, come out up to 15 % low on either side (320 x 3584 -> 37888: 94 for 110).  From
// 1024 rows on the 256 x 256 tiles are ahead (1024 x 3072 -> 12288 83 us against 89).  8 bits in groups of 32 stay with the other
// kernels: the scales of a quad are sixteen registers more than there are, and 879 rows x 10240 -> 4096 took 163 us against 101.
inline WidePlan choose_wide(int64_t M, int64_t N, int64_t K, int gs, int bits, bool may_cut) {
  const WidePlan none{0, 0, 0, 0.f};
  if (bits != 4 && (bits != 8 || gs == 32)) return none;
  if (M >= 1024 || K % (4 * TK) || M * K >= (int64_t)1 << 31 || N * K >= (int64_t)1 << 31) return none;
  const WidePlan plan = plan_wide(M, N, K, bits, may_cut);
  const float share = M <= 128 ? 0.8f : M <= 768 ? 0.9f : 0.84f;
  return plan.us < share * qmm_others_estimate_us(M, N, K, gs, bits) ? plan : none;
}

template <typename T, int GS, int BITS, bool kShort>
int launch_tiles(const WidePlan& plan, const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                  const void* biases, const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream, LowRank lr,
                  Epilogue epi) {
  const int tiles_m = (int)((M + TM - 1) / TM), tiles_n = (int)((N + TN - 1) / TN);
  hipLaunchKernelGGL((qmm_wide_kernel<T, GS, BITS, kShort>), dim3((unsigned)(tiles_m * tiles_n * plan.splits)), dim3(kThreads), kLds,
                     stream, (const uint16_t*)x, wq, (const uint16_t*)scales, (const uint16_t*)biases, (const uint16_t*)bias, y,
                     (int)(y_dtype == MFQ_F32), (int)M, (int)N, (int)K, tiles_m, tiles_n, plan.quads, plan.n_long,
                     (const uint16_t*)lr.t, (const uint16_t*)lr.bs, lr.R, epi);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

template <typename T, int GS, int BITS>
int launch_kernel(const WidePlan& plan, const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                  const void* biases, const void* bias, int64_t N, void* y, int y_dtype, hipStream_t stream, LowRank lr,
                  Epilogue epi) {
  const auto go = [&](auto launch) { return launch(plan, x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream, lr, epi); };
  return short_tiles(M) ? go(launch_tiles<T, GS, BITS, true>) : go(launch_tiles<T, GS, BITS, false>);
}

template <typename T>
int launch_type(const WidePlan& plan, const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype, hipStream_t stream,
                LowRank lr, Epilogue epi) {
  const auto go = [&](auto launch) { return launch(plan, x, M, K, wq, scales, biases, bias, N, y, y_dtype, stream, lr, epi); };
  if (gs == 32) return bits == 4 ? go(launch_kernel<T, 32, 4>) : MFQ_EUNSUPPORTED;  // (choose_wide() takes no 8 bits here)
  if (gs == 64) return bits == 4 ? go(launch_kernel<T, 64, 4>) : go(launch_kernel<T, 64, 8>);
  return bits == 4 ? go(launch_kernel<T, 128, 4>) : go(launch_kernel<T, 128, 8>);
}

}  // namespace

int qmm_wide_ranges(int64_t M, int64_t N, int64_t K, int gs, int bits) { return choose_wide(M, N, K, gs, bits, true).splits; }

int launch_qmm_wide(const void* x, int dtype, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                    const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype,
                    void* workspace, size_t workspace_bytes, hipStream_t stream, LowRank low_rank, Epilogue epi) {
  if (dtype != MFQ_BF16 && dtype != MFQ_F16) return MFQ_EUNSUPPORTED;
  // scales and biases are read as 32-bit words (two groups); an epilogue lives in the 16-bit staged store
  if (((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) ||
      (epi.kind != kEpiNone && (y_dtype == MFQ_F32 || N % 8)))
    return MFQ_EUNSUPPORTED;
  WidePlan plan = choose_wide(M, N, K, gs, bits, true);
  if (plan.splits > 1 && (!workspace || !aligned16(workspace) || workspace_bytes < (size_t)plan.splits * M * N * sizeof(float)))
    plan = choose_wide(M, N, K, gs, bits, false);
  if (plan.splits == 0) return MFQ_EUNSUPPORTED;
  const auto go = [&](auto launch) {
    if (plan.splits == 1)
      return launch(plan, x, M, K, wq, scales, biases, bias, N, gs, bits, y, y_dtype, stream, low_rank, epi);
    // K cut into ranges: float32 planes, and the second kernel applies bias and epilogue
    const int rc = launch(plan, x, M, K, wq, scales, biases, nullptr, N, gs, bits, workspace, MFQ_F32, stream, low_rank, Epilogue());
    return rc ? rc : launch_splitk_reduce(dtype, workspace, plan.splits, M, N, bias, y, y_dtype, stream, epi);
  };
  return dtype == MFQ_BF16 ? go(launch_type<BF16>) : go(launch_type<F16>);
}

}  // namespace mfq
