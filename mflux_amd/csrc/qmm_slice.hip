// Quantized matmul for shapes with too few output tiles to fill the chip (17 to some hundred activation rows against the
// hidden size: the text stream of mflux's joint transformer blocks, e.g.
// src/mflux/models/flux/model/flux_transformer/joint_transformer_block.py, short prompts in the text encoders):
//   y[M, N] = x[M, K] @ dequant(wq[N, K])^T (+ bias), in one launch.
//
// The 128-column-tile kernel (qmm_mid.hip) fills the chip on such shapes by cutting K into ranges, each with a float32
// plane of the output that a second launch reads back.  Here a tile is small enough that there is one for every compute
// unit with K whole -- 64 rows x 32, 48, 64, 80 or 96 columns, 32 x 32 -- and K is cut over the four wavefronts of its workgroup,
// whose partial tiles meet in LDS at the end: no planes, no second launch.
//   - Each wavefront has a ring of its own in LDS (40 KiB) that it fills with global_load_lds and reads back as matrix
//     fragments: no barrier in the loop, no registers for what is on its way, and as no load in the loop is the compiler's
//     every wait is by count and leaves the younger requests of x in flight (and of codes, where that pays: see step).
//   - A request costs the memory path of a compute unit some 1.2 to 2.5 ns per cache line touched, whatever it takes of
//     the line, so everything comes in whole lines or long runs of one: x in 128 bytes of a row (64 k), codes in chunks
//     of 128 bytes of a row where the ring has room, scales and biases eight groups at a time.
//   - One wavefront to a SIMD issues in order: dequantisation (one float32 fma per code, single rounding to the 16-bit
//     type, every code once per workgroup), requests and LDS reads are dealt out between the matrix instructions by
//     hand, and the steady state has no branch but one for a chunk's and one for a window's end (with a branch around
//     every request 16.0 us on the shape below instead of 13.8).
// Measured, 4 bits in groups of 64, stream of launches, a gigabyte of weights in turn: 256 rows x 3072 -> 3072 22.6 us on the
// other kernel (two launches), 15.3 here; 512 rows 26.4 -> 22.7; 64 rows 16.2 -> 10.6.  (The figures of attempts, above and
// below, are of fewer weights in turn, where this kernel took 13.5 to 13.8.)  What bounds it: a sub-step of 64 k on the four
// wavefronts takes 0.67 us (64 x 48), of which the matrix instructions with the dequantisation between them are 0.34 and
// 39 KB of direct loads 0.35 to 0.4, which a lone wavefront overlaps in part; 5 us are launch, first bytes and the sum.
// Tried on this tile and not faster: eight wavefronts with a barrier per step and shared staging (13.9 us; slower from
// larger tiles on), x requested into L2 ahead of its use (14.8), half-length steps in a deeper ring (15.5).
#include <type_traits>

#include "common.h"
#include "epilogue.h"

namespace mfq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;  // one to a SIMD
constexpr int kThreads = kWaves * kWave;
constexpr int kLdsMax = 160 * 1024;

template <int BITS, int kA, int kB>
struct Shape {
  static constexpr int TM = 16 * kA, TN = 16 * kB;
  static constexpr int kXSlot = TM * 128;                      // 64 k of the tile's rows of x
  static constexpr int kXLoads = TM / 8;                       // load instructions of a slot
  static constexpr int kXGroup = 4;                            // that share a write of m0
  static constexpr int kInstr = 2 * kA * kB;                   // matrix instructions of a sub-step
  static constexpr int kReadsAt = kInstr / 3;                  // the next sub-step's fragments are read behind these
  // load l of a slot is requested behind matrix instruction load_slot(l), kXGroup of them together; those requested when the
  // reads begin
  static constexpr int load_slot(int l) { return l / kXGroup * kXGroup * kInstr / kXLoads; }
  static constexpr int loads_before_reads() {
    int n = 0;
    for (int l = 0; l < kXLoads; ++l) n += load_slot(l) <= kReadsAt;
    return n;
  }
  static constexpr int kWinBytes = TN * 16;                    // a window: scales (or biases) of eight groups
  static constexpr int kSLoads = (TN * 4 + 63) / 64;
  static constexpr int kGran = (BITS == 3 || BITS == 5) ? 2 : 1;  // sub-steps of a wavefront come in multiples of this
  static constexpr int ring(int x_slots, int chunk) { return x_slots * kXSlot + 2 * TN * chunk * 8 * BITS + 4 * kWinBytes; }
  static constexpr bool fits(int x_slots, int chunk) { return ring(x_slots, chunk) <= kLdsMax / kWaves; }
  // sub-steps of 64 k of a chunk of codes (whole cache lines of a row where there is room), slots of x
  static constexpr int kLine = BITS == 8 ? 2 : 4;
  static constexpr int kXSlots = fits(3, kGran) ? 3 : 2;
  static constexpr int kChunk = fits(kXSlots, kLine) ? kLine : (kLine == 4 && fits(kXSlots, 2)) ? 2 : kGran;
  static constexpr int kRowPieces = kChunk * BITS / 2;         // 16-byte pieces of a row's codes in a chunk
  static constexpr int kWPieces = TN * kRowPieces;
  static constexpr int kWSlot = kWPieces * 16;
  static constexpr int kWLoads = (kWPieces + 63) / 64;
  static constexpr int kWBase = kXSlots * kXSlot, kSBase = kWBase + 2 * kWSlot;
  static constexpr int kRing = kSBase + 4 * kWinBytes;         // LDS of a wavefront
  static constexpr int kStride = TN * 4 + 16;                  // a row of the partial tile in LDS
  // row blocks of the partial tiles that meet in LDS at a time
  static constexpr int kFit = kLdsMax / (kWaves * 16 * kStride), kBands = (kA + kFit - 1) / kFit, kBand = (kA + kBands - 1) / kBands;
  static constexpr int kPart = kBand * 16 * kStride;
  static constexpr int kLds = kWaves * (kRing > kPart ? kRing : kPart);
  static_assert(kLds <= kLdsMax && (kChunk * BITS) % 2 == 0, "");
};

// the 16-byte column of a 128-byte row XORed with this: see qmm_frag.hip (fragments of columns 2 (lane / 16) + pass)
__device__ inline int swz_mask(int row) {
  const int i = (row >> 1) & 7;
  return (i & 4) | ((i & 1) << 1) | ((i >> 2) ^ ((i >> 1) & 1));
}

// Position of 16-byte piece `piece` of row `row` of a chunk in the row's LDS image (an involution), so that the rows of a
// fragment spread over the banks.  The 3-, 5- and 6-bit packs lie as they are.
template <int BITS, int kPieces>
__device__ inline int w_piece(int row, int piece) {
  if constexpr (BITS != 4 && BITS != 8) return piece;
  else if constexpr (BITS == 8 && kPieces == 4) return piece ^ ((0x1320 >> (((row >> 2) & 3) * 4)) & 3);
  else return piece ^ ((row * kPieces / 16) & (kPieces - 1));
}

template <typename T, int BITS, int kA, int kB>
__global__ __launch_bounds__(kThreads, 1) void qmm_slice_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint16_t* __restrict__ bias, void* __restrict__ y, int y_is_f32, int M,
    int N, int K, int gs_shift, int tiles_m, int tiles_n, int splits, const uint16_t* __restrict__ lr_t,
    const uint16_t* __restrict__ lr_bs, int lr_rank, Epilogue epi) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  using vec8 = typename T::vec8;
  using S = Shape<BITS, kA, kB>;
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int r = lane & 15, q = lane >> 4;

  // Work item = (k range, tile).  Workgroups are dealt round-robin to the 8 XCDs; an XCD walks a contiguous run of the tile
  // sequence (tile row fastest), sharing x and codes in its L2.
  const int n_tiles = tiles_m * tiles_n;
  const int split = __builtin_amdgcn_readfirstlane((int)blockIdx.x / n_tiles);
  int tile = blockIdx.x - split * n_tiles;
  {
    const int per_xcd = n_tiles / 8;
    if (tile < per_xcd * 8) tile = (tile & 7) * per_xcd + (tile >> 3);
  }
  const int m0 = (tile % tiles_m) * S::TM;
  const int n0 = (tile / tiles_m) * S::TN;
  // The weight row (output column of the linear) of the tile's column c.  SwiGLU: half of a tile's columns are consecutive
  // columns of the gate projection, the other half those of the up projection, which lie in alternating blocks of 32.
  const bool swiglu = epi.kind == kEpiSwiglu;
  auto weight_row = [&](int c) __attribute__((always_inline)) {
    if (!swiglu) return min(n0 + c, N - 1);
    const int up = c >= S::TN / 2, g = min(n0 / 2 + c - up * (S::TN / 2), N / 2 - 1);
    return (g >> 5) * 64 + up * 32 + (g & 31);
  };

  // the wavefront's sub-steps of 64 k: [begin, begin + n)
  const int parts = kWaves * splits, part = kWaves * split + wave, grains = K / (64 * S::kGran);
  const int begin = part * grains / parts * S::kGran;
  const int n = (part + 1) * grains / parts * S::kGran - begin;

  char* ring = lds + wave * S::kRing;
  const uint32_t ring_addr = (uint32_t)(uintptr_t)ring;
  // LDS destination of a lane: lds_addr + offset (a constant) + 16 (4) times its number.  A load into LDS wants one wait
  // state behind the write of m0, which the compiler does not see to inside a statement of assembly: the s_nop.
  auto dma16 = [&](const char* sbase, uint32_t voff, uint32_t lds_addr, int offset) __attribute__((always_inline)) {
    asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 ::"v"(voff), "s"(sbase), "s"(lds_addr), "i"(offset) : "memory", "m0", "scc");
  };
  // Four of them to consecutive KiB of LDS: the instruction's offset counts on both sides, in LDS and in memory.
  auto dma16x4 = [&](const char* sbase, const uint32_t* voff, uint32_t lds_addr, int offset) __attribute__((always_inline)) {
    asm volatile("s_add_i32 m0, %5, %6\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %4\n\tglobal_load_lds_dwordx4 %1, %4 offset:1024"
                 "\n\tglobal_load_lds_dwordx4 %2, %4 offset:2048\n\tglobal_load_lds_dwordx4 %3, %4 offset:3072"
                 ::"v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(sbase), "s"(lds_addr), "i"(offset) : "memory", "m0", "scc");
  };
  auto dma4 = [&](const char* sbase, uint32_t voff, uint32_t lds_addr, int offset) __attribute__((always_inline)) {
    asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 ::"v"(voff), "s"(sbase), "s"(lds_addr), "i"(offset) : "memory", "m0", "scc");
  };

  // ---- what the lane loads
  uint32_t xoff[S::kXLoads];  // eight rows, 128 bytes each; what the instruction's offset adds is taken off here
#pragma unroll
  for (int i = 0; i < S::kXLoads; ++i) {
    const int row = 8 * i + (lane >> 3);
    xoff[i] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)K + 8u * (uint32_t)((lane & 7) ^ swz_mask(row))) * 2u +
              1024u * (uint32_t)(S::kXGroup - 1 - i % S::kXGroup);
  }
  // codes: piece p of a chunk is piece p % kRowPieces of row p / kRowPieces
  uint32_t wrow[S::kWLoads], wcol[S::kWLoads];
#pragma unroll
  for (int i = 0; i < S::kWLoads; ++i) {
    const int p = min(64 * i + lane, S::kWPieces - 1), row = p / S::kRowPieces;
    wrow[i] = (uint32_t)weight_row(row) * (uint32_t)(K * BITS / 8);
    wcol[i] = 16u * (uint32_t)w_piece<BITS, S::kRowPieces>(row, p % S::kRowPieces);
  }
  // scales and biases: dword d of a window is groups 2 (d % 4), + 1 of row d / 4
  const int row_groups = K >> gs_shift;
  uint32_t srow[S::kSLoads];
#pragma unroll
  for (int i = 0; i < S::kSLoads; ++i)
    srow[i] = (uint32_t)weight_row(min(16 * i + (lane >> 2), S::TN - 1)) * (uint32_t)row_groups * 2u;
  const int first_dword = (begin * 64 >> gs_shift) >> 1;  // of the first window; a window begins at an even group
  const int g_first = (begin * 64 >> gs_shift) & ~1, g_last = ((begin + n) * 64 - 1) >> gs_shift;

  const char* xbytes = reinterpret_cast<const char*>(x) + (ptrdiff_t)begin * 128 - 1024 * (S::kXGroup - 1);
  const char* wbytes = reinterpret_cast<const char*>(wq);
  const uint32_t w_begin = (uint32_t)begin * 8u * BITS, w_end = (uint32_t)(K * BITS / 8 - 16);
  auto load_x = [&](int j, int slot, int i) __attribute__((always_inline)) {  // loads i to i + kXGroup - 1
    dma16x4(xbytes + (size_t)j * 128, xoff + i, ring_addr + slot * S::kXSlot, 1024 * i);
  };
  auto load_w = [&](int c) __attribute__((always_inline)) {  // chunk c; pieces past the row's end repeat its last one
#pragma unroll
    for (int i = 0; i < S::kWLoads; ++i)
      if ((i + 1) * 64 <= S::kWPieces || 64 * i + lane < S::kWPieces)
        dma16(wbytes, wrow[i] + min(wcol[i] + w_begin + (uint32_t)(c * S::kRowPieces * 16), w_end),
              ring_addr + (c & 1) * S::kWSlot, S::kWBase + 1024 * i);
  };
  auto load_s = [&](int win) __attribute__((always_inline)) {
    const uint32_t col = 4u * (uint32_t)min(first_dword + 4 * win + (lane & 3), row_groups / 2 - 1);
    const uint32_t addr = ring_addr + (win & 1) * 2 * S::kWinBytes;
#pragma unroll
    for (int i = 0; i < S::kSLoads; ++i)
      if ((i + 1) * 64 <= S::TN * 4 || 64 * i + lane < S::TN * 4) {
        dma4(reinterpret_cast<const char*>(scales), srow[i] + col, addr, S::kSBase + 256 * i);
        dma4(reinterpret_cast<const char*>(biases), srow[i] + col, addr, S::kSBase + S::kWinBytes + 256 * i);
      }
  };

  constexpr int kRaw = BITS == 8 ? 4 : (BITS == 4 || BITS == 3) ? 2 : 3;  // words that hold a lane's 16 codes of a sub-step
  struct Frag {
    vec8 x[kA][2];
    uint32_t w[kB][kRaw + 1];
    uint16_t sraw[kB], braw[kB];
    float s[kB], b[kB];
  };
  const int rd_x[2] = {r * 128 + (((2 * q) ^ swz_mask(r)) << 4), r * 128 + (((2 * q + 1) ^ swz_mask(r)) << 4)};
  auto read_x = [&](Frag& f, int slot, int i) __attribute__((always_inline)) {
    f.x[i % kA][i / kA] = *reinterpret_cast<const vec8*>(ring + slot * S::kXSlot + i % kA * 2048 + rd_x[i / kA]);
  };
  // What of the addresses of codes and scales is the lane's own.  The rows 16 b + r of the column blocks share the swizzle
  // and lie at fixed distances; the pieces of sub-step jj of a chunk and the lane's part of them use different bits.
  constexpr int kRowBytes = S::kRowPieces * 16;
  const int q_byte = 2 * BITS * q;
  const int lane_w = BITS == 4 || BITS == 8 ? r * kRowBytes + (q_byte & 15) : r * kRowBytes + (q_byte & ~3);
  const int lane_piece = BITS == 4 || BITS == 8 ? (w_piece<BITS, S::kRowPieces>(r, 0) ^ (q_byte >> 4)) << 4 : 0;
  const int lane_s = r * 16 + (gs_shift == 5 ? (q >> 1) * 2 : 0);
  auto read_codes = [&](Frag& f, int j, int b) __attribute__((always_inline)) {  // of column block b
    const int jj = j % S::kChunk, g = ((begin + j) * 64 >> gs_shift) - g_first;
    const char* p = ring + S::kWBase + (j / S::kChunk & 1) * S::kWSlot + b * 16 * kRowBytes + lane_w;
    if constexpr (BITS == 4 || BITS == 8) {
      p += (jj * 8 * BITS) ^ lane_piece;
      if constexpr (kRaw == 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        f.w[b][0] = v.x;
        f.w[b][1] = v.y;
      } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e) f.w[b][e] = v[e];
      }
    } else {
      const uint32_t* pw = reinterpret_cast<const uint32_t*>(p + jj * 8 * BITS);
#pragma unroll
      for (int e = 0; e < kRaw; ++e) f.w[b][e] = pw[e];
    }
    const char* ss = ring + S::kSBase + ((g >> 3) & 1) * 2 * S::kWinBytes + (g & 7) * 2 + lane_s + b * 256;
    f.sraw[b] = *reinterpret_cast<const uint16_t*>(ss);
    f.braw[b] = *reinterpret_cast<const uint16_t*>(ss + S::kWinBytes);
  };
  auto align_codes = [&](Frag& f) __attribute__((always_inline)) {
    if constexpr (BITS == 3 || BITS == 5) {
      const uint32_t sh = (q & 1) * 16;  // 2 BITS q bytes: odd q start in the middle of a word
#pragma unroll
      for (int b = 0; b < kB; ++b)
#pragma unroll
        for (int e = 0; e < kRaw; ++e) f.w[b][e] = __builtin_amdgcn_alignbit(e + 1 < kRaw ? f.w[b][e + 1] : 0u, f.w[b][e], sh);
    }
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      f.w[b][kRaw] = 0;
      f.s[b] = T::to_f32(f.sraw[b]);
      f.b[b] = T::to_f32(f.braw[b]);
    }
  };

  f32x4 acc[kA][kB];  // row 16 a + r, columns 16 b + 4 q + e
#pragma unroll
  for (int a = 0; a < kA; ++a)
#pragma unroll
    for (int b = 0; b < kB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // codes 2 p, 2 p + 1 of fragment i (column block i % kB, pass i / kB), dequantised (called for p = 0 .. 3 in order)
  uint32_t even, odd;
  f32x2 ev, ov;
  auto pair = [&](const Frag& f, int i, int p) __attribute__((always_inline)) {
    const int b = i % kB, h = i / kB;
    if constexpr (BITS == 4) {
      if (p == 0) {
        even = f.w[b][h] & 0x0f0f0f0fu;
        odd = (f.w[b][h] >> 4) & 0x0f0f0f0fu;
        ev = nibble_pair_f32<false>(even);
        ov = nibble_pair_f32<false>(odd);
      } else if (p == 2) {
        ev = nibble_pair_f32<true>(even);
        ov = nibble_pair_f32<true>(odd);
      }
      return T::pack2(__builtin_fmaf(ev[p & 1], f.s[b], f.b[b]), __builtin_fmaf(ov[p & 1], f.s[b], f.b[b]));
    } else if constexpr (BITS == 8) {
      const uint32_t v = f.w[b][2 * h + (p >> 1)];
      return T::pack2(__builtin_fmaf(ubyte_f32(v, 2 * (p & 1)), f.s[b], f.b[b]),
                      __builtin_fmaf(ubyte_f32(v, 2 * (p & 1) + 1), f.s[b], f.b[b]));
    } else {
      return T::pack2(__builtin_fmaf((float)stream_code<BITS>(f.w[b], 8 * h + 2 * p), f.s[b], f.b[b]),
                      __builtin_fmaf((float)stream_code<BITS>(f.w[b], 8 * h + 2 * p + 1), f.s[b], f.b[b]));
    }
  };

  // Sub-step j + 1's operands have arrived, near the end, where nothing is requested any more: behind x(j + 1) there are
  // the loads of x of at most kXSlots - 1 sub-steps (chunks and windows, not counted, are requested in front of x in the
  // same sub-step).
  auto wait_next = [&](int j) __attribute__((always_inline)) {
    const int behind = min(n - 2 - j, S::kXSlots - 1);
    if (S::kXSlots >= 3 && behind >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S::kXLoads) : "memory");
    else if (behind >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::kXLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  u32x4 cur, nxt;
  constexpr int kInstr = S::kInstr, kReadsAt = S::kReadsAt;
  auto step = [&](auto more_x_c, auto more_c, Frag& f, Frag& next, int j, int slot) __attribute__((always_inline)) {
    constexpr bool more_x = decltype(more_x_c)::value, more = decltype(more_c)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this sub-step's operands are in registers: their slots are free
    // a chunk's (a window's) last sub-step: its slot takes the one after the next
    const bool chunk = j % S::kChunk == S::kChunk - 1 && (j / S::kChunk + 2) * S::kChunk < n;
    if (chunk) load_w(j / S::kChunk + 2);
    if (more) {
      const int g = (((begin + j) * 64 + 48) >> gs_shift) - g_first, g_next = (((begin + j + 1) * 64) >> gs_shift) - g_first;
      if ((g >> 3) != (g_next >> 3) && ((g >> 3) + 2) * 8 + g_first <= g_last) load_s((g >> 3) + 2);
    }
    const int after = slot + 1 == S::kXSlots ? 0 : slot + 1;
    // Younger than x(j + 1), which the reads below wait for: the slots behind it, and of x(j + kXSlots) what is requested by
    // then.  A chunk requested in this sub-step lies between the two: counted where every sub-step requests one (as long as
    // there is x to request there are codes), and by a branch in rings of two slots of x, which would wait for what they
    // have just requested (uncounted: 8 bits, 64 x 96, 4 % of the call, 5 bits 2 to 3 %).  In the others that branch costs 1
    // to 2 %, and a chunk's own sub-step (one in two or four) waits for a part of x(j + 2) instead; a window's (one in
    // eight groups) does everywhere.
    constexpr int kYounger = (S::kXSlots - 2) * S::kXLoads + S::loads_before_reads();
#pragma unroll
    for (int i = 0; i < 2 * kB; ++i) {
#pragma unroll
      for (int a = 0; a < kA; ++a) {
        const int at = i * kA + a;
        acc[a][i % kB] = mfma16(__builtin_bit_cast(vec8, cur), f.x[a][i / kB], acc[a][i % kB]);
        if (more_x) {
#pragma unroll
          for (int l = 0; l < S::kXLoads; l += S::kXGroup)
            if (S::load_slot(l) == at) load_x(j + S::kXSlots, slot, l);
        }
        if (more) {
          if (at == kReadsAt) {
            if constexpr (!more_x) wait_next(j);
            else if (S::kChunk == 1 || (S::kXSlots == 2 && chunk)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger + S::kWLoads) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger) : "memory");
          }
#pragma unroll
          for (int b = 0; b < kB; ++b)
            if (at == kReadsAt + b) read_codes(next, j + 1, b);
#pragma unroll
          for (int l = 0; l < 2 * kA; ++l)
            if (at == kReadsAt + l * (kInstr - kReadsAt - kA) / (2 * kA)) read_x(next, after, l);
        }
        if (more && i == 2 * kB - 1 && a == 0) align_codes(next);
#pragma unroll
        for (int p = 4 * a / kA; p < 4 * (a + 1) / kA; ++p) if (more || i + 1 < 2 * kB) nxt[p] = i + 1 < 2 * kB ? pair(f, i + 1, p) : pair(next, 0, p);
        __builtin_amdgcn_sched_barrier(0);
      }
      cur = nxt;
    }
  };

  if (n > 0) {
    load_w(0);
    load_s(0);
#pragma unroll
    for (int j = 0; j < S::kXSlots; ++j)
      if (j < n) {
#pragma unroll
        for (int i = 0; i < S::kXLoads; i += S::kXGroup) load_x(j, j, i);
        if (j == 0) {
          if (n > S::kChunk) load_w(1);
          if (8 + g_first <= g_last) load_s(1);
        }
      }
    Frag f0, f1;
    wait_next(-1);
#pragma unroll
    for (int b = 0; b < kB; ++b) read_codes(f0, 0, b);
#pragma unroll
    for (int l = 0; l < 2 * kA; ++l) read_x(f0, 0, l);
    align_codes(f0);
#pragma unroll
    for (int p = 0; p < 4; ++p) cur[p] = pair(f0, 0, p);
    int slot = 0, j = 0;
    auto advance = [&]() __attribute__((always_inline)) { slot = slot + 1 == S::kXSlots ? 0 : slot + 1; };
    const std::true_type yes{};
    const std::false_type no{};
    for (; j + S::kXSlots + 1 < n; j += 2) {
      step(yes, yes, f0, f1, j, slot);
      advance();
      step(yes, yes, f1, f0, j + 1, slot);
      advance();
    }
    // at most kXSlots + 1 are left, of which the first may have an x to request
    bool odd_frag = false;
    for (; j < n; ++j) {
      const bool mx = j + S::kXSlots < n;
      if (!odd_frag) {
        if (mx) step(yes, yes, f0, f1, j, slot);
        else if (j + 1 < n) step(no, yes, f0, f1, j, slot);
        else step(no, no, f0, f1, j, slot);
      } else {
        if (j + 1 < n) step(no, yes, f1, f0, j, slot);
        else step(no, no, f1, f0, j, slot);
      }
      odd_frag = !odd_frag;
      advance();
    }
  }

  // low-rank update: 32 of its k at a time, dealt to the wavefronts; of the k ranges of a tile the first one adds it
  for (int k = 32 * wave; split == 0 && k < lr_rank; k += 32 * kWaves) {
    const bool in = k + 8 * q < lr_rank;
    const int kk = in ? k + 8 * q : 0;
    vec8 zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = 0;
    vec8 wf[kB], xf[kA];
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      wf[b] = *reinterpret_cast<const vec8*>(lr_bs + (int64_t)weight_row(16 * b + r) * lr_rank + kk);
      if (!in) wf[b] = zero;
    }
#pragma unroll
    for (int a = 0; a < kA; ++a) {
      xf[a] = *reinterpret_cast<const vec8*>(lr_t + (int64_t)min(m0 + 16 * a + r, M - 1) * lr_rank + kk);
      if (!in) xf[a] = zero;
    }
#pragma unroll
    for (int a = 0; a < kA; ++a)
#pragma unroll
      for (int b = 0; b < kB; ++b) acc[a][b] = mfma16(wf[b], xf[a], acc[a][b]);
  }

  // ---- the partial tiles meet in LDS, kBand row blocks at a time; a thread finishes eight columns of a row
  constexpr int kChunks = S::TN / 8;
#pragma unroll
  for (int a0 = 0; a0 < kA; a0 += S::kBand) {
    __syncthreads();
#pragma unroll
    for (int a = a0; a < a0 + S::kBand && a < kA; ++a)
#pragma unroll
      for (int b = 0; b < kB; ++b)
        *reinterpret_cast<f32x4*>(lds + wave * S::kPart + (16 * (a - a0) + r) * S::kStride + (16 * b + 4 * q) * 4) = acc[a][b];
    __syncthreads();
    for (int c = t; c < S::kBand * 16 * kChunks; c += kThreads) {
      const int in_band = c / kChunks, col = (c % kChunks) * 8, row = m0 + 16 * a0 + in_band;
      if (16 * a0 + in_band >= S::TM || row >= M) break;
      if (swiglu ? col >= S::TN / 2 || n0 / 2 + col >= N / 2 : n0 + col >= N) continue;
      // the linear layer's value: rounded, then the bias added and rounded again (float32 y: one float32 sum)
      auto linear8 = [&](int cc, float (&v)[8]) __attribute__((always_inline)) {
        f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
        const char* p = lds + in_band * S::kStride + cc * 4;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          lo += *reinterpret_cast<const f32x4*>(p + w * S::kPart);
          hi += *reinterpret_cast<const f32x4*>(p + w * S::kPart + 16);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = lo[e];
          v[4 + e] = hi[e];
        }
        if (!y_is_f32) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = round_to<T>(v[e]);
        }
        if (bias) {
          const uint16_t* b = bias + weight_row(cc);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += T::to_f32(b[e]);
          if (!y_is_f32) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = round_to<T>(v[e]);
          }
        }
      };
      float v[8];
      linear8(col, v);
      const int64_t o = (int64_t)row * N + n0 + col;
      if (y_is_f32) {
        float* dst = reinterpret_cast<float*>(y) + (int64_t)split * M * N + o;  // (split > 0 only with float32 planes)
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
        continue;
      }
      int64_t dst = o;
      if (swiglu) {
        float up[8];
        linear8(col + S::TN / 2, up);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = epi_swiglu<T>(v[e], up[e]);
        dst = (int64_t)row * (N / 2) + n0 / 2 + col;
      } else if (epi.kind == kEpiGelu && n0 + col >= epi.act_from) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = epi_gelu<T>(v[e]);
      } else if (epi.kind == kEpiGateResidual) {
        const u32x4 g = *reinterpret_cast<const u32x4*>(epi.gate + n0 + col);
        const u32x4 res = *reinterpret_cast<const u32x4*>(epi.residual + o);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] = epi_gate_residual<T>(v[2 * e], lo_f32<T>(g[e]), lo_f32<T>(res[e]));
          v[2 * e + 1] = epi_gate_residual<T>(v[2 * e + 1], hi_f32<T>(g[e]), hi_f32<T>(res[e]));
        }
      }
      u32x4 out;
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = T::pack2(v[2 * e], v[2 * e + 1]);
      *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(y) + dst) = out;
    }
  }
}

// ---- which tile, and whether at all.
//
// Time of a call by tile, from 3000 drawn shapes on each tile (2 to 1023 rows, 3 to 8 bits, groups of 32 to 128, cold weights,
// a stream of launches; the fit is 7 to 8 % rms): 3.1 us and, for each round of workgroups, `first` (first bytes, partial tiles,
// store; it grows with the tile) and `step` for every sub-step of a wavefront.  A cut of K over workgroups costs the launch of
// the second kernel and its planes, 3.4 us and 1.3 bytes/ps.  (With one first cost for all tiles the wide tiles on short K
// came out up to 40 % too low.)
// 80 columns: the widest tile whose ring still holds three slots of x with two sub-steps of 4-bit codes (96 columns: one), or
// with 8-bit codes (96: two slots of x).  Where 64 columns take a round more, or the 128-column kernel a cut: 170 drawn calls
// of 17 to 512 rows, K whole, 0.70 to 1.02 of the time without it, 0.88 in the mean (48 rows x 3584 -> 37888 at 4 bits 44.0 us ->
// 38.8, at 6 bits 21 rows 55.4 -> 42.0; 35 x 4096 -> 20480 at 8 bits 25.8 -> 24.3; 512 x 3072 -> 2560 at 4 bits 18.9 -> 17.0).
// With K cut over workgroups 0.97 to 1.06 (6 bits 44 x 18944 -> 3584 in groups of 32 31.6 -> 33.1): such cuts keep the other
// tiles.  At 3 bits 96 columns take no longer where they are no more rounds (17 x 4096 -> 20480 24.1, 25.0): its step is set
// above theirs.
struct Tile {
  int rows, columns;
  float first, step[5];  // us; the step at 3, 4, 5, 6, 8 bits
};
constexpr Tile kTiles[] = {
    {32, 32, 1.8f, {0.43f, 0.47f, 0.58f, 0.60f, 0.54f}}, {64, 32, 2.7f, {0.58f, 0.55f, 0.64f, 0.65f, 0.59f}},
    {64, 48, 3.9f, {0.74f, 0.67f, 0.80f, 0.81f, 0.70f}}, {64, 64, 4.8f, {0.91f, 0.74f, 0.97f, 0.96f, 0.83f}},
    {64, 80, 5.9f, {1.33f, 0.87f, 1.15f, 1.10f, 0.94f}}, {64, 96, 6.9f, {1.22f, 1.01f, 1.33f, 1.50f, 1.05f}},
};

struct SlicePlan {
  int rows = 0, columns = 0, splits = 0;
  float us = 0.f;
};

// *without_80 (0 on entry): the time of the best of the other tiles
inline SlicePlan plan_slice(int64_t M, int64_t N, int64_t K, int bits, bool may_cut, float* without_80) {
  const int64_t cus = compute_units();
  const int gran = bits == 3 || bits == 5 ? 2 : 1, grains = (int)(K / (64 * gran));
  const int width = bits == 3 ? 0 : bits == 4 ? 1 : bits == 5 ? 2 : bits == 6 ? 3 : 4;
  SlicePlan best;
  for (const Tile& t : kTiles) {
    if (t.rows == 32 && M > 128) continue;  // (every code is then dequantised for five row tiles and more)
    const int64_t tiles = ((M + t.rows - 1) / t.rows) * ((N + t.columns - 1) / t.columns);
    for (int s = 1; s == 1 || (may_cut && t.columns != 80 && s <= 8 && tiles * s <= cus && K / 64 / s >= 8); ++s) {
      const int64_t rounds = (tiles * s + cus - 1) / cus;
      const int subs = (grains + kWaves * s - 1) / (kWaves * s) * gran;
      float us = 3.1f + (float)rounds * (t.first + (float)subs * t.step[width]);
      if (s > 1) us += 3.4f + (float)(s * M * N) * (4.f / 1.3e6f);
      if (t.columns != 80 && (*without_80 == 0.f || us < *without_80)) *without_80 = us;
      if (best.splits == 0 || us < best.us) best = SlicePlan{t.rows, t.columns, s, us};
    }
  }
  return best;
}

// What the 128-column-tile kernel takes on the same shapes: its own estimate leaves out 4.3 us of launch and first bytes,
// 0.15 us for each plane of a cut, and what a bit stream's codes cost it (3, 5 and 6 bits).
inline float others_us(int64_t M, int64_t N, int64_t K, int gs, int bits) {
  const int ranges = qmm_mid_ranges(M, N, K, gs);
  const float width = bits == 3 ? 1.08f : bits == 4 ? 1.02f : bits == 5 ? 1.16f : bits == 6 ? 1.12f : 1.03f;
  return 4.3f + width * qmm_mid_estimate_us(M, N, K, gs) + (ranges > 1 ? 0.15f * (float)ranges : 0.f);
}

// Taken where its estimate is a tenth below that one.  Of 11900 drawn calls (2 to 1023 rows at 3, 5 and 6 bits, 17 to 1023 at 4
// and 8; model sizes and short K) 6900 are, in 0.71 of the other kernel's time (geometric mean; 2 to 16 rows 0.77), 15 of them
// 3 % or more behind it and 5 by 6 to 9 % (6 bits 126 rows x 3072 -> 12288 31.0 -> 33.8 us): both estimates are off by some 7 %.
// Before the tiles' first costs were told apart (2.4 us each) and the other kernel's planes and widths counted, 235 calls were
// 3 % behind, 123 by more than 6 (6 bits 33 x 768 -> 37888 19.8 -> 27.3 us, 76 x 3072 -> 12288 28.8 -> 33.0).
inline SlicePlan choose_slice(int64_t M, int64_t N, int64_t K, int gs, int bits, bool may_cut) {
  const int64_t gran = bits == 3 || bits == 5 ? 128 : 64;
  if (M > 1024 || N % 8 || K % gran || (K / gs) % 2 || M * K >= ((int64_t)1 << 31) - 2048 || N * K >= (int64_t)1 << 31) return SlicePlan();
  float without_80 = 0.f;
  const SlicePlan plan = plan_slice(M, N, K, bits, may_cut, &without_80);
  // (the 80 columns were measured against the other kernel in groups of 32 and 64: in groups of 128 they take no calls from it)
  return (gs == 128 ? without_80 : plan.us) < 0.9f * others_us(M, N, K, gs, bits) ? plan : SlicePlan();
}

template <typename T, int BITS, int kA, int kB>
int launch_kernel(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales, const void* biases,
                  const void* bias, int64_t N, int gs, int splits, void* y, int y_dtype, hipStream_t stream, LowRank lr,
                  Epilogue epi) {
  auto kernel = qmm_slice_kernel<T, BITS, kA, kB>;
  using S = Shape<BITS, kA, kB>;
  static PerDeviceInt configured;
  if (!raise_lds_limit(configured, reinterpret_cast<const void*>(kernel), S::kLds)) return MFQ_ELAUNCH;
  const int tiles_m = (int)((M + S::TM - 1) / S::TM), tiles_n = (int)((N + S::TN - 1) / S::TN);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(kThreads), S::kLds, stream, (const uint16_t*)x, wq,
                     (const uint16_t*)scales, (const uint16_t*)biases, (const uint16_t*)bias, y,
                     (int)(y_dtype == MFQ_F32), (int)M, (int)N, (int)K, gs == 32 ? 5 : gs == 64 ? 6 : 7, tiles_m, tiles_n, splits,
                     (const uint16_t*)lr.t, (const uint16_t*)lr.bs, lr.R, epi);
  return hipGetLastError() == hipSuccess ? MFQ_OK : MFQ_ELAUNCH;
}

template <typename T, int BITS>
int launch_tile(SlicePlan plan, const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                   const void* biases, const void* bias, int64_t N, int gs, void* y, int y_dtype, hipStream_t stream,
                   LowRank lr, Epilogue epi) {
  const auto go = [&](auto launch) {
    return launch(x, M, K, wq, scales, biases, bias, N, gs, plan.splits, y, y_dtype, stream, lr, epi);
  };
  if (plan.rows == 32) return go(launch_kernel<T, BITS, 2, 2>);
  switch (plan.columns) {
    case 32: return go(launch_kernel<T, BITS, 4, 2>);
    case 48: return go(launch_kernel<T, BITS, 4, 3>);
    case 64: return go(launch_kernel<T, BITS, 4, 4>);
    case 80: return go(launch_kernel<T, BITS, 4, 5>);
    default: return go(launch_kernel<T, BITS, 4, 6>);
  }
}

template <typename T>
int launch_bits(SlicePlan plan, const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype,
                hipStream_t stream, LowRank lr, Epilogue epi) {
  switch (bits) {
    case 3: return launch_tile<T, 3>(plan, x, M, K, wq, scales, biases, bias, N, gs, y, y_dtype, stream, lr, epi);
    case 4: return launch_tile<T, 4>(plan, x, M, K, wq, scales, biases, bias, N, gs, y, y_dtype, stream, lr, epi);
    case 5: return launch_tile<T, 5>(plan, x, M, K, wq, scales, biases, bias, N, gs, y, y_dtype, stream, lr, epi);
    case 6: return launch_tile<T, 6>(plan, x, M, K, wq, scales, biases, bias, N, gs, y, y_dtype, stream, lr, epi);
    default: return launch_tile<T, 8>(plan, x, M, K, wq, scales, biases, bias, N, gs, y, y_dtype, stream, lr, epi);
  }
}

}  // namespace

int qmm_slice_ranges(int64_t M, int64_t N, int64_t K, int gs, int bits) { return choose_slice(M, N, K, gs, bits, true).splits; }

void qmm_slice_tile(int64_t M, int64_t N, int64_t K, int gs, int bits, int* rows, int* columns) {
  const SlicePlan plan = choose_slice(M, N, K, gs, bits, true);
  *rows = plan.rows;
  *columns = plan.columns;
}

float qmm_slice_estimate_us(int64_t M, int64_t N, int64_t K, int gs, int bits) {
  return choose_slice(M, N, K, gs, bits, true).us;
}

int launch_qmm_slice(const void* x, int dtype, int64_t M, int64_t K, const uint32_t* wq, const void* scales,
                     const void* biases, const void* bias, int64_t N, int gs, int bits, void* y, int y_dtype,
                     void* workspace, size_t workspace_bytes, hipStream_t stream, LowRank low_rank, Epilogue epi) {
  if (dtype != MFQ_BF16 && dtype != MFQ_F16) return MFQ_EUNSUPPORTED;
  // scales and biases are requested a dword (two groups) at a time; a float32 y has no epilogue
  if (((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) || (epi.kind != kEpiNone && y_dtype == MFQ_F32))
    return MFQ_EUNSUPPORTED;
  SlicePlan plan = choose_slice(M, N, K, gs, bits, true);
  const bool cut = plan.splits > 1;
  if (cut && (!workspace || !aligned16(workspace) || workspace_bytes < (size_t)plan.splits * M * N * sizeof(float)))
    plan = choose_slice(M, N, K, gs, bits, false);
  if (plan.splits == 0) return MFQ_EUNSUPPORTED;
  const auto go = [&](auto launch) {
    if (plan.splits == 1)
      return launch(plan, x, M, K, wq, scales, biases, bias, N, gs, bits, y, y_dtype, stream, low_rank, epi);
    // K cut over workgroups: float32 planes, and the second kernel applies bias and epilogue
    const int rc = launch(plan, x, M, K, wq, scales, biases, nullptr, N, gs, bits, workspace, MFQ_F32, stream, low_rank, Epilogue());
    return rc ? rc : launch_splitk_reduce(dtype, workspace, plan.splits, M, N, bias, y, y_dtype, stream, epi);
  };
  return dtype == MFQ_BF16 ? go(launch_bits<BF16>) : go(launch_bits<F16>);
}

}  // namespace mfq
