// Output-tile schedules and their product kernels.
//
// The same block products as the triplet kernels (m_kern_max / m_kern_min,
// src/multiply_kernel_default.f90:204-214 and :392-402), grouped so that
// operand blocks are read from HBM once per tile instead of once per product:
//
//  * a tile is 8 primary atoms (rows, consecutive in primary order) x 8 column
//    atoms (consecutive in the Morton order of their halo partitions) of the
//    output matrix: type 1 C(i,j), columns in the C halo, contraction over the
//    A-halo atom k; type 2 X(i,k), columns in the A halo, contraction over the
//    C-halo atom j;
//  * an entry of a tile is one contraction atom x with its (up to 8) left
//    operand blocks P(row, x) and (up to 8) right operand blocks Q(column, x);
//    entries of a tile are in ascending x (type 1: the reference's k order);
//  * uniform sizes: each 4x4-block quadrant of a tile is the work of one
//    wavefront of its own, driven by a list of records (k_wave_products,
//    k_quad4);
//  * the other kernels run a tile with one workgroup (4 wavefronts, three
//    workgroups per CU). Chunks of entries have their operand blocks copied
//    HBM->LDS (global_load_lds, no registers) into one of two stages while the
//    previous chunk is computed from the other (one barrier per chunk); each
//    wavefront accumulates 16 output blocks of the tile with MFMA from LDS.
//    Mixed sizes: ownership is a Latin square (two blocks per tile row and
//    column per wavefront), chosen when the plan is built to balance the
//    wavefronts' product counts, and the plan holds each wavefront's products
//    of each chunk as a list of packed LDS offsets sorted by the wavefront's
//    output block and, within a block, by entry, with the count per block in
//    one 64-bit word (16 x 4 bits): no product discovery at run time;
//  * every output block is written once (zeros where it has no products), so
//    the output is fully overwritten as mat_mult overwrites it
//    (src/multiply_module.f90:204-208).
// Summation order per output block is fixed (ascending x), so results are
// bitwise reproducible run to run.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include <rocprim/rocprim.hpp>

#include "../../include/cqmm.h"
#include "cq_common.h"
#include "cq_device.h"

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// Four split-BF16 words -> their hi halves (bits 0-15) or lo halves (bits
// 16-31) as the four BF16 elements of an MFMA operand.
__device__ inline s16x4 pack_bf16_lo(const uint32_t w[4]) {
  const uint32_t x = __builtin_amdgcn_perm(w[1], w[0], 0x05040100u);
  const uint32_t y = __builtin_amdgcn_perm(w[3], w[2], 0x05040100u);
  return __builtin_bit_cast(s16x4, (uint64_t)x | ((uint64_t)y << 32));
}
__device__ inline s16x4 pack_bf16_hi(const uint32_t w[4]) {
  const uint32_t x = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u);
  const uint32_t y = __builtin_amdgcn_perm(w[3], w[2], 0x07060302u);
  return __builtin_bit_cast(s16x4, (uint64_t)x | ((uint64_t)y << 32));
}

// In place: split-BF16 words of contraction indices 4g..4g+3 (indices >= NSF
// zeroed) -> the hi (registers 0, 1) and lo (2, 3) operands of
// v_mfma_f32_16x16x16_bf16.
template <int NSF>
__device__ inline void split_words(float *k, int g) {
  uint32_t x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = (NSF < 16 && 4 * g + i >= NSF) ? 0u : __float_as_uint(k[i]);
  k[0] = __uint_as_float(__builtin_amdgcn_perm(x[1], x[0], 0x05040100u));
  k[1] = __uint_as_float(__builtin_amdgcn_perm(x[3], x[2], 0x05040100u));
  k[2] = __uint_as_float(__builtin_amdgcn_perm(x[1], x[0], 0x07060302u));
  k[3] = __uint_as_float(__builtin_amdgcn_perm(x[3], x[2], 0x07060302u));
}
__device__ inline s16x4 half_of(const float *k, int i) {
  return __builtin_bit_cast(s16x4, (uint64_t)__float_as_uint(k[i]) | ((uint64_t)__float_as_uint(k[i + 1]) << 32));
}

constexpr int kWaves = 4;                    // wavefronts per workgroup (one tile)
constexpr int kTileThreads = 64 * kWaves;
constexpr int kSlots = 64 / kWaves;          // output blocks per wavefront
static_assert(8 % kWaves == 0, "a tile row of 8 blocks is split evenly over the wavefronts");
// LDS reads of a block product never mask rows or columns beyond NSF: those
// lanes only feed accumulator rows/columns >= NSF, which are never written.
// Only the contraction index 4*s+g >= NSF at the last k-step is zeroed (both
// operands), so the padding of the 16x16x4 steps adds nothing. kLdsPad doubles
// after each stage keep the over-reads of its last block inside the array.
constexpr int kLdsPad = 256;
constexpr int kChunkEntries = 15;            // entries per chunk at most (4-bit product counts)
constexpr int kWaveProducts = 64;            // products per wavefront per chunk at most (one per lane)
constexpr int kDenseNsf = 4;                 // block size of the dense-quadrant kernel
constexpr int kDenseEntries = 64;            // entries per chunk at most there (one per lane)

// Prefetch loads are unconditional (indices clamped or arrays padded) so that
// no value is consumed before the next barrier: a use right after the load
// would make the wavefront wait for every outstanding load, including the
// stage copies that are meant to overlap the compute.

// One 256-byte piece of a block copy: lane l moves dword OFF/4 + l. The
// immediate offset applies to both the global and the LDS address (one M0 per
// block).
template <int OFF>
__device__ inline void dma_piece(const uint32_t *src, uint32_t *dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                   (__attribute__((address_space(3))) void *)dst, 4, OFF, 0);
}

using cq::TileArgs;
using cq::TileGroup;
using cq::TileOne;
using cq::kMaxGroup;

// Launch units [lo, hi) of this workgroup's XCD: workgroup b runs on XCD b % 8, and
// each XCD takes consecutive units (same rows), which share its L2. All nine
// bounds are read at fixed places of the arguments: one load indexed by the XCD
// costs the mixed sizes 1.5% (4096 atoms 4/9/13 27.6 -> 28.0 ms).
__device__ inline void xcd_units(const int32_t (&xcd)[cq::kXcds + 1], int32_t &lo, int32_t &hi) {
  const int32_t x = (int32_t)(blockIdx.x & 7);
  lo = xcd[0];
  hi = xcd[1];
#pragma unroll
  for (int k = 1; k < cq::kXcds; ++k) {
    lo = x == k ? xcd[k] : lo;
    hi = x == k ? xcd[k + 1] : hi;
  }
}

// This workgroup's launch unit, -1 past its XCD's last.
__device__ inline int32_t xcd_tile(const int32_t (&xcd)[cq::kXcds + 1]) {
  int32_t lo, hi;
  xcd_units(xcd, lo, hi);
  const int32_t t = lo + (int32_t)(blockIdx.x >> 3);
  return t < hi ? t : -1;
}

__device__ inline int32_t tile_select(const TileOne &one, TileArgs &a) {
  a = one.a;
  return xcd_tile(one.xcd);
}

// A grouped launch numbers the tiles of its products consecutively (product j
// from g.a[j].tile_base); the arguments (kernel-argument memory, read with
// scalar loads) are those of the product the tile belongs to.
__device__ inline int32_t tile_select(const TileGroup &g, TileArgs &a) {
  const int32_t t = xcd_tile(g.xcd);
  if (t < 0) return -1;
  int32_t j = 0;
#pragma unroll
  for (int k = 1; k < kMaxGroup; ++k) j += (k < g.ngrp && g.a[k].tile_base <= t) ? 1 : 0;
  a = g.a[j];
  return t - a.tile_base;
}

__device__ inline int64_t readlane64(int64_t v, int k) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, k);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), k);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// MODE 0: FP64 operands, v_mfma_f64_16x16x4 (accumulator D[(l/16)+4e][l%16]).
// MODE 1: FP32 operands, v_mfma_f32_16x16x4, FP32 accumulation.
// MODE 2: FP32 operands and MFMA, each product's result added into FP64
//         registers (accumulator D[4(l/16)+e][l%16]).
// MODE 4: split-BF16 words, three v_mfma_f32_16x16x16_bf16 per product, each
//         product's FP32 sum added into FP64 registers.
//
// Operand registers of one NSF x NSF block, as the lane (r, g) = (l%16, l/16)
// supplies them to the matrix instruction.
template <int MODE, int NSF>
struct Frag {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  static constexpr int KS = (NSF + 3) / 4;               // k-steps of 4 contraction indices
  static constexpr bool R1 = MODE != 4 && NSF % 4 == 1;  // the last contraction index on the VALU
  static constexpr int KM = MODE == 4 ? 4 : (R1 ? KS - 1 : KS);  // registers of the matrix steps
  static_assert(NSF % 4 <= 1, "block sizes 4m and 4m + 1");
  // A lane's accumulator rows that can lie in a block (FP64 g + 4e, FP32 4g + e).
  static constexpr int ROWS = MODE == 0 ? KS : 4;
  T k[KM];       // element of each matrix step (MODE 4: hi and lo operands, two registers each)
  T last[ROWS];  // R1: left, A[row][NSF-1] of these rows; right, B[NSF-1][r] in last[0]
};

// A block's bytes go to LDS 16 per lane; where they end inside the last lane's
// 16, that lane takes the block's last 16 bytes instead, so the last element
// lies wave_shift elements further than its index says (a copy instruction of
// its own for the 4 or 8 bytes left would be the third of a 13x13 FP64 block).
constexpr int wave_stride(int nsf, int size) { return (nsf * nsf * size + 15) / 16 * 16; }
constexpr int wave_shift(int nsf, int size) { return (wave_stride(nsf, size) - nsf * nsf * size) / size; }

// Element offsets in a block (as it lies in LDS) of a lane's operands: of its
// first register (MODE 4: of each) and of the last contraction index. Lanes
// beyond the block's rows, columns or indices read an element that feeds only
// results that are not written.
template <int MODE, bool RIGHT, bool QT, int NSF>
struct FragOff {
  using F = Frag<MODE, NSF>;
  static constexpr bool KMAJ = RIGHT && !QT;   // contraction index fastest
  static constexpr int N = MODE == 4 ? 4 : 1;
  static constexpr int END = NSF * NSF - 1, SHIFT = wave_shift(NSF, MODE == 0 ? 8 : 4);
  static_assert(SHIFT == 0 || (NSF % 4 == 1 && SHIFT == (MODE == 0 ? 1 : 3)), "only the last element is shifted");
  int first[N], last;
  __device__ inline FragOff(int r, int g) {
    const int n = min(r, NSF - 1);
    auto at = [](int i) { return i == END ? i + SHIFT : i; };
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int k = MODE == 4 ? min(4 * g + i, NSF - 1) : g;
      first[i] = at(KMAJ ? k + NSF * n : n + NSF * k);
    }
    if (RIGHT) last = at(QT ? n + NSF * (NSF - 1) : NSF - 1 + NSF * n);
    // Accumulator rows: FP64 g + 4e (load() shifts row NSF - 1), FP32 4g + e.
    else last = MODE == 0 ? NSF * (NSF - 1) + g : at(NSF * (NSF - 1) + 4 * g);
  }
  template <class T>
  __device__ inline void load(const T *blk, int g, F &f) const {
    constexpr int STEP = KMAJ ? 4 : 4 * NSF;
#pragma unroll
    for (int i = 0; i < F::KM; ++i) f.k[i] = blk[first[N == 1 ? 0 : i] + (N == 1 ? STEP * i : 0)];
    if constexpr (F::R1) {
#pragma unroll
      for (int e = 0; e < (RIGHT ? 1 : F::ROWS); ++e)
        f.last[e] = blk[last + (MODE == 0 ? 4 * e + (!RIGHT && 4 * e == NSF - 1 ? SHIFT : 0) : e)];
    }
    if constexpr (MODE == 4) split_words<NSF>(f.k, g);
  }
};

// Wavefronts per SIMD. FP64 blocks of 13 and 16: two, with all operands of a record
// in registers. The others: three, with the left operands of one row at a time.
// FP64 9x9 needs the third to cover a record's scalar work, as its matrix steps
// are short: 2000 atoms, C(16 A) = A(8 A).B(12 A), 10.3 ms with two, 7.9 with three.
constexpr int wave_per_simd(int mode, int nsf) { return mode == 0 && nsf > 9 ? 2 : 3; }
// Ring of operand blocks of a wavefront: what its share of the 160 KB LDS
// holds beside the record words.
constexpr int kWaveWords = 256;  // record words in LDS
constexpr int kWavePad = 128;    // words after a plan's last record
constexpr int wave_dmas(int nsf, int size) { return (nsf * nsf * size + 1023) / 1024; }  // copies per block
constexpr int wave_ring(int mode, int nsf) {
  const int size = mode == 0 ? 8 : 4;
  const int r = ((wave_per_simd(mode, nsf) == 2 ? 20480 : 12800) - 4 * kWaveWords) / wave_stride(nsf, size);
  const int v = 63 / wave_dmas(nsf, size);  // the wait counts at most 63 copies
  return (r < v ? r : v) < 28 ? (r < v ? r : v) : 28;
}

// The lane, worked out where it is needed and not held in a register until then.
__device__ inline int lane_again() {
  uint32_t ones = ~0u;
  asm volatile("" : "+s"(ones));
  return (int)__builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u));
}

// One operand block from memory to LDS. `lane16`: 16 * lane, and `end16` that of
// the last copy (its last lane takes the block's last 16 bytes); opaque, so that
// they stay 32-bit offsets from the scalar block address.
template <int BYTES>
__device__ inline void dma_block(const char *src, char *dst, uint32_t &lane16, uint32_t &end16, int lane) {
  constexpr int LANES = (BYTES + 15) / 16, N = (LANES + 63) / 64, REST = LANES - 64 * (N - 1);
  auto d = (__attribute__((address_space(3))) void *)dst;
  if constexpr (N > 1) {
    asm volatile("" : "+v"(lane16));
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + lane16), d, 16, 0, 0);
  }
  static_assert(N <= 2, "blocks of at most 2 KB");
  if (REST == 64 || lane < REST) {
    asm volatile("" : "+v"(end16));
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + end16), d, 16,
                                     1024 * (N - 1), 0);
  }
}

// Waits until at most `after` blocks of PER copies each are in flight, `after`
// rounded down to N, N/2, .., 4 or 0.
template <int PER, int N>
__device__ inline void wait_blocks(int32_t after) {
  constexpr int v = N < 4 ? 0 : PER * N;
  __builtin_amdgcn_s_waitcnt((v & 15) | (v >> 4 << 14) | 0xf70);  // vmcnt only
  if constexpr (N >= 4) {
    if (after < N) wait_blocks<PER, N / 2>(after);
  }
}

// Uniform block sizes 9, 13, 16: one wavefront computes 4x4 output blocks (a
// quadrant of a tile) in 16 accumulators, on its own: no barrier, no other
// wavefront to wait for. Its records (contraction atoms, ascending) list the
// present blocks of 4 rows and 4 columns. The blocks of the next records are
// copied memory -> LDS into a ring while the oldest record's products run from
// registers: every operand element is read from LDS once per record, and every
// present pair with an output block is a bit test and the matrix steps.
//
// What bounds it (gfx950): a VALU instruction holds the SIMD as a matrix
// instruction does (3 f64 MFMA take 217 cycles, with 16 VALU instructions of any
// wavefront between them 292), so a product costs its matrix steps plus 4.6
// cycles per VALU instruction, and the design keeps these few. What is left
// is the scalar work and the branches of a record (4096 atoms 13x13, type 2: 31
// scalar instructions and 7 branches per product against 3 matrix steps and 7
// other VALU instructions, the matrix cores busy 48%) and, at thousands of
// atoms, the copies beyond L2 (copies alone 34.5 ms, everything else 37.5 ms).
// Against one workgroup per 8x8 tile with its four wavefronts in step (a barrier
// per chunk; the busiest wavefront has 1.25 to 1.56 times the mean products):
// 13x13 FP64 4096 atoms type 2 50.6 -> 44.8 ms, 1024 atoms symmetric
// 15.8 -> 13.15 ms, 9x9 FP32 with FP64 sums 1500 atoms 11.0 -> 8.74 ms, 13x13 split
// BF16 1024 atoms 5.92 -> 4.02 ms (0.8 of it the FP64 result written here, not
// widened by a pass of its own), 9x9 FP64 2000 atoms 8/12/16 A 9.97 -> 7.80 ms, 16x16 FP64
// 1500 atoms 8/12/16 A 29.3 -> 14.2 ms, type 2 12/12/8 A 10.0 -> 7.73 ms, one LNV
// evaluation of 60 atoms 9x9 12.4 -> 9.6 ms.
// Tried and slower: operands straight to registers (4096 atoms 58 ms: 18 to 33
// address cycles per load), two stages instead of the ring (split BF16 6.2 ms),
// three wavefronts per SIMD with right operands read per product (9x9 11.1 ms).
//
// NSF = 4m + 1: the last contraction index is a rank-1 update on the VALU (four
// fused multiply-adds after the matrix steps; a matrix step with three zeroed
// indices takes 72 cycles in FP64).
template <int MODE, bool QT, int NSF, class ARG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(wave_per_simd(MODE, NSF))))
k_wave_products(const ARG arg) {
  using F = Frag<MODE, NSF>;
  using T = typename F::T;
  constexpr int NS2 = NSF * NSF;
  constexpr int BYTES = NS2 * (int)sizeof(T);
  constexpr int LB = wave_stride(NSF, (int)sizeof(T));
  constexpr int RING = wave_ring(MODE, NSF), PER = wave_dmas(NSF, (int)sizeof(T));
  static_assert(RING >= 8, "the ring holds every record");
  constexpr bool ALL_LEFT = wave_per_simd(MODE, NSF) == 2;  // left operands of the record in registers, or of a row
  constexpr bool TIGHT = MODE == 0 && !ALL_LEFT;            // every register of the three wavefronts' share is used
  __shared__ __attribute__((aligned(16))) char lds[RING * LB + 4 * kWaveWords];
  TileArgs a;
  const int32_t tile = tile_select(arg, a);
  if (tile < 0) return;
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  const char *P = static_cast<const char *>(a.P), *Q = static_cast<const char *>(a.Q);
  // The quadrant's output blocks (-1: none), in scalar registers, and bit
  // 4*row + column of `valid`. Read here: a load per block between the stores
  // of the results would wait for the stores before it (13x13 FP64, 3000 atoms,
  // 6/6/12 A, lists of some 25 records: 1.66 ms that way, 1.56 ms this way).
  const int32_t my_out = a.wave_out[(int64_t)tile * 16 + r];
  const uint32_t valid = (uint32_t)__ballot(my_out >= 0) & 0xffffu;
  int32_t out_blk[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) out_blk[u] = __builtin_amdgcn_readlane(my_out, u);
  dbl4 a64[16];
  flt4 a32[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    a64[u] = dbl4{0.0, 0.0, 0.0, 0.0};
    a32[u] = flt4{0.f, 0.f, 0.f, 0.f};
  }
  const int64_t w0 = a.pstart[tile];
  const int32_t nw = (int32_t)(a.pstart[tile + 1] - w0);
  {
    const FragOff<MODE, false, QT, NSF> oP(r, g);
    const FragOff<MODE, true, QT, NSF> oQ(r, g);
    constexpr int LANES = (BYTES + 15) / 16, LAST = (LANES - 1) % 64;
    uint32_t l4 = 4u * (uint32_t)lane, lane16 = 16u * (uint32_t)lane;
    uint32_t end16 = lane16 - (lane == LAST ? (uint32_t)(LB - BYTES) : 0u);
    // Record words: a record is rows present | columns present << 4, then the
    // present blocks (left by row, right by column). They come to LDS in pieces
    // of 64 words, three pieces ahead, and from there to a register of the
    // lanes, word `i` of the list in lane i - base. A piece is first read at
    // least 43 block copies after it was issued (65 words, two of three of them
    // blocks), more than the ring's, so the waits for blocks cover it.
    const char *words = (const char *)(a.prod + w0);
    char *wring = lds + RING * LB;
    auto piece = [&](int32_t j) {
      if (64 * j >= nw) return;
      if constexpr (TIGHT) l4 = 4u * (uint32_t)lane_again();
      asm volatile("" : "+v"(l4));
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(words + 256 * (int64_t)j + l4),
                                       (__attribute__((address_space(3))) void *)(wring + 256 * (j & 3)), 4, 0, 0);
    };
    int32_t at = 0, base = 0;
    uint32_t win;
    auto refill = [&]() {
      base = at;
      win = ((const uint32_t *)wring)[(at + (TIGHT ? lane_again() : lane)) % kWaveWords];
    };
    auto word = [&](int32_t i) { return (uint32_t)__builtin_amdgcn_readlane((int)win, i - base); };
    for (int32_t j = 0; j < 4; ++j) piece(j);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
    refill();
    uint64_t queue = 0;             // masks of the records in the ring, oldest in the low byte
    int32_t nq = 0, held = 0;       // records, blocks in the ring
    int32_t head = 0, tail = 0;     // LDS offsets of the oldest block and of the next free slot
    uint32_t coming = nw > 0 ? word(0) : 0u;  // masks of the record at `at`, 0 past the last
    auto fits = [&]() {
      return (nq < 8) & (coming != 0) & (held + __builtin_popcount(coming) <= RING);
    };
    auto issue = [&]() {
      const uint32_t m = coming;
      held += __builtin_popcount(m);
      queue |= (uint64_t)m << (8 * nq++);
      ++at;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (!(m >> k & 1u)) continue;
        dma_block<BYTES>((k < 4 ? P : Q) + (int64_t)word(at++) * BYTES, lds + tail, lane16, end16, lane);
        tail = tail == (RING - 1) * LB ? 0 : tail + LB;
      }
      if (at + 9 > base + 64) {
        const int32_t j = at >> 6;
        if (j != base >> 6) piece(j + 3);
        refill();
      }
      coming = at < nw ? word(at) : 0u;
    };
    while (fits()) issue();
    if (nq > 0) do {
      const uint32_t m = (uint32_t)queue & 0xffu;
      const int32_t n = __builtin_popcount(m);
      queue >>= 8;
      --nq;
      asm volatile("" ::: "memory");
      wait_blocks<PER, (RING >= 20 ? 16 : 8)>(held - n);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // no LDS read is pending here; the compiler takes note
      asm volatile("" ::: "memory");
      const uint32_t cols = m >> 4;
      auto step = [&](int32_t &o, int32_t by) {
        o += by * LB;
        o = o >= RING * LB ? o - RING * LB : o;
        o = __builtin_amdgcn_readfirstlane(o);
      };
      int32_t pq = head;
      step(pq, __builtin_popcount(m & 15u));
      F right[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (!(cols >> k & 1u)) continue;
        oQ.load((const T *)(lds + pq), g, right[k]);
        step(pq, 1);
      }
      F left[ALL_LEFT ? 4 : 1];
      if constexpr (ALL_LEFT) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (!(m >> u & 1u)) continue;
          oP.load((const T *)(lds + head), g, left[u]);
          step(head, 1);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (!(m >> u & 1u)) continue;
        if constexpr (!ALL_LEFT) {
          oP.load((const T *)(lds + head), g, left[0]);
          step(head, 1);
        }
        const F &x = left[ALL_LEFT ? u : 0];
        const uint32_t todo = (valid >> (4 * u)) & cols;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (!(todo >> k & 1u)) continue;
          const F &y = right[k];
          if constexpr (MODE == 0) {
            dbl4 &d = a64[4 * u + k];
#pragma unroll
            for (int i = 0; i < F::KM; ++i) d = __builtin_amdgcn_mfma_f64_16x16x4f64(x.k[i], y.k[i], d, 0, 0, 0);
            if constexpr (F::R1) {
#pragma unroll
              for (int i = 0; i < F::ROWS; ++i) d[i] = __builtin_fma(x.last[i], y.last[0], d[i]);
            }
          } else {
            flt4 t = MODE == 1 ? a32[4 * u + k] : flt4{0.f, 0.f, 0.f, 0.f};
            if constexpr (MODE == 4) {
              t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(half_of(x.k, 0), half_of(y.k, 0), t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(half_of(x.k, 0), half_of(y.k, 2), t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(half_of(x.k, 2), half_of(y.k, 0), t, 0, 0, 0);
            } else {
#pragma unroll
              for (int i = 0; i < F::KM; ++i) t = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i], y.k[i], t, 0, 0, 0);
              if constexpr (F::R1) {
#pragma unroll
                for (int i = 0; i < F::ROWS; ++i) t[i] = __builtin_fmaf(x.last[i], y.last[0], t[i]);
              }
            }
            if constexpr (MODE == 1) {
              a32[4 * u + k] = t;
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i) a64[4 * u + k][i] += (double)t[i];
            }
          }
        }
      }
      head = pq;
      held -= n;
      while (fits()) issue();
    } while (nq > 0);
  }
  const int rw = TIGHT ? lane_again() & 15 : r, gw = TIGHT ? lane_again() >> 4 : g;
  auto write = [&](auto *out) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (!(valid >> u & 1u)) continue;
      auto *o = out + (int64_t)out_blk[u] * NS2 + NSF * rw;
#pragma unroll
      for (int i = 0; i < F::ROWS; ++i) {
        const int row = MODE == 0 ? gw + 4 * i : 4 * gw + i;
        if (rw < NSF && row < NSF) o[row] = MODE == 1 ? (T)a32[u][i] : (T)a64[u][i];
      }
    }
  };
  if (MODE != 0 && a.wide) write(static_cast<double *>(a.O));
  else write(static_cast<T *>(a.O));
}

// 4x4 blocks: one wavefront computes 4x4 output blocks (a quadrant of a tile), on
// its own. A record (contraction atom) is eight block indices, four rows and
// four columns, -1 where the block does not exist. One matrix step covers the
// record's whole contraction (4) for all 16 blocks at once: lane (r, g) supplies
// left row r/4, element [r%4][g], and right column r/4, element [g][r%4]. A block pair
// whose output block does not exist only feeds accumulator elements that are
// never written; every output block sums its products in ascending
// contraction atom, one fused step per product, as the triplet kernel does.
//
// A record's blocks are copied memory -> LDS by one instruction (16 bytes a
// lane, absent blocks from a block of zeros), three records ahead. FP64: in LDS
// the halves (type 1 right operands: the 16-byte pairs) of blocks 2 and 3 of
// the rows and of the columns are swapped, so that the operand reads have no
// bank conflict.
//
// What bounds it: a record takes one 72-cycle f64 matrix step and about ten VALU
// instructions, and copies from L2 (13 to 16 TB/s) what its products read: 512
// atoms, 2.0e7 products, 0.21 ms. One workgroup per 8x8 tile with a barrier per
// chunk took 0.80 ms; a list of products per output block with v_mfma_f64_4x4x4
// (four output blocks to a wavefront) 0.45 ms, as it copies 2 blocks per product
// and not the 0.6 to 0.9 of a record. One McWeeny batch of 4 x 64 atoms
// 73.7 -> 26.8 ms.
__device__ __attribute__((aligned(128))) uint32_t g_zero_block[32];

template <int MODE, bool QT, class ARG>
__global__ void __launch_bounds__(64) k_quad4(const ARG arg) {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int BYTES = 16 * (int)sizeof(T), LPB = BYTES / 16, SLOT = 8 * BYTES, AHEAD = 3;
  __shared__ __attribute__((aligned(256))) char lds[(AHEAD + 1) * SLOT];
  TileArgs a;
  const int32_t tile = tile_select(arg, a);
  if (tile < 0) return;
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  dbl4 a64 = {0.0, 0.0, 0.0, 0.0};
  flt4 a32 = {0.f, 0.f, 0.f, 0.f};
  const int64_t w0 = a.pstart[tile];
  const int32_t n = (int32_t)((a.pstart[tile + 1] - w0) >> 3);
  if (n > 0) {
    // Copy lanes: LPB lanes for each of the record's blocks.
    const int blk = lane / LPB, piece = lane % LPB;
    const int swap = MODE == 0 && (blk & 2) ? (blk < 4 || QT ? 4 : 1) : 0;
    const char *base = static_cast<const char *>(blk < 4 ? a.P : a.Q) + 16 * (piece ^ swap);
    const char *zero = (const char *)g_zero_block + 16 * piece;
    auto copy = [&](uint32_t words, int i, int slot) {
      const uint32_t x = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (8 * i + (blk & 7)), (int)words);
      const char *src = x == ~0u ? zero : base + (uint64_t)x * BYTES;
      if (LPB == 8 || lane < 8 * LPB)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                         (__attribute__((address_space(3))) void *)(lds + slot * SLOT), 16, 0, 0);
    };
    // Operand lanes: byte offset of the lane's element in a record's stage.
    const int u = r >> 2, m = r & 3;
    const int fa = BYTES * u + ((int)sizeof(T) * (m + 4 * g) ^ (MODE == 0 && (u & 2) ? 64 : 0));
    const int fb = BYTES * (4 + u) + (QT ? (int)sizeof(T) * (m + 4 * g) ^ (MODE == 0 && (u & 2) ? 64 : 0)
                                         : (int)sizeof(T) * (g + 4 * m) ^ (MODE == 0 && (u & 2) ? 16 : 0));
    // The words of 8 records, one per lane, and of the 8 after them. The copies
    // and words past the quadrant's last record are those of the next quadrant
    // (or the list's 16 records of padding), never used.
    const uint32_t *words = a.prod + w0 + lane;
    uint32_t w = words[0];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) copy(w, i, i);
    for (int32_t rec = 0; rec < n; rec += 8) {
      // The load of wn stays between the copies before it and those after it:
      // the waits below count on that order.
      asm volatile("" ::: "memory");
      const uint32_t wn = words[8 * (int64_t)(rec + 8)];
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (rec + i >= n) break;
        copy(i + AHEAD < 8 ? w : wn, (i + AHEAD) & 7, (i + AHEAD) & 3);
        asm volatile("" ::: "memory");
        // The record's copy is older than AHEAD others and, for the first AHEAD
        // records of the eight, the load of wn.
        if (i < AHEAD) __builtin_amdgcn_s_waitcnt((AHEAD + 1) | 0xf70);
        else __builtin_amdgcn_s_waitcnt(AHEAD | 0xf70);
        asm volatile("" ::: "memory");
        const T x = *(const T *)(lds + (i & 3) * SLOT + fa), y = *(const T *)(lds + (i & 3) * SLOT + fb);
        if constexpr (MODE == 0) {
          a64 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, a64, 0, 0, 0);
        } else if constexpr (MODE == 1) {
          a32 = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, a32, 0, 0, 0);
        } else {
          const flt4 t = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, flt4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) a64[e] += (double)t[e];
        }
      }
      w = wn;
    }
    __builtin_amdgcn_s_waitcnt(0xf70);  // no copy into LDS outlives the wavefront
  }
  // FP64 accumulator D[g+4e][r], FP32 D[4g+e][r]: quadrant row R, column r is
  // element (R % 4, r % 4) of block (R / 4, r / 4).
  const int32_t *wo = a.wave_out + (int64_t)tile * 16;
  // The matrix step also multiplies the zeros of an absent block by the other
  // operand, which is NaN where that is infinite or NaN. A NaN is therefore
  // summed again from the products that exist (no cost without one).
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) nan |= MODE == 1 ? a32[e] != a32[e] : a64[e] != a64[e];
  if (__builtin_expect(__ballot(nan) != 0, 0)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (MODE == 1 ? a32[e] == a32[e] : a64[e] == a64[e]) continue;
      const int rq = MODE == 0 ? e : g, ri = MODE == 0 ? g : e;
      const uint32_t *rec = a.prod + w0;
      double sum = 0.0;
      float sum32 = 0.f;
      for (int32_t i = 0; i < n; ++i, rec += 8) {
        const uint32_t bp = rec[rq], bq = rec[4 + (r >> 2)];
        if (bp == ~0u || bq == ~0u) continue;
        const T *x = static_cast<const T *>(a.P) + (int64_t)bp * 16 + ri;
        const T *y = static_cast<const T *>(a.Q) + (int64_t)bq * 16 + (QT ? r & 3 : 4 * (r & 3));
        float part = MODE == 1 ? sum32 : 0.f;
        for (int k = 0; k < 4; ++k) {
          const T xk = x[4 * k], yk = y[QT ? 4 * k : k];
          if constexpr (MODE == 0) sum = __builtin_fma(xk, yk, sum);
          else part = __builtin_fmaf(xk, yk, part);
        }
        if constexpr (MODE == 1) sum32 = part;
        if constexpr (MODE == 2) sum += (double)part;
      }
      if constexpr (MODE == 1) a32[e] = sum32;
      else a64[e] = sum;
    }
  }
  auto write = [&](auto *out) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int rq = MODE == 0 ? e : g, ri = MODE == 0 ? g : e;
      const int32_t o = wo[rq * 4 + (r >> 2)];
      if (o >= 0) out[(int64_t)o * 16 + ri + 4 * (r & 3)] = MODE == 1 ? (T)a32[e] : (T)a64[e];
    }
  };
  if (MODE != 0 && a.wide) write(static_cast<double *>(a.O));
  else write(static_cast<T *>(a.O));
}

// ---------------------------------------------------------------- builder

inline unsigned grid1(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

__global__ void k_fill_i32(int32_t *__restrict__ v, int64_t n, int32_t val) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) v[t] = val;
}

__global__ void k_chunk_lbeg(const int32_t *__restrict__ chunk_entry, const int64_t *__restrict__ entry_lbeg,
                             int64_t nc1, int64_t *__restrict__ out) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < nc1) out[c] = entry_lbeg[chunk_entry[c]];
}

__global__ void k_iota32(int32_t *__restrict__ v, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) v[t] = (int32_t)t;
}

// Products per output slot of each tile.
__global__ void k_slot_counts(const uint64_t *__restrict__ key, const uint8_t *__restrict__ slot, int64_t n,
                              int64_t nx, int32_t *__restrict__ cnt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) atomicAdd(&cnt[(int64_t)(key[t] / (uint64_t)nx) * 64 + slot[t]], 1);
}

// flag[pos] = 1 where a new (tile, x) key starts in the sorted list.
__global__ void k_entry_flags(const uint64_t *__restrict__ key, int64_t n, int32_t *__restrict__ flag) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) flag[t] = (t == 0 || key[t] != key[t - 1]) ? 1 : 0;
}

// Scatter each product's operand blocks into its entry's row / column slots.
// Products of one entry that share a row (column) write the same block index.
__global__ void k_entry_fill(const uint64_t *__restrict__ key, const int32_t *__restrict__ perm,
                             const int32_t *__restrict__ eid, const uint8_t *__restrict__ slot,
                             const int64_t *__restrict__ p, const int64_t *__restrict__ q, int64_t n, int64_t nx,
                             int64_t ns2, int32_t *__restrict__ ep, int32_t *__restrict__ eq,
                             int32_t *__restrict__ etile) {
  const int64_t pos = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pos >= n) return;
  const int64_t e = (int64_t)eid[pos] - 1;
  const int32_t t = perm[pos];
  const int sl = slot[t];
  ep[e * 8 + (sl >> 3)] = (int32_t)(p[t] / ns2);
  eq[e * 8 + (sl & 7)] = (int32_t)(q[t] / ns2);
  if (pos == 0 || eid[pos - 1] != eid[pos]) etile[e] = (int32_t)(key[pos] / (uint64_t)nx);
}

// tebeg[t] = first entry of tile t (entries are sorted by tile), t = 0..n_tiles.
__global__ void k_tile_ebeg(const int32_t *__restrict__ etile, int64_t ne, int32_t n_tiles,
                            int32_t *__restrict__ tebeg) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > n_tiles) return;
  int64_t lo = 0, hi = ne;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (etile[mid] < t) lo = mid + 1;
    else hi = mid;
  }
  tebeg[t] = (int32_t)lo;
}

// Wavefront products of entry e (tile t): rows u of the entry's left blocks x
// columns of its right blocks whose output block exists (owner != 0xff);
// owner byte = wavefront * kSlots + slot.
__device__ inline void entry_wave_counts(uint32_t m, const uint8_t *__restrict__ own, int pw[kWaves]) {
#pragma unroll
  for (int w = 0; w < kWaves; ++w) pw[w] = 0;
  for (uint32_t ym = m & 0xffu; ym; ym &= ym - 1u) {
    const int u = __builtin_ctz(ym);
    for (uint32_t bm = (m >> 8) & 0xffu; bm; bm &= bm - 1u) {
      const uint8_t o = own[u * 8 + __builtin_ctz(bm)];
      if (o != 0xff) ++pw[o / kSlots];
    }
  }
}

// Tile of each chunk.
__global__ void k_chunk_tile(const int32_t *__restrict__ tchunk, int32_t n_tiles, int32_t *__restrict__ ctile) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tiles) return;
  for (int32_t c = tchunk[t]; c < tchunk[t + 1]; ++c) ctile[c] = t;
}

// Where each 64th of the work begins, of n launch units with the work w[at[t]]
// before unit t (at null: w[t]); out[64] = n, then the work of all.
template <class W>
__global__ void k_work_parts(const W *__restrict__ w, const int32_t *__restrict__ at, int32_t n,
                             int64_t *__restrict__ out) {
  const int k = threadIdx.x;
  if (k > cq::kWorkParts) return;
  auto before = [&](int32_t t) { return (int64_t)w[at ? at[t] : t]; };
  const int64_t all = before(n);
  const int64_t want = all / cq::kWorkParts * k + all % cq::kWorkParts * k / cq::kWorkParts;
  int32_t lo = 0, hi = n;
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if (before(mid) < want) lo = mid + 1;
    else hi = mid;
  }
  out[k] = k == cq::kWorkParts ? n : lo;
  if (k == 0) out[cq::kWorkParts + 1] = all;
}

// Records of the quadrant kernels, one wavefront per quadrant q (src[q] =
// tile * 4 + quadrant): of the tile's entries (ascending contraction atom) those
// with a product in the quadrant. k_wave_products (QUAD4 unset): rows and
// columns that have one, then their block indices. k_quad4: eight block indices,
// -1 for the rows and columns without. Count pass (FILL unset): words, products
// and blocks of each quadrant.
template <bool FILL, bool QUAD4>
__global__ void __launch_bounds__(256) k_wave_records(
    const int32_t *__restrict__ src, int32_t n_wave, const int32_t *__restrict__ wave_out,
    const int32_t *__restrict__ tebeg, const int32_t *__restrict__ ep, const int32_t *__restrict__ eq,
    int64_t *__restrict__ nword, int64_t *__restrict__ nprod, int64_t *__restrict__ nload,
    const int64_t *__restrict__ beg, uint32_t *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int32_t q = (int32_t)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
  if (q >= n_wave) return;
  const int32_t t = src[q] >> 2, w = src[q] & 3;
  const int qr = 4 * (w >> 1), qc = 4 * (w & 1);
  const uint32_t valid = (uint32_t)__ballot(wave_out[(int64_t)q * 16 + (lane & 15)] >= 0) & 0xffffu;
  int64_t at = FILL ? beg[q] : 0;
  int64_t prods = 0, loads = 0;
  for (int32_t e0 = tebeg[t]; e0 < tebeg[t + 1]; e0 += 64) {
    const int32_t e = e0 + lane;
    int32_t b[8];
    uint32_t rows = 0, cols = 0;
    int np = 0;
    if (e < tebeg[t + 1]) {
      uint32_t pm = 0, qm = 0;
      for (int k = 0; k < 4; ++k) {
        b[k] = ep[(int64_t)e * 8 + qr + k];
        b[4 + k] = eq[(int64_t)e * 8 + qc + k];
        pm |= (uint32_t)(b[k] >= 0) << k;
        qm |= (uint32_t)(b[4 + k] >= 0) << k;
      }
      for (int k = 0; k < 4; ++k) {
        const uint32_t c = (pm >> k & 1u) ? (valid >> (4 * k)) & qm : 0u;
        np += __popc(c);
        cols |= c;
        rows |= (uint32_t)(c != 0) << k;
      }
    }
    const int nb = __popc(rows) + __popc(cols), len = rows == 0 ? 0 : QUAD4 ? 8 : 1 + nb;
    int before = len;  // inclusive prefix sum of the records' words over the lanes
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(before, off, 64);
      if (lane >= off) before += v;
    }
    if (FILL && rows != 0) {
      int64_t o = at + before - len;
      const uint32_t here = rows | cols << 4;
      if (!QUAD4) out[o++] = here;
      for (int k = 0; k < 8; ++k) {
        if (here >> k & 1u) out[o++] = (uint32_t)b[k];
        else if (QUAD4) out[o++] = ~0u;
      }
    }
    at += __shfl(before, 63, 64);
    prods += np;
    loads += nb;
  }
  if (!FILL) {
    for (int off = 32; off > 0; off >>= 1) {
      prods += __shfl_down(prods, off, 64);
      loads += __shfl_down(loads, off, 64);
    }
    if (lane == 0) {
      nword[q] = at;
      nprod[q] = prods;
      nload[q] = loads;
    }
  }
}

template <class T>
int inclusive_scan(const T *in, T *out, size_t n, hipStream_t s) {
  if (n == 0) return CQMM_OK;
  size_t bytes = 0;
  hipError_t e = rocprim::inclusive_scan(nullptr, bytes, in, out, n, rocprim::plus<T>(), s);
  if (e != hipSuccess) return cq::hip_check(e, "inclusive_scan (size)");
  cq::DevBuf tmp;
  int st = tmp.alloc(bytes);
  if (st) return st;
  e = rocprim::inclusive_scan(tmp.p, bytes, in, out, n, rocprim::plus<T>(), s);
  if (e != hipSuccess) return cq::hip_check(e, "inclusive_scan");
  // tmp is freed on return: wait for the scan that uses it.
  return cq::hip_check(hipStreamSynchronize(s), "inclusive_scan");
}

// Kernel family of a tile schedule: schedules of one family (with the same
// precision mode and operand transposition) can share a grouped launch.
enum TileKind {
  kKindDense4 = 1,
  kKindDenseMx = 2,
  kKindMixedSmall = 3,
  kKindMixedLarge = 4,
  kKindQuadSmall = 5,
  kKindQuadLarge = 6,
  kKindUniform = 16
};
int tile_kind(const cq::TilePlan &tp);

// ------------------------------------------------ mixed block sizes
// Same schedule with per-atom block dimensions (up to 16): operands are
// addressed by element offset and packed in LDS by size; each product word
// carries its contraction dimension; the k-steps of a product (1-4) and the
// lane offsets follow the dimensions of its blocks.

// Operand elements a chunk stage holds: STG_SMALL for blocks up to 13x13
// (three workgroups per CU), STG_LARGE up to 16x16 (an entry brings at most
// 16 blocks, so it always fits).
constexpr int kStgSmall = 3072;
constexpr int kStgLarge = 4096;
int stage_elems(int maxn) { return maxn <= 13 ? kStgSmall : kStgLarge; }

__global__ void k_entry_fill_mx(const uint64_t *__restrict__ key, const int32_t *__restrict__ perm,
                                const int32_t *__restrict__ eid, const uint8_t *__restrict__ slot,
                                const int64_t *__restrict__ p, const int64_t *__restrict__ q, int64_t n, int64_t nx,
                                int64_t *__restrict__ ep, int64_t *__restrict__ eq, int32_t *__restrict__ etile,
                                int32_t *__restrict__ ex) {
  const int64_t pos = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pos >= n) return;
  const int64_t e = (int64_t)eid[pos] - 1;
  const int32_t t = perm[pos];
  const int sl = slot[t];
  ep[e * 8 + (sl >> 3)] = p[t];
  eq[e * 8 + (sl & 7)] = q[t];
  if (pos == 0 || eid[pos - 1] != eid[pos]) {
    etile[e] = (int32_t)(key[pos] / (uint64_t)nx);
    ex[e] = (int32_t)(key[pos] % (uint64_t)nx);
  }
}

// Mask (left rows | right columns << 8 | (contraction dimension - 1) << 16),
// operand elements and operand count of each entry.
__global__ void k_entry_mask_mx(const int64_t *__restrict__ ep, const int64_t *__restrict__ eq,
                                const int32_t *__restrict__ etile, const int32_t *__restrict__ ex,
                                const uint8_t *__restrict__ rdim, const uint8_t *__restrict__ cdim,
                                const uint8_t *__restrict__ xdim, int64_t ne, uint32_t *__restrict__ mask,
                                int32_t *__restrict__ esz, int64_t *__restrict__ cnt) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  const int64_t t = etile[e];
  const int32_t nxd = xdim[ex[e]];
  uint32_t m = 0;
  int32_t sz = 0;
  for (int u = 0; u < 8; ++u) {
    if (ep[e * 8 + u] >= 0) {
      m |= 1u << u;
      sz += rdim[t * 8 + u] * nxd;
    }
    if (eq[e * 8 + u] >= 0) {
      m |= 1u << (8 + u);
      sz += nxd * cdim[t * 8 + u];
    }
  }
  mask[e] = m | (uint32_t)(nxd - 1) << 16;  // contraction dimension in bits 16-19
  esz[e] = sz;
  cnt[e] = __popc(m);
}

// Operand list of each entry (left blocks by row, then right blocks by
// column): element offsets (bit 63: right operand) and element counts.
__global__ void k_list_fill_mx(const int64_t *__restrict__ ep, const int64_t *__restrict__ eq,
                               const int32_t *__restrict__ etile, const int32_t *__restrict__ ex,
                               const uint8_t *__restrict__ rdim, const uint8_t *__restrict__ cdim,
                               const uint8_t *__restrict__ xdim, const int64_t *__restrict__ lbeg, int64_t ne,
                               uint64_t *__restrict__ list, uint16_t *__restrict__ lsz) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  const int64_t t = etile[e];
  const int32_t nxd = xdim[ex[e]];
  int64_t o = lbeg[e];
  for (int u = 0; u < 8; ++u)
    if (ep[e * 8 + u] >= 0) {
      list[o] = (uint64_t)ep[e * 8 + u];
      lsz[o++] = (uint16_t)(rdim[t * 8 + u] * nxd);
    }
  for (int u = 0; u < 8; ++u)
    if (eq[e * 8 + u] >= 0) {
      list[o] = (uint64_t)eq[e * 8 + u] | (1ull << 63);
      lsz[o++] = (uint16_t)(nxd * cdim[t * 8 + u]);
    }
}

// Chunks of a tile by operand elements (at most cap), entries, operand
// blocks (at most kWaves * 64) and products per wavefront (kWaveProducts). Count
// pass (FILL unset): chunks of each tile. Fill pass: each chunk's first entry.
template <bool FILL>
__global__ void k_chunks_mx(const int32_t *__restrict__ tebeg, const uint32_t *__restrict__ mask,
                            const int32_t *__restrict__ esz, const uint8_t *__restrict__ owner, int32_t n_tiles,
                            int32_t cap, int32_t max_entries, const int32_t *__restrict__ tchunk,
                            int32_t *__restrict__ out) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tiles) return;
  int32_t nch = 0, sum = 0, ne = 0, nb = 0;
  int wc[kWaves] = {};
  for (int32_t e = tebeg[t]; e < tebeg[t + 1]; ++e) {
    const uint32_t m = mask[e];
    const int32_t c = esz[e];
    const int32_t b = __popc(m & 0xffffu);
    int pw[kWaves] = {};
    if (owner) entry_wave_counts(m, owner + (int64_t)t * 64, pw);  // no owner: no per-wavefront limit
    bool over = false;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) over |= wc[w] + pw[w] > kWaveProducts;
    // A chunk's operand blocks are spread over the lanes of the wavefronts'
    // operand lists: at most kWaves * 64 of them.
    if (nch == 0 || sum + c > cap || ne == max_entries || nb + b > kWaves * 64 || over) {
      if (FILL) out[tchunk[t] + nch] = e;
      ++nch;
      sum = 0;
      ne = 0;
      nb = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) wc[w] = 0;
    }
    sum += c;
    nb += b;
    ++ne;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) wc[w] += pw[w];
  }
  if (!FILL) out[t] = nch;
}

// First LDS element of each entry in its chunk's stage.
__global__ void k_entry_coff_mx(const int32_t *__restrict__ chunk_entry, const int32_t *__restrict__ esz, int64_t nc,
                                int32_t *__restrict__ coff) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  int32_t run = 0;
  for (int32_t e = chunk_entry[c]; e < chunk_entry[c + 1]; ++e) {
    coff[e] = run;
    run += esz[e];
  }
}

// LDS element offset | elements << 16 of each operand of each chunk.
__global__ void k_list_lds_mx(const int64_t *__restrict__ chunk_lbeg, const uint16_t *__restrict__ lsz, int64_t nc,
                              uint32_t *__restrict__ listls) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  uint32_t run = 0;
  for (int64_t o = chunk_lbeg[c]; o < chunk_lbeg[c + 1]; ++o) {
    listls[o] = run | ((uint32_t)lsz[o] << 16);
    run += lsz[o];
  }
}

// Work of a chunk in the mixed-size kernel for the split over the XCDs, in parts of
// a k-step: three per product beside its k-steps, 100 for the chunk (its barrier and
// copies). With products alone the 4096-atom 4/9/13 mix takes 27.0 to 27.2 ms, so 26.8.
constexpr int kWorkProduct = 3, kWorkChunk = 100;

// Product lists of each chunk, sorted by (wavefront, slot, entry). Count pass (FILL
// unset): products per chunk into np, its work into `work`. Fill pass, with pbase = the chunk's first
// product: pstart and pcnt of its wavefronts, and the product words. Word = left
// LDS offset | right LDS offset << 12 | (contraction dimension nx - 1) << 24 | (k-steps - 1) << 28 |
// (contraction indices of the last k-step - 1) << 30.
template <bool FILL>
__global__ void k_chunk_prods_mx(int32_t nch, const int32_t *__restrict__ chunk_entry,
                                 const int32_t *__restrict__ ctile, const uint32_t *__restrict__ mask,
                                 const int32_t *__restrict__ coff, const int32_t *__restrict__ ex,
                                 const uint8_t *__restrict__ owner, const uint8_t *__restrict__ rdim,
                                 const uint8_t *__restrict__ cdim, const uint8_t *__restrict__ xdim,
                                 int64_t *__restrict__ np, int64_t *__restrict__ work,
                                 const int64_t *__restrict__ pbase, int64_t *__restrict__ pstart,
                                 uint64_t *__restrict__ pcnt, uint32_t *__restrict__ prod) {
  const int32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nch) return;
  const int64_t t = ctile[c];
  const uint8_t *own = owner + t * 64;
  const int32_t e0 = chunk_entry[c], e1 = chunk_entry[c + 1];
  uint8_t cnt[64];
  for (int i = 0; i < 64; ++i) cnt[i] = 0;
  int32_t tot = 0, steps = 0;
  for (int32_t e = e0; e < e1; ++e) {
    const uint32_t m = mask[e];
    const int32_t before = tot;
    for (uint32_t ym = m & 0xffu; ym; ym &= ym - 1u) {
      const int u = __builtin_ctz(ym);
      for (uint32_t bm = (m >> 8) & 0xffu; bm; bm &= bm - 1u) {
        const uint8_t o = own[u * 8 + __builtin_ctz(bm)];
        if (o != 0xff) {
          ++cnt[o];
          ++tot;
        }
      }
    }
    steps += (tot - before) * ((xdim[ex[e]] + 3) >> 2);
  }
  if (!FILL) {
    np[c] = tot;
    work[c] = kWorkProduct * tot + steps + kWorkChunk;
    return;
  }
  uint16_t off[64];
  int32_t run = 0;
  for (int w = 0; w < kWaves; ++w) {
    pstart[(int64_t)c * kWaves + w] = pbase[c] + run;
    uint64_t word = 0;
    for (int l = 0; l < kSlots; ++l) {
      off[w * kSlots + l] = (uint16_t)run;
      run += cnt[w * kSlots + l];
      word |= (uint64_t)cnt[w * kSlots + l] << (4 * l);
    }
    pcnt[(int64_t)c * kWaves + w] = word;
  }
  for (int32_t e = e0; e < e1; ++e) {
    const uint32_t m = mask[e];
    const uint32_t ym = m & 0xffu, bmask = (m >> 8) & 0xffu;
    const uint32_t nxd = xdim[ex[e]];
    uint32_t rows = 0;  // left elements of the entry
    for (uint32_t yb = ym; yb; yb &= yb - 1u) rows += rdim[t * 8 + __builtin_ctz(yb)] * nxd;
    uint32_t aoff = (uint32_t)coff[e];
    for (uint32_t yb = ym; yb; yb &= yb - 1u) {
      const int u = __builtin_ctz(yb);
      uint32_t boff = (uint32_t)coff[e] + rows;
      for (uint32_t bm = bmask; bm; bm &= bm - 1u) {
        const int col = __builtin_ctz(bm);
        const uint8_t o = own[u * 8 + col];
        if (o != 0xff) {
          const uint32_t ks = (nxd + 3u) >> 2, rem = nxd - 4u * (ks - 1u);
          prod[pbase[c] + off[o]++] = aoff | (boff << 12) | ((nxd - 1u) << 24) | ((ks - 1u) << 28) | ((rem - 1u) << 30);
        }
        boff += nxd * cdim[t * 8 + col];
      }
      aoff += rdim[t * 8 + u] * nxd;
    }
  }
}

// Copies of one operand block (up to 16x16) with one M0: pieces I < NP of
// 256 bytes, the last masked to the block's dwords.
template <int... I>
__device__ inline void dma_block_pieces(const uint32_t *src, uint32_t *dst, int dwords, int lane,
                                        std::integer_sequence<int, I...>) {
  ((I * 64 < dwords ? (I * 64 + lane < dwords ? (dma_piece<I * 256>(src, dst), 0) : 0) : 0), ...);
}

template <class T>
__device__ inline void issue_stage_mx(uint64_t lv, uint32_t lls, int32_t nb, const T *__restrict__ P,
                                      const T *__restrict__ Q, T *stage, int w, int lane) {
  constexpr int MAXP = 256 * (int)sizeof(T) / 4 / 64;  // pieces of a 16x16 block
  const int32_t nbw = nb > w ? (nb - w + kWaves - 1) / kWaves : 0;
  for (int32_t k = 0; k < nbw; ++k) {
    const uint64_t g = (uint64_t)readlane64((int64_t)lv, k);
    const uint32_t ls = (uint32_t)__builtin_amdgcn_readlane((int)lls, k);
    const T *base = (g >> 63) ? Q : P;
    const uint32_t *src = (const uint32_t *)(base + (int64_t)(g & 0x7fffffffffffffffull)) + lane;
    uint32_t *dst = (uint32_t *)(stage + (ls & 0xffffu));
    const int dwords = (int)(ls >> 16) * (int)sizeof(T) / 4;
    dma_block_pieces(src, dst, dwords, lane, std::make_integer_sequence<int, MAXP>{});
  }
}

// Mixed-size tile kernel: per-slot output dimensions (wave_dim) and per-product
// contraction dimension (product word bits 24-27). Pipeline per chunk c (one
// barrier): wait for chunk c's copies and the prefetched registers, issue chunk
// c+1's copies into the other stage and the register loads of chunk c+1's
// product list and chunk c+2's operand list, then compute chunk c from LDS.
template <int MODE, bool QT, int STG, class ARG>
__global__ void __launch_bounds__(kTileThreads) k_tile_mixed(
    const ARG arg) {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int STAGE = STG + kLdsPad * (int)(8 / sizeof(T));
  __shared__ T stage0[STAGE];
  __shared__ T stage1[STAGE];
  TileArgs a;
  const int32_t tile = tile_select(arg, a);
  if (tile < 0) return;  // the whole workgroup leaves together
  const int32_t *__restrict__ tile_chunk = a.tile_chunk;
  const int64_t *__restrict__ chunk_lbeg = a.chunk_lbeg;
  const uint64_t *__restrict__ list64 = a.list64;
  const uint32_t *__restrict__ listls = a.listls;
  const int64_t *__restrict__ pstart = a.pstart;
  const uint64_t *__restrict__ pcnt = a.pcnt;
  const uint32_t *__restrict__ prod = a.prod;
  const int64_t *__restrict__ wave_out = a.wave_out64;
  const uint8_t *__restrict__ wave_dim = a.wave_dim;
  const T *__restrict__ P = static_cast<const T *>(a.P);
  const T *__restrict__ Q = static_cast<const T *>(a.Q);
  T *__restrict__ O = static_cast<T *>(a.O);
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int64_t wbase = ((int64_t)tile * kWaves + w) * kSlots;
  int64_t oblk[kSlots];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) oblk[u] = wave_out[wbase + u];
  const uint32_t *wd32 = (const uint32_t *)(wave_dim + wbase);
  uint32_t wdim[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) wdim[k] = wd32[k];
  dbl4 a64[kSlots];
  flt4 a32[kSlots];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) {
    a64[u] = dbl4{0.0, 0.0, 0.0, 0.0};
    a32[u] = flt4{0.f, 0.f, 0.f, 0.f};
  }
  const int32_t c0 = tile_chunk[tile], c1 = tile_chunk[tile + 1];
  if (c0 < c1) {
    int32_t wb = c0;
    int32_t cc = min(wb + lane, c1);
    int64_t wcl = chunk_lbeg[cc];
    int64_t wps = pstart[(int64_t)cc * kWaves + w];
    int64_t wpc = (int64_t)pcnt[(int64_t)cc * kWaves + w];
    auto cl_at = [&](int32_t x) { return readlane64(wcl, min(x, c1) - wb); };
    auto ps_at = [&](int32_t x) { return readlane64(wps, min(x, c1) - wb); };
    auto pc_at = [&](int32_t x) { return (uint64_t)readlane64(wpc, min(x, c1) - wb); };
    auto list_idx = [&](int64_t lbeg, int32_t nb) { return lbeg + min(w + kWaves * lane, nb - 1); };
    uint32_t pl;
    uint64_t lvn = 0;
    uint32_t lsn = 0;
    {
      const int64_t cl0 = cl_at(c0), cl1 = cl_at(c0 + 1);
      const int64_t i0 = list_idx(cl0, (int32_t)(cl1 - cl0));
      const uint64_t lv0 = list64[i0];
      const uint32_t ls0 = listls[i0];
      issue_stage_mx<T>(lv0, ls0, (int32_t)(cl1 - cl0), P, Q, stage0, w, lane);
      pl = prod[ps_at(c0) + lane];
      if (c0 + 1 < c1) {
        const int64_t i1 = list_idx(cl1, (int32_t)(cl_at(c0 + 2) - cl1));
        lvn = list64[i1];
        lsn = listls[i1];
      }
    }
    for (int32_t c = c0; c < c1; ++c) {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      const bool odd = ((c - c0) & 1) != 0;
      const T *cur = odd ? stage1 : stage0;
      const uint32_t plc = pl;
      const uint64_t cnt = pc_at(c);
      if (c + 1 < c1) {
        const int64_t cl1 = cl_at(c + 1), cl2 = cl_at(c + 2);
        issue_stage_mx<T>(lvn, lsn, (int32_t)(cl2 - cl1), P, Q, odd ? stage0 : stage1, w, lane);
        pl = prod[ps_at(c + 1) + lane];
        if (c + 2 < c1) {
          const int64_t i2 = list_idx(cl2, (int32_t)(cl_at(c + 3) - cl2));
          lvn = list64[i2];
          lsn = listls[i2];
        }
      }
      // Lane coordinates made opaque per chunk, so the per-slot lane offsets
      // below are computed where used instead of being kept for all 16 slots
      // across the chunk loop (which costs 32 registers).
      int lr = r, lg = g;
      asm volatile("" : "+v"(lr), "+v"(lg));
      int p = 0;
#pragma unroll
      for (int u = 0; u < kSlots; ++u) {
        const int n = (int)((cnt >> (4 * u)) & 15u);
        if (n == 0) continue;
        const uint32_t dm = (wdim[u >> 2] >> (8 * (u & 3))) & 0xffu;
        const int nrow = (int)(dm & 15u) + 1, ncol = (int)(dm >> 4) + 1;
        // Lanes past the block's rows (left) or columns (right) read the last
        // valid row/column (a broadcast, no bank conflicts); they feed only
        // accumulator rows/columns that are never written.
        const int rA = min(lr, nrow - 1), rB = min(lr, ncol - 1);
        const int oA = rA + nrow * lg, SA = 4 * nrow;
        for (int i = 0; i < n; ++i, ++p) {
          const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)plc, p);
          const int nx = (int)((v >> 24) & 15u) + 1;
          const int ks1 = (int)((v >> 28) & 3u), rem = (int)(v >> 30) + 1;
          const T *la = cur + (int)(v & 0xfffu) + oA;
          const T *lq = cur + (int)((v >> 12) & 0xfffu) + (QT ? rB + ncol * lg : lg + nx * rB);
          const int SB = QT ? 4 * ncol : 4;
          flt4 t = {0.f, 0.f, 0.f, 0.f};
          // Full k-steps, then the last one (contraction indices >= nx zeroed).
#pragma unroll
          for (int s4 = 0; s4 < 3; ++s4) {
            if (s4 < ks1) {
              const T a = la[SA * s4], bb = lq[SB * s4];
              if constexpr (MODE == 0) a64[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bb, a64[u], 0, 0, 0);
              else if constexpr (MODE == 1) a32[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bb, a32[u], 0, 0, 0);
              else t = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bb, t, 0, 0, 0);
            }
          }
          {
            T a = la[SA * ks1], bb = lq[SB * ks1];
            if (lg >= rem) {
              a = (T)0;
              bb = (T)0;
            }
            if constexpr (MODE == 0) a64[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bb, a64[u], 0, 0, 0);
            else if constexpr (MODE == 1) a32[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bb, a32[u], 0, 0, 0);
            else t = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bb, t, 0, 0, 0);
          }
          if constexpr (MODE == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) a64[u][e] += (double)t[e];
          }
        }
      }
      if (c + 4 > wb + 63 && c + 1 < c1) {
        wb = c + 1;
        cc = min(wb + lane, c1);
        wcl = chunk_lbeg[cc];
        wps = pstart[(int64_t)cc * kWaves + w];
        wpc = (int64_t)pcnt[(int64_t)cc * kWaves + w];
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kSlots; ++u) {
    if (oblk[u] < 0) continue;
    const uint32_t dm = (wdim[u >> 2] >> (8 * (u & 3))) & 0xffu;
    const int nrow = (int)(dm & 15u) + 1, ncol = (int)(dm >> 4) + 1;
    if (r >= ncol) continue;
    T *o = O + oblk[u];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = MODE == 0 ? g + 4 * e : 4 * g + e;
      if (row < nrow) o[row + nrow * r] = MODE == 0 ? (T)a64[u][e] : (MODE == 1 ? (T)a32[u][e] : (T)a64[u][e]);
    }
  }
}

// Mixed block sizes of at most 4x4 (e.g. C and H with single-zeta bases):
// the dense-quadrant scheme of one matrix step per entry over the mixed-size schedule.
// Wavefront w owns quadrant (w / 2, w % 2) of the tile (4x4 blocks, each
// inside a 4x4 corner of the quadrant's 16x16 MFMA tile) and issues one
// 16x16x4 MFMA per entry: lane (r, g) supplies element (r % 4, g) of
// P(row 4*(w/2) + r/4, x) and element (g, r % 4) of Q(column 4*(w%2) + r/4, x),
// zero outside the blocks' shapes or where the entry lacks the block. A
// block's LDS offset within its entry is the entry offset plus nx times the
// rows (columns) of the entry's blocks before it, summed from the tile's
// block-shape bit masks with three popcounts.
template <int MODE, bool QT, class ARG>
__global__ void __launch_bounds__(kTileThreads) k_tile_dense_mx(
    const ARG arg) {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int STAGE = kStgSmall + kLdsPad * (int)(8 / sizeof(T));
  __shared__ T stage0[STAGE];
  __shared__ T stage1[STAGE];
  TileArgs a;
  const int32_t tile = tile_select(arg, a);
  if (tile < 0) return;  // the whole workgroup leaves together
  const int32_t *__restrict__ tile_chunk = a.tile_chunk;
  const int64_t *__restrict__ chunk_lbeg = a.chunk_lbeg;
  const uint64_t *__restrict__ list64 = a.list64;
  const uint32_t *__restrict__ listls = a.listls;
  const int32_t *__restrict__ chunk_entry = a.chunk_entry;
  const uint32_t *__restrict__ emask = a.emask;
  const int32_t *__restrict__ ecoff = a.ecoff;
  const uint8_t *__restrict__ rdim = a.rdim;
  const uint8_t *__restrict__ cdim = a.cdim;
  const int64_t *__restrict__ wave_out = a.wave_out64;
  const T *__restrict__ P = static_cast<const T *>(a.P);
  const T *__restrict__ Q = static_cast<const T *>(a.Q);
  T *__restrict__ O = static_cast<T *>(a.O);
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, r = lane & 15, g = lane >> 4, rr = r & 3;
  const int qr = w >> 1, qc = w & 1;
  const int ua = 4 * qr + (r >> 2), cb = 4 * qc + (r >> 2);
  // Block shapes of the tile: this lane's row and column, and bit masks of the
  // rows (columns) whose size has bit 0, 1 or 2 set.
  const int rd = rdim[(int64_t)tile * 8 + ua], cd = cdim[(int64_t)tile * 8 + cb];
  uint32_t rb0 = 0, rb1 = 0, rb2 = 0, cb0 = 0, cb1 = 0, cb2 = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t a = rdim[(int64_t)tile * 8 + k], c = cdim[(int64_t)tile * 8 + k];
    rb0 |= (a & 1u) << k;
    rb1 |= ((a >> 1) & 1u) << k;
    rb2 |= ((a >> 2) & 1u) << k;
    cb0 |= (c & 1u) << k;
    cb1 |= ((c >> 1) & 1u) << k;
    cb2 |= ((c >> 2) & 1u) << k;
  }
  auto rows_of = [&](uint32_t m) { return __popc(m & rb0) + 2 * __popc(m & rb1) + 4 * __popc(m & rb2); };
  auto cols_of = [&](uint32_t m) { return __popc(m & cb0) + 2 * __popc(m & cb1) + 4 * __popc(m & cb2); };
  const uint32_t below_a = (1u << ua) - 1u, below_b = (1u << cb) - 1u;
  const uint32_t quad_rows = 0xfu << (4 * qr), quad_cols = 0xfu << (8 + 4 * qc);
  dbl4 a64 = {0.0, 0.0, 0.0, 0.0};
  flt4 a32 = {0.f, 0.f, 0.f, 0.f};
  const int32_t c0 = tile_chunk[tile], c1 = tile_chunk[tile + 1];
  if (c0 < c1) {
    int32_t wb = c0;
    int32_t cc = min(wb + lane, c1);
    int64_t wcl = chunk_lbeg[cc];
    int32_t wce = chunk_entry[cc];
    auto cl_at = [&](int32_t x) { return readlane64(wcl, min(x, c1) - wb); };
    auto ce_at = [&](int32_t x) { return __builtin_amdgcn_readlane(wce, min(x, c1) - wb); };
    auto list_idx = [&](int64_t lbeg, int32_t nb) { return lbeg + min(w + kWaves * lane, nb - 1); };
    auto entry_regs = [&](int32_t e0, int32_t e1, uint32_t &m, int32_t &o) {
      const int32_t e = min(e0 + lane, e1 - 1);
      m = emask[e];
      o = ecoff[e];
    };
    uint32_t em, emn = 0;
    int32_t eo, eon = 0;
    uint64_t lvn = 0;
    uint32_t lsn = 0;
    {
      const int64_t cl0 = cl_at(c0), cl1 = cl_at(c0 + 1);
      const int64_t i0 = list_idx(cl0, (int32_t)(cl1 - cl0));
      issue_stage_mx<T>(list64[i0], listls[i0], (int32_t)(cl1 - cl0), P, Q, stage0, w, lane);
      entry_regs(ce_at(c0), ce_at(c0 + 1), emn, eon);
      if (c0 + 1 < c1) {
        const int64_t i1 = list_idx(cl1, (int32_t)(cl_at(c0 + 2) - cl1));
        lvn = list64[i1];
        lsn = listls[i1];
      }
    }
    for (int32_t c = c0; c < c1; ++c) {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      const bool odd = ((c - c0) & 1) != 0;
      const T *cur = odd ? stage1 : stage0;
      em = emn;
      eo = eon;
      const int32_t ne = ce_at(c + 1) - ce_at(c);
      if (c + 1 < c1) {
        const int64_t cl1 = cl_at(c + 1), cl2 = cl_at(c + 2);
        issue_stage_mx<T>(lvn, lsn, (int32_t)(cl2 - cl1), P, Q, odd ? stage0 : stage1, w, lane);
        entry_regs(ce_at(c + 1), ce_at(c + 2), emn, eon);
        if (c + 2 < c1) {
          const int64_t i2 = list_idx(cl2, (int32_t)(cl_at(c + 3) - cl2));
          lvn = list64[i2];
          lsn = listls[i2];
        }
      }
      for (int i = 0; i < ne; ++i) {
        const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)em, i);
        if ((m & quad_rows) == 0 || (m & quad_cols) == 0) continue;  // no block pair in this quadrant
        const int32_t base = __builtin_amdgcn_readlane(eo, i);
        const uint32_t ym = m & 0xffu, bm = (m >> 8) & 0xffu;
        const int nx = (int)((m >> 16) & 15u) + 1;
        const bool va = ((ym >> ua) & 1u) != 0 && rr < rd && g < nx;
        const bool vb = ((bm >> cb) & 1u) != 0 && rr < cd && g < nx;
        const int pa = base + nx * rows_of(ym & below_a);
        const int pb = base + nx * (rows_of(ym) + cols_of(bm & below_b));
        const int ia = va ? pa + rr + rd * g : 0;
        const int ib = vb ? (QT ? pb + rr + cd * g : pb + g + nx * rr) : 0;
        T a = cur[ia], b = cur[ib];
        if (!va) a = (T)0;
        if (!vb) b = (T)0;
        if constexpr (MODE == 0) {
          a64 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, a64, 0, 0, 0);
        } else if constexpr (MODE == 1) {
          a32 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, a32, 0, 0, 0);
        } else {
          const flt4 t = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, flt4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) a64[e] += (double)t[e];
        }
      }
      if (c + 4 > wb + 63 && c + 1 < c1) {
        wb = c + 1;
        cc = min(wb + lane, c1);
        wcl = chunk_lbeg[cc];
        wce = chunk_entry[cc];
      }
    }
  }
  // Quadrant row R, column r: element (R % 4, r % 4) of block (R / 4, r / 4);
  // written where it lies inside that block's shape.
  const int64_t *wo = wave_out + ((int64_t)tile * kWaves + w) * 16;
  // As in k_quad4, a NaN is summed again from the products that exist.
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) nan |= MODE == 1 ? a32[e] != a32[e] : a64[e] != a64[e];
  if (__builtin_expect(__ballot(nan) != 0, 0)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (MODE == 1 ? a32[e] == a32[e] : a64[e] == a64[e]) continue;
      const int u = 4 * qr + (MODE == 0 ? e : g), ri = MODE == 0 ? g : e;
      const int nr = rdim[(int64_t)tile * 8 + u];
      if (ri >= nr || rr >= cd) continue;
      double sum = 0.0;
      float sum32 = 0.f;
      int64_t at = chunk_lbeg[c0];
      for (int32_t i = chunk_entry[c0]; i < chunk_entry[c1]; ++i) {
        const uint32_t m = emask[i], ym = m & 0xffu, bm = (m >> 8) & 0xffu;
        if ((ym >> u & 1u) && (bm >> cb & 1u)) {
          const int nx = (int)((m >> 16) & 15u) + 1;
          const T *x = P + list64[at + __popc(ym & ((1u << u) - 1u))] + ri;
          const T *y = Q + (list64[at + __popc(ym) + __popc(bm & below_b)] & ~(1ull << 63)) + (QT ? rr : nx * rr);
          float part = MODE == 1 ? sum32 : 0.f;
          for (int k = 0; k < nx; ++k) {
            const T xk = x[nr * k], yk = y[QT ? cd * k : k];
            if constexpr (MODE == 0) sum = __builtin_fma(xk, yk, sum);
            else part = __builtin_fmaf(xk, yk, part);
          }
          if constexpr (MODE == 1) sum32 = part;
          if constexpr (MODE == 2) sum += (double)part;
        }
        at += __popc(m & 0xffffu);
      }
      if constexpr (MODE == 1) a32[e] = sum32;
      else a64[e] = sum;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int rq = MODE == 0 ? e : g, ri = MODE == 0 ? g : e;
    const int64_t off = wo[rq * 4 + (r >> 2)];
    const int nr = rdim[(int64_t)tile * 8 + 4 * qr + rq];
    if (off >= 0 && ri < nr && rr < cd) O[off + ri + nr * rr] = MODE == 1 ? (T)a32[e] : (T)a64[e];
  }
}

// Class tiles (species mixes, blocks up to 16x16): the tile's rows all have
// one block size NI and its columns one size NJ (the plan groups tile rows
// and columns by species), so the tile's blocks pack into 16x16-element MFMA
// tiles of RP row blocks x CP column blocks (RP = 4, 2, 1 for NI <= 4, <= 8,
// <= 16; CP likewise): sixteen 4x4 block pairs share one MFMA, four 4x13
// pairs, one 13x13 pair. Wavefront w owns quadrant (w / 2, w % 2) of the tile
// (4 block rows x 4 block columns, 16 / (RP CP) MFMA tiles). Per chunk entry
// (contraction atom x with nx contraction indices; at most 64 entries per
// chunk, one per lane) and k-step of 4 indices, each lane reads one element
// of each of the wavefront's row units and column units from LDS (its block's
// offset from the entry's offset and the popcount of the entry's blocks
// before it) and every MFMA tile with a block pair present accumulates;
// absent blocks, rows or columns past NI / NJ and indices past nx read as
// zero. Each output block sums its products in entry (x) order. The entry
// list replaces per-product lists: no product decode at run time.
template <int MODE, bool QT>
__device__ __forceinline__ void quad_tile(const TileArgs &a, const int32_t tile,
                                          typename std::conditional<MODE == 0, double, float>::type *stage0,
                                          typename std::conditional<MODE == 0, double, float>::type *stage1) {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  const int32_t *__restrict__ tile_chunk = a.tile_chunk;
  const int64_t *__restrict__ chunk_lbeg = a.chunk_lbeg;
  const uint64_t *__restrict__ list64 = a.list64;
  const uint32_t *__restrict__ listls = a.listls;
  const int32_t *__restrict__ chunk_entry = a.chunk_entry;
  const uint32_t *__restrict__ emask = a.emask;
  const int32_t *__restrict__ ecoff = a.ecoff;
  const uint8_t *__restrict__ rdim = a.rdim;
  const uint8_t *__restrict__ cdim = a.cdim;
  const int64_t *__restrict__ wave_out = a.wave_out64;
  const T *__restrict__ P = static_cast<const T *>(a.P);
  const T *__restrict__ Q = static_cast<const T *>(a.Q);
  T *__restrict__ O = static_cast<T *>(a.O);
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int qr = w >> 1, qc = w & 1;
  // Block sizes of the tile (rows of absent tile rows read 0).
  int NI = 0, NJ = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    NI = max(NI, (int)rdim[(int64_t)tile * 8 + k]);
    NJ = max(NJ, (int)cdim[(int64_t)tile * 8 + k]);
  }
  NI = __builtin_amdgcn_readfirstlane(NI);
  NJ = __builtin_amdgcn_readfirstlane(NJ);
  // Packing: RP row blocks of RH element rows per MFMA tile (CP, CH for columns).
  const int lrh = NI <= 4 ? 2 : NI <= 8 ? 3 : 4, lch = NJ <= 4 ? 2 : NJ <= 8 ? 3 : 4;
  const int RP = 16 >> lrh, CP = 16 >> lch;
  const int NTA = 4 / RP, NTB = 4 / CP;
  const int ir = r & ((1 << lrh) - 1), jc = r & ((1 << lch) - 1);
  const int ru = r >> lrh, cu = r >> lch;
  const bool rowok = ir < NI, colok = jc < NJ;
  dbl4 a64[16];
  flt4 a32[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    a64[u] = dbl4{0.0, 0.0, 0.0, 0.0};
    a32[u] = flt4{0.f, 0.f, 0.f, 0.f};
  }
  const int32_t c0 = tile_chunk[tile], c1 = tile_chunk[tile + 1];
  if (c0 < c1) {
    int32_t wb = c0;
    int32_t cc = min(wb + lane, c1);
    int64_t wcl = chunk_lbeg[cc];
    int32_t wce = chunk_entry[cc];
    auto cl_at = [&](int32_t x) { return readlane64(wcl, min(x, c1) - wb); };
    auto ce_at = [&](int32_t x) { return __builtin_amdgcn_readlane(wce, min(x, c1) - wb); };
    auto list_idx = [&](int64_t lbeg, int32_t nb) { return lbeg + min(w + kWaves * lane, nb - 1); };
    auto entry_regs = [&](int32_t e0, int32_t e1, uint32_t &m, int32_t &o) {
      const int32_t e = min(e0 + lane, e1 - 1);
      m = emask[e];
      o = ecoff[e];
    };
    uint32_t em, emn = 0;
    int32_t eo, eon = 0;
    uint64_t lvn = 0;
    uint32_t lsn = 0;
    {
      const int64_t cl0 = cl_at(c0), cl1 = cl_at(c0 + 1);
      const int64_t i0 = list_idx(cl0, (int32_t)(cl1 - cl0));
      issue_stage_mx<T>(list64[i0], listls[i0], (int32_t)(cl1 - cl0), P, Q, stage0, w, lane);
      entry_regs(ce_at(c0), ce_at(c0 + 1), emn, eon);
      if (c0 + 1 < c1) {
        const int64_t i1 = list_idx(cl1, (int32_t)(cl_at(c0 + 2) - cl1));
        lvn = list64[i1];
        lsn = listls[i1];
      }
    }
    const uint32_t quad_rows = 0xfu << (4 * qr), quad_cols = 0xfu << (4 * qc);
    for (int32_t c = c0; c < c1; ++c) {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      const bool odd = ((c - c0) & 1) != 0;
      const T *cur = odd ? stage1 : stage0;
      em = emn;
      eo = eon;
      const int32_t ne = ce_at(c + 1) - ce_at(c);
      if (c + 1 < c1) {
        const int64_t cl1 = cl_at(c + 1), cl2 = cl_at(c + 2);
        issue_stage_mx<T>(lvn, lsn, (int32_t)(cl2 - cl1), P, Q, odd ? stage0 : stage1, w, lane);
        entry_regs(ce_at(c + 1), ce_at(c + 2), emn, eon);
        if (c + 2 < c1) {
          const int64_t i2 = list_idx(cl2, (int32_t)(cl_at(c + 3) - cl2));
          lvn = list64[i2];
          lsn = listls[i2];
        }
      }
      for (int i = 0; i < ne; ++i) {
        const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)em, i);
        const uint32_t ym = m & 0xffu, bm = (m >> 8) & 0xffu;
        if ((ym & quad_rows) == 0 || (bm & quad_cols) == 0) continue;  // no block pair in this quadrant
        const int32_t base = __builtin_amdgcn_readlane(eo, i);
        const int nx = (int)((m >> 16) & 15u) + 1;
        const int ablk = NI * nx, bblk = nx * NJ;
        const int bbase = base + ablk * __popc(ym);
        if constexpr (MODE == 4) {
          // Split-BF16 x3: one K = 16 step (nx <= 16); lane (r, g) holds
          // contraction indices 4g..4g+3 of its row (column) as four LDS words
          // (bits 0-15 hi, 16-31 lo), repacked into the hi and lo operands of
          // v_mfma_f32_16x16x16_bf16; hi.hi + hi.lo + lo.hi chain in FP32 and
          // each entry's sum is added into the FP64 accumulator.
          s16x4 ahi[4], alo[4], bhi[4], blo[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int u = 4 * qr + t * RP + ru, v = 4 * qc + t * CP + cu;
            const bool oka = t < NTA && rowok && ((ym >> u) & 1u) != 0;
            const bool okb = t < NTB && colok && ((bm >> v) & 1u) != 0;
            const int a0 = base + ablk * __popc(ym & ((1u << u) - 1u)) + ir + NI * 4 * g;
            const int b0 = bbase + bblk * __popc(bm & ((1u << v) - 1u)) + (QT ? jc + NJ * 4 * g : 4 * g + nx * jc);
            uint32_t wa[4], wb[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool kin = 4 * g + i < nx;
              const bool ra = oka && kin, rb = okb && kin;
              wa[i] = __float_as_uint(cur[ra ? a0 + NI * i : 0]);
              wb[i] = __float_as_uint(cur[rb ? b0 + (QT ? NJ * i : i) : 0]);
              if (!ra) wa[i] = 0u;
              if (!rb) wb[i] = 0u;
            }
            ahi[t] = pack_bf16_lo(wa);
            alo[t] = pack_bf16_hi(wa);
            bhi[t] = pack_bf16_lo(wb);
            blo[t] = pack_bf16_hi(wb);
          }
#pragma unroll
          for (int ta = 0; ta < 4; ++ta) {
            if (ta >= NTA || (ym & (((1u << RP) - 1u) << (4 * qr + ta * RP))) == 0) continue;
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) {
              if (tb >= NTB || (bm & (((1u << CP) - 1u) << (4 * qc + tb * CP))) == 0) continue;
              const int u = ta * 4 + tb;
              flt4 t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ahi[ta], bhi[tb], flt4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ahi[ta], blo[tb], t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(alo[ta], bhi[tb], t, 0, 0, 0);
#pragma unroll
              for (int e = 0; e < 4; ++e) a64[u][e] += (double)t[e];
            }
          }
          continue;
        }
        // This lane's element of each row unit (ta) and column unit (tb) at k-step 0.
        int pa[4], pb[4];
        bool va[4], vb[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int u = 4 * qr + t * RP + ru, v = 4 * qc + t * CP + cu;
          va[t] = t < NTA && rowok && ((ym >> u) & 1u) != 0;
          vb[t] = t < NTB && colok && ((bm >> v) & 1u) != 0;
          pa[t] = base + ablk * __popc(ym & ((1u << u) - 1u)) + ir + NI * g;
          pb[t] = bbase + bblk * __popc(bm & ((1u << v) - 1u)) + (QT ? jc + NJ * g : g + nx * jc);
        }
        const int KS = (nx + 3) >> 2;
        const int sa = 4 * NI, sb = QT ? 4 * NJ : 4;
        for (int s4 = 0; s4 < KS; ++s4) {
          const bool kv = s4 + 1 < KS || 4 * s4 + g < nx;
          T av[4], bv[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const bool oka = va[t] && kv, okb = vb[t] && kv;
            av[t] = cur[oka ? pa[t] + sa * s4 : 0];
            bv[t] = cur[okb ? pb[t] + sb * s4 : 0];
            if (!oka) av[t] = (T)0;
            if (!okb) bv[t] = (T)0;
          }
#pragma unroll
          for (int ta = 0; ta < 4; ++ta) {
            if (ta >= NTA || (ym & (((1u << RP) - 1u) << (4 * qr + ta * RP))) == 0) continue;
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) {
              if (tb >= NTB || (bm & (((1u << CP) - 1u) << (4 * qc + tb * CP))) == 0) continue;
              const int u = ta * 4 + tb;
              if constexpr (MODE == 0) {
                a64[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ta], bv[tb], a64[u], 0, 0, 0);
              } else if constexpr (MODE == 1) {
                a32[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[ta], bv[tb], a32[u], 0, 0, 0);
              } else {
                const flt4 t = __builtin_amdgcn_mfma_f32_16x16x4f32(av[ta], bv[tb], flt4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) a64[u][e] += (double)t[e];
              }
            }
          }
        }
      }
      if (c + 4 > wb + 63 && c + 1 < c1) {
        wb = c + 1;
        cc = min(wb + lane, c1);
        wcl = chunk_lbeg[cc];
        wce = chunk_entry[cc];
      }
    }
  }
  // Element (R, r) of MFMA tile (ta, tb): row R % RH of quadrant block row
  // ta RP + R / RH, column r % CH of quadrant block column tb CP + r / CH;
  // written where it lies inside that block's shape.
  const int64_t *wo = wave_out + ((int64_t)tile * kWaves + w) * 16;
#pragma unroll
  for (int ta = 0; ta < 4; ++ta) {
    if (ta >= NTA) continue;
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      if (tb >= NTB) continue;
      const int u = ta * 4 + tb;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // FP64 MFMA accumulators hold D[g + 4e][r]; FP32 ones (modes 1 and 2,
        // whose FP64 sums add FP32 results element for element) D[4g + e][r].
        const int R = MODE == 0 ? g + 4 * e : 4 * g + e;
        const int bu = ta * RP + (R >> lrh), rowi = R & ((1 << lrh) - 1);
        const int bv = tb * CP + cu;
        const int64_t off = wo[bu * 4 + bv];
        if (off >= 0 && rowi < NI && colok) O[off + rowi + (int64_t)NI * jc] = MODE == 1 ? (T)a32[u][e] : (T)a64[u][e];
      }
    }
  }
}

// Global tile number of a launch -> the product's arguments and its tile.
__device__ inline int32_t tile_at(const TileOne &one, int32_t t, TileArgs &a) {
  a = one.a;
  return t;
}
__device__ inline int32_t tile_at(const TileGroup &g, int32_t t, TileArgs &a) {
  int32_t j = 0;
#pragma unroll
  for (int k = 1; k < kMaxGroup; ++k) j += (k < g.ngrp && g.a[k].tile_base <= t) ? 1 : 0;
  a = g.a[j];
  return t - a.tile_base;
}

// Persistent launch of class tiles: the grid (a multiple of 8 workgroups) gives
// each XCD (workgroup b runs on XCD b % 8) its tiles, and each workgroup takes
// every (grid/8)-th of them, so neighbouring tiles (same rows) share an L2. With
// one workgroup per tile this is the order of the other tile kernels.
template <int MODE, bool QT, int STG, class ARG>
__global__ void __launch_bounds__(kTileThreads) k_tile_quad(const ARG arg) {
  using T = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int STAGE = STG + kLdsPad * (int)(8 / sizeof(T));
  __shared__ T stage0[STAGE];
  __shared__ T stage1[STAGE];
  int32_t tbeg, tend;
  xcd_units(arg.xcd, tbeg, tend);
  for (int32_t tg = tbeg + (int32_t)(blockIdx.x >> 3); tg < tend; tg += (int32_t)(gridDim.x >> 3)) {
    __syncthreads();  // the previous tile's last chunk is read before this tile's first copies
    TileArgs a;
    const int32_t tile = tile_at(arg, tg, a);
    quad_tile<MODE, QT>(a, tile, stage0, stage1);
  }
}

// Workgroups that give every XCD enough for its units.
unsigned xcd_grid(const int32_t *xcd) {
  int32_t most = 0;
  for (int x = 0; x < cq::kXcds; ++x) most = std::max(most, xcd[x + 1] - xcd[x]);
  return (unsigned)cq::kXcds * (unsigned)most;
}

template <int MODE, bool QT, class ARG>
int launch_kind(int kind, const ARG &arg, int32_t wgs, hipStream_t s) {
  // One workgroup per tile; the class-tile kernel also runs persistent grids
  // of wgs workgroups (rounded up to a multiple of 8).
  unsigned gridx = xcd_grid(arg.xcd);
  if ((kind == kKindQuadSmall || kind == kKindQuadLarge) && wgs > 0)
    gridx = std::min(gridx, 8u * (unsigned)((wgs + 7) / 8));
  const dim3 blk(kTileThreads);
  switch (kind) {
    case kKindDense4: hipLaunchKernelGGL((k_quad4<MODE, QT, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    case kKindDenseMx: hipLaunchKernelGGL((k_tile_dense_mx<MODE, QT, ARG>), dim3(gridx), blk, 0, s, arg); break;
    case kKindMixedSmall: hipLaunchKernelGGL((k_tile_mixed<MODE, QT, kStgSmall, ARG>), dim3(gridx), blk, 0, s, arg); break;
    case kKindMixedLarge: hipLaunchKernelGGL((k_tile_mixed<MODE, QT, kStgLarge, ARG>), dim3(gridx), blk, 0, s, arg); break;
    case kKindQuadSmall: hipLaunchKernelGGL((k_tile_quad<MODE, QT, kStgSmall, ARG>), dim3(gridx), blk, 0, s, arg); break;
    case kKindQuadLarge: hipLaunchKernelGGL((k_tile_quad<MODE, QT, kStgLarge, ARG>), dim3(gridx), blk, 0, s, arg); break;
    case kKindUniform + 9: hipLaunchKernelGGL((k_wave_products<MODE, QT, 9, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    case kKindUniform + 13: hipLaunchKernelGGL((k_wave_products<MODE, QT, 13, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    case kKindUniform + 16: hipLaunchKernelGGL((k_wave_products<MODE, QT, 16, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    default: return cq::set_errorf(CQMM_ERR_ARG, "tile products: kernel kind %d has no instance", kind);
  }
  return cq::hip_check(hipGetLastError(), "tile-product kernel launch");
}

template <int MODE, bool QT, class ARG>
int launch_uniform(int kind, const ARG &arg, hipStream_t s) {
  const unsigned gridx = xcd_grid(arg.xcd);
  switch (kind) {
    case kKindUniform + 9: hipLaunchKernelGGL((k_wave_products<MODE, QT, 9, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    case kKindUniform + 13: hipLaunchKernelGGL((k_wave_products<MODE, QT, 13, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    case kKindUniform + 16: hipLaunchKernelGGL((k_wave_products<MODE, QT, 16, ARG>), dim3(gridx), dim3(64), 0, s, arg); break;
    default: return cq::set_errorf(CQMM_ERR_ARG, "tile products: kernel kind %d has no instance", kind);
  }
  return cq::hip_check(hipGetLastError(), "tile-product kernel launch");
}

template <int MODE, bool QT, class ARG>
int launch_quad(int kind, const ARG &arg, int32_t wgs, hipStream_t s) {
  unsigned gridx = xcd_grid(arg.xcd);
  if (wgs > 0) gridx = std::min(gridx, 8u * (unsigned)((wgs + 7) / 8));
  if (kind == kKindQuadSmall) hipLaunchKernelGGL((k_tile_quad<MODE, QT, kStgSmall, ARG>), dim3(gridx), dim3(kTileThreads), 0, s, arg);
  else hipLaunchKernelGGL((k_tile_quad<MODE, QT, kStgLarge, ARG>), dim3(gridx), dim3(kTileThreads), 0, s, arg);
  return cq::hip_check(hipGetLastError(), "class-tile kernel launch");
}

template <class ARG>
int launch_any(int mode, bool qt, int kind, const ARG &arg, int32_t wgs, hipStream_t s) {
  switch (mode * 2 + (qt ? 1 : 0)) {
    case 0: return launch_kind<0, false, ARG>(kind, arg, wgs, s);
    case 1: return launch_kind<0, true, ARG>(kind, arg, wgs, s);
    case 2: return launch_kind<1, false, ARG>(kind, arg, wgs, s);
    case 3: return launch_kind<1, true, ARG>(kind, arg, wgs, s);
    case 4: return launch_kind<2, false, ARG>(kind, arg, wgs, s);
    case 5: return launch_kind<2, true, ARG>(kind, arg, wgs, s);
    // Mode 3 (a block's products of one chunk may be summed in FP32) runs as
    // mode 2, which adds every product in FP64.
    case 6: return launch_kind<2, false, ARG>(kind, arg, wgs, s);
    case 7: return launch_kind<2, true, ARG>(kind, arg, wgs, s);
    // Split-BF16 x3 (mode 4) runs in the class-tile kernel and the fixed-size
    // kernels of 9x9, 13x13 and 16x16 blocks.
    case 8:
    case 9:
      if (kind == kKindQuadSmall || kind == kKindQuadLarge)
        return qt ? launch_quad<4, true, ARG>(kind, arg, wgs, s) : launch_quad<4, false, ARG>(kind, arg, wgs, s);
      if (kind == kKindUniform + 9 || kind == kKindUniform + 13 || kind == kKindUniform + 16)
        return qt ? launch_uniform<4, true, ARG>(kind, arg, s) : launch_uniform<4, false, ARG>(kind, arg, s);
      return cq::set_error(CQMM_ERR_STATE, "split-BF16 products need blocks of 9 to 16 or a class-tile schedule");
    default: return cq::set_errorf(CQMM_ERR_ARG, "tile products: precision mode %d", mode);
  }
}

int tile_kind(const cq::TilePlan &tp) {
  if (tp.maxn) {
    if (tp.dense) return kKindDenseMx;
    if (tp.quad) return stage_elems(tp.maxn) == kStgSmall ? kKindQuadSmall : kKindQuadLarge;
    return stage_elems(tp.maxn) == kStgSmall ? kKindMixedSmall : kKindMixedLarge;
  }
  if (tp.dense) return kKindDense4;
  return kKindUniform + tp.nsf;
}

}  // namespace

namespace cq {

int launch_tile_products_f32(const TilePlan &tp, bool q_trans, const float *P, const float *Q, float *O, int mode,
                             hipStream_t s) {
  if (tp.n_tiles == 0) return CQMM_OK;
  return launch_tile_args(tp, q_trans, mode, tile_launch_args(tp, P, Q, O), s);
}

bool tiles_write_f64(const TilePlan &tp) { return tp.n_wave > 0; }

TileArgs tile_launch_args(const TilePlan &tp, const void *P, const void *Q, void *O) {
  TileArgs a;
  std::memset(&a, 0, sizeof(a));
  a.tile_chunk = tp.tile_chunk.as<int32_t>();
  a.chunk_lbeg = tp.chunk_lbeg.as<int64_t>();
  a.list64 = tp.list64.as<uint64_t>();
  a.listls = tp.listls.as<uint32_t>();
  a.pstart = tp.pstart.as<int64_t>();
  a.pcnt = tp.pcnt.as<uint64_t>();
  a.prod = tp.prod.as<uint32_t>();
  a.wave_out = tp.wave_out.as<int32_t>();
  a.wave_out64 = tp.wave_out64.as<int64_t>();
  a.wave_dim = tp.wave_dim.as<uint8_t>();
  a.chunk_entry = tp.chunk_entry.as<int32_t>();
  a.emask = tp.entry_mask.as<uint32_t>();
  a.ecoff = tp.entry_coff.as<int32_t>();
  a.rdim = tp.tile_rdim.as<uint8_t>();
  a.cdim = tp.tile_cdim.as<uint8_t>();
  a.P = P;
  a.Q = Q;
  a.O = O;
  a.n_tiles = tp.n_wave ? tp.n_wave : tp.n_tiles;
  a.tile_base = 0;
  a.plan = &tp;
  return a;
}

bool tiles_take_bf16x3(const TilePlan &tp) {
  if (tp.n_tiles == 0) return false;
  const int k = tile_kind(tp);
  return k == kKindQuadSmall || k == kKindQuadLarge || k == kKindUniform + 9 || k == kKindUniform + 13 ||
         k == kKindUniform + 16;
}

int tile_family(const TilePlan &tp) {
  const int k = tile_kind(tp);
  if (k == kKindQuadSmall || k == kKindQuadLarge) return CQMM_TILES_CLASS;
  if (k == kKindMixedSmall || k == kKindMixedLarge) return CQMM_TILES_MIXED;
  return k;  // dense 1, dense mixed 2, uniform 16 + n
}

int tile_group_key(const TilePlan &tp, bool q_trans, int mode) {
  return (tile_kind(tp) * 2 + (q_trans ? 1 : 0)) * 4 + mode;
}

// Units that are split over the XCDs by count: k_quad4's that fit the card at once
// (32 wavefronts on each of 256 compute units) and have at most 256 records on
// average (64 atoms, type 1 8/10/14 A: 27.7 us by work, 26.3 by count). Long units
// are better split by work at any number (64 atoms, type 2 12/20/28 A: 479 us by
// work, 515 by count), and so are the other kernels' (32 atoms 16x16, some 3000
// units: 406 us by work, 484 by count).
constexpr int32_t kBriefWords = 2048;
static int32_t units_at_once(const TilePlan &tp) { return tile_kind(tp) == kKindDense4 ? 32 * 256 : 0; }

int launch_tile_args(const TilePlan &tp, bool q_trans, int mode, const TileArgs &a, hipStream_t s) {
  if (a.n_tiles <= 0) return CQMM_OK;
  TileOne one;
  one.a = a;
  const WorkParts *p = &tp.parts;
  xcd_split(&p, 1, units_at_once(tp), kBriefWords, one.xcd);
  return launch_any(mode, q_trans, tile_kind(tp), one, tp.wgs, s);
}

int launch_tile_group(const TilePlan &tp, bool q_trans, int mode, TileGroup &g, hipStream_t s) {
  if (g.ngrp <= 0 || g.total <= 0) return CQMM_OK;
  if (g.ngrp > kMaxGroup) return set_errorf(CQMM_ERR_ARG, "grouped tile launch: %d products (at most %d)", g.ngrp, kMaxGroup);
  const WorkParts *p[kMaxGroup];
  for (int j = 0; j < g.ngrp; ++j) p[j] = &g.a[j].plan->parts;
  xcd_split(p, g.ngrp, units_at_once(tp), kBriefWords, g.xcd);
  return launch_any(mode, q_trans, tile_kind(tp), g, tp.wgs, s);
}

// CQMM_TILES=0 builds plans without the tile schedule (triplet kernels only).
bool tiles_enabled() {
  static const bool v = [] {
    const char *e = getenv("CQMM_TILES");
    return !(e && std::string(e) == "0");
  }();
  return v;
}

// Read at every plan build, so that one process can build both schedules.
bool class_tiles_enabled() {
  const char *e = getenv("CQMM_MIXED_TILES");
  return e && std::string(e) == "class";
}

// CQMM_TILE_ROWS=morton: plans built from a system order their tile rows like
// the tile columns (symmetric-result plans always do).
bool morton_rows_enabled() {
  const char *e = getenv("CQMM_TILE_ROWS");
  return e && std::string(e) == "morton";
}

// CQMM_TILE_ROWS=primary: symmetric-result plans keep primary-order tile rows.
bool primary_rows_forced() {
  const char *e = getenv("CQMM_TILE_ROWS");
  return e && std::string(e) == "primary";
}

bool uniform_class_tiles_enabled() {
  const char *e = getenv("CQMM_UNIFORM_TILES");
  return e && std::string(e) == "class";
}

std::vector<int32_t> group_ranks_by_size(const std::vector<int32_t> &rank, const int32_t *size) {
  const int32_t n = (int32_t)rank.size();
  std::vector<int32_t> idx(n), out(n);
  for (int32_t i = 0; i < n; ++i) idx[i] = i;
  std::sort(idx.begin(), idx.end(), [&](int32_t a, int32_t b) {
    return size[a] != size[b] ? size[a] < size[b] : rank[a] < rank[b];
  });
  int32_t pos = 0, prev = -1;
  for (int32_t k = 0; k < n; ++k) {
    const int32_t i = idx[k];
    if (size[i] != prev) {
      pos = (pos + 7) & ~7;
      prev = size[i];
    }
    out[i] = pos++;
  }
  return out;
}

std::vector<int32_t> halo_morton_rank(int32_t np_in_halo, const int32_t *nh_part, const int32_t *lab_hcover,
                                      int32_t ncovery, int32_t ncoverz) {
  std::vector<uint64_t> code(np_in_halo);
  const int64_t nyz = (int64_t)ncovery * ncoverz;
  for (int32_t p = 0; p < np_in_halo; ++p) {
    const int64_t l = (int64_t)lab_hcover[p] - 1;
    const uint64_t x = (uint64_t)(l / nyz), y = (uint64_t)((l / ncoverz) % ncovery), z = (uint64_t)(l % ncoverz);
    uint64_t c = 0;
    for (int bit = 0; bit < 20; ++bit)
      c |= (((x >> bit) & 1u) << (3 * bit)) | (((y >> bit) & 1u) << (3 * bit + 1)) | (((z >> bit) & 1u) << (3 * bit + 2));
    code[p] = c;
  }
  std::vector<int32_t> order(np_in_halo);
  for (int32_t p = 0; p < np_in_halo; ++p) order[p] = p;
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return code[a] < code[b]; });
  std::vector<int64_t> first(np_in_halo + 1, 0);
  for (int32_t p = 0; p < np_in_halo; ++p) first[p + 1] = first[p] + nh_part[p];
  std::vector<int32_t> rank(first[np_in_halo]);
  int32_t next = 0;
  for (int32_t p : order)
    for (int64_t k = first[p]; k < first[p + 1]; ++k) rank[k] = next++;
  return rank;
}

// Output slots to wavefronts, per tile: a Latin square over (tile row,
// column) — with k = (row + perm[column]) % 8, wavefront k % kWaves owns the
// block as its slot (8 / kWaves) * row + k / kWaves, so every wavefront owns
// 8 / kWaves blocks of each tile row and column, which spreads every entry's
// rectangle of products evenly — chosen among kLatinTries column permutations
// (the first with the smallest largest wavefront product count).
// owner[tile*64 + row*8 + col] = wavefront * kSlots + slot, or 0xff where the
// tile has no such output block; wave_out[tile*64 + owner] = that block.
constexpr int kLatinTries = 24;
struct LatinPerms {
  int8_t p[kLatinTries][8];
};

__global__ void k_assign_slots(const int32_t *__restrict__ cnt, const int32_t *__restrict__ tile_out,
                               LatinPerms perms, int32_t n_tiles, uint8_t *__restrict__ owner,
                               int32_t *__restrict__ wave_out) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tiles) return;
  const int32_t *c = cnt + (int64_t)t * 64;
  int32_t cs[64];
  for (int sl = 0; sl < 64; ++sl) cs[sl] = c[sl];
  int best = 0;
  int64_t best_max = -1;
  for (int k = 0; k < kLatinTries; ++k) {
    int64_t load[kWaves] = {};
    for (int sl = 0; sl < 64; ++sl) load[(((sl >> 3) + perms.p[k][sl & 7]) & 7) % kWaves] += cs[sl];
    int64_t m = 0;
    for (int w = 0; w < kWaves; ++w) m = load[w] > m ? load[w] : m;
    if (best_max < 0 || m < best_max) {
      best_max = m;
      best = k;
    }
  }
  for (int u = 0; u < 8; ++u)
    for (int col = 0; col < 8; ++col) {
      const int64_t sl = (int64_t)t * 64 + u * 8 + col;
      const int32_t ob = tile_out[sl];
      if (ob < 0) {
        owner[sl] = 0xff;
        continue;
      }
      const int k = (u + perms.p[best][col]) & 7;
      const int o = (k % kWaves) * kSlots + (8 / kWaves) * u + k / kWaves;
      owner[sl] = (uint8_t)o;
      wave_out[(int64_t)t * 64 + o] = ob;
    }
}

// The kLatinTries column permutations (the first is the identity; the others
// a fixed pseudo-random sequence, so plans are reproducible).
LatinPerms latin_perms() {
  LatinPerms lp;
  uint64_t lcg = 0x9e3779b97f4a7c15ull;
  for (int k = 0; k < kLatinTries; ++k) {
    int q[8];
    for (int i = 0; i < 8; ++i) q[i] = i;
    for (int i = 7; k > 0 && i > 0; --i) {
      lcg = lcg * 6364136223846793005ull + 1442695040888963407ull;
      const int j = (int)((lcg >> 33) % (uint64_t)(i + 1));
      std::swap(q[i], q[j]);
    }
    for (int i = 0; i < 8; ++i) lp.p[k][i] = (int8_t)q[i];
  }
  return lp;
}

// Device owner table and wave_out (tile_out32: the tiles' output blocks on
// the device) from the products per output slot.
int assign_slots(const TileBuildInput &in, const int32_t *tile_out32, DevBuf &d_owner, DevBuf &wave_out,
                 hipStream_t s) {
  const int64_t n = in.n_trip;
  const size_t ns = (size_t)in.n_tiles * 64;
  int st;
  DevBuf d_cnt;
  if ((st = d_cnt.alloc(ns * 4)) || (st = d_owner.alloc(ns)) || (st = wave_out.alloc(ns * 4))) return st;
  if ((st = hip_check(hipMemsetAsync(d_cnt.p, 0, ns * 4, s), "memset slot counts"))) return st;
  hipLaunchKernelGGL(k_slot_counts, dim3(grid1(n, 256)), dim3(256), 0, s, in.key, in.slot, n, in.nx, d_cnt.as<int32_t>());
  hipLaunchKernelGGL(k_fill_i32, dim3(grid1((int64_t)ns, 256)), dim3(256), 0, s, wave_out.as<int32_t>(), (int64_t)ns, -1);
  hipLaunchKernelGGL(k_assign_slots, dim3(grid1(in.n_tiles, 128)), dim3(128), 0, s, d_cnt.as<int32_t>(), tile_out32,
                     latin_perms(), in.n_tiles, d_owner.as<uint8_t>(), wave_out.as<int32_t>());
  if ((st = hip_check(hipGetLastError(), "slot assignment launch"))) return st;
  // d_cnt is freed on return: wait for the kernels that read it.
  return hip_check(hipStreamSynchronize(s), "slot assignment");
}

// The plan's work and where its 64ths begin, from the device prefix w (k_work_parts).
template <class W>
int work_parts(const W *w, const int32_t *at, int32_t n, TilePlan &tp, hipStream_t s) {
  DevBuf d;
  int64_t h[kWorkParts + 2];
  int st;
  if ((st = d.alloc(sizeof(h)))) return st;
  hipLaunchKernelGGL((k_work_parts<W>), dim3(1), dim3(128), 0, s, w, at, n, d.as<int64_t>());
  if ((st = hip_check(hipMemcpyAsync(h, d.p, sizeof(h), hipMemcpyDeviceToHost, s), "D2H work parts")) ||
      (st = hip_check(hipStreamSynchronize(s), "work parts")))
    return st;
  for (int k = 0; k <= kWorkParts; ++k) tp.parts.at[k] = (int32_t)h[k];
  tp.parts.work = h[kWorkParts + 1];
  return CQMM_OK;
}

int build_tiles_mixed(const TileBuildInput &in, TilePlan &tp, hipStream_t s);

int build_tiles(const TileBuildInput &in, TilePlan &tp, hipStream_t s) {
  if (in.nsf == 0) return build_tiles_mixed(in, tp, s);
  cq::PhaseTimer pt;
  const int64_t n = in.n_trip;
  const int64_t ns2 = (int64_t)in.nsf * in.nsf;
  int st;
  tp = TilePlan();
  tp.nsf = in.nsf;
  tp.n_tiles = in.n_tiles;
  tp.dense = in.nsf == kDenseNsf;
  // Output blocks of the tiles' quadrants by block index (element offset /
  // NSF^2): quadrant (w / 2, w % 2) has rows 4*(w/2)..+3, columns 4*(w%2)..+3.
  std::vector<int32_t> wave_out((size_t)in.n_tiles * 64, -1), src;
  parallel_for(in.n_tiles, [&](int64_t b, int64_t e) {
    for (int64_t t = b; t < e; ++t)
      for (int u = 0; u < 8; ++u)
        for (int c = 0; c < 8; ++c) {
          const int64_t o = in.tile_out[t * 64 + u * 8 + c];
          if (o >= 0) wave_out[(t * kWaves + (u >> 2) * 2 + (c >> 2)) * 16 + (u & 3) * 4 + (c & 3)] = (int32_t)(o / ns2);
        }
  });
  // Only the quadrants with output blocks are work.
  src.reserve((size_t)in.n_tiles * kWaves);
  for (int64_t q = 0; q < (int64_t)in.n_tiles * kWaves; ++q) {
    bool any = false;
    for (int k = 0; k < 16; ++k) any |= wave_out[q * 16 + k] >= 0;
    if (!any) continue;
    if ((int64_t)src.size() != q)
      for (int k = 0; k < 16; ++k) wave_out[src.size() * 16 + k] = wave_out[q * 16 + k];
    src.push_back((int32_t)q);
  }
  wave_out.resize(src.size() * 16);
  tp.n_wave = (int32_t)src.size();
  if ((st = tp.wave_out.alloc(wave_out.size() * 4))) return st;
  if ((st = hip_check(hipMemcpyAsync(tp.wave_out.p, wave_out.data(), wave_out.size() * 4, hipMemcpyHostToDevice, s),
                      "H2D wave_out")) ||
      (st = hip_check(hipStreamSynchronize(s), "wave_out")))
    return st;
  pt.mark("  tiles: quadrants");
  // Sort the products by (tile, contraction atom).
  unsigned end_bit = 1;
  const uint64_t kmax = (uint64_t)in.n_tiles * (uint64_t)in.nx;
  while (end_bit < 64 && ((uint64_t)1 << end_bit) < kmax) ++end_bit;
  DevBuf d_perm, d_key2, d_perm2, d_tmp;
  if ((st = d_perm.alloc(n * 4)) || (st = d_key2.alloc(n * 8)) || (st = d_perm2.alloc(n * 4))) return st;
  hipLaunchKernelGGL(k_iota32, dim3(grid1(n, 256)), dim3(256), 0, s, d_perm.as<int32_t>(), n);
  size_t bytes = 0;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, bytes, in.key, d_key2.as<uint64_t>(), d_perm.as<int32_t>(),
                                           d_perm2.as<int32_t>(), (size_t)n, 0, end_bit, s);
  if ((st = hip_check(e, "radix_sort_pairs (tiles, size)"))) return st;
  if ((st = d_tmp.alloc(bytes))) return st;
  e = rocprim::radix_sort_pairs(d_tmp.p, bytes, in.key, d_key2.as<uint64_t>(), d_perm.as<int32_t>(),
                                d_perm2.as<int32_t>(), (size_t)n, 0, end_bit, s);
  if ((st = hip_check(e, "radix_sort_pairs (tiles)"))) return st;
  if ((st = hip_check(hipStreamSynchronize(s), "tile sort"))) return st;
  d_tmp.release();
  d_perm.release();
  pt.mark("  tiles: sort");
  // Entries = distinct keys.
  DevBuf d_flag, d_eid;
  if ((st = d_flag.alloc(n * 4)) || (st = d_eid.alloc(n * 4))) return st;
  hipLaunchKernelGGL(k_entry_flags, dim3(grid1(n, 256)), dim3(256), 0, s, d_key2.as<uint64_t>(), n, d_flag.as<int32_t>());
  if ((st = inclusive_scan(d_flag.as<int32_t>(), d_eid.as<int32_t>(), (size_t)n, s))) return st;
  d_flag.release();
  int32_t ne32 = 0;
  if ((st = hip_check(hipMemcpyAsync(&ne32, d_eid.as<int32_t>() + (n - 1), 4, hipMemcpyDeviceToHost, s), "D2H entries")) ||
      (st = hip_check(hipStreamSynchronize(s), "entry count")))
    return st;
  const int64_t ne = ne32;
  tp.n_entries = ne;
  DevBuf d_ep, d_eq, d_etile, d_tebeg;
  if ((st = d_ep.alloc(ne * 8 * 4)) || (st = d_eq.alloc(ne * 8 * 4)) || (st = d_etile.alloc(ne * 4)) ||
      (st = d_tebeg.alloc(((size_t)in.n_tiles + 1) * 4)))
    return st;
  hipLaunchKernelGGL(k_fill_i32, dim3(grid1(ne * 8, 256)), dim3(256), 0, s, d_ep.as<int32_t>(), ne * 8, -1);
  hipLaunchKernelGGL(k_fill_i32, dim3(grid1(ne * 8, 256)), dim3(256), 0, s, d_eq.as<int32_t>(), ne * 8, -1);
  hipLaunchKernelGGL(k_entry_fill, dim3(grid1(n, 256)), dim3(256), 0, s, d_key2.as<uint64_t>(), d_perm2.as<int32_t>(),
                     d_eid.as<int32_t>(), in.slot, in.p, in.q, n, in.nx, ns2, d_ep.as<int32_t>(), d_eq.as<int32_t>(),
                     d_etile.as<int32_t>());
  d_eid.release();
  d_perm2.release();
  d_key2.release();
  hipLaunchKernelGGL(k_tile_ebeg, dim3(grid1((int64_t)in.n_tiles + 1, 256)), dim3(256), 0, s, d_etile.as<int32_t>(), ne,
                     in.n_tiles, d_tebeg.as<int32_t>());
  // Entry records of the quadrants: count, first record of each, fill.
  const size_t nq = src.size();
  DevBuf d_src, d_nrec, d_nprod, d_nload;
  if ((st = d_src.alloc(nq * 4)) || (st = d_nrec.alloc(nq * 8)) || (st = d_nprod.alloc(nq * 8)) ||
      (st = d_nload.alloc(nq * 8)) || (st = tp.pstart.alloc((nq + 1) * 8)))
    return st;
  if ((st = hip_check(hipMemcpyAsync(d_src.p, src.data(), nq * 4, hipMemcpyHostToDevice, s), "H2D quadrants"))) return st;
  const dim3 grid(grid1((int64_t)nq, 4));
  auto *count = tp.dense ? &k_wave_records<false, true> : &k_wave_records<false, false>;
  hipLaunchKernelGGL(count, grid, dim3(256), 0, s, d_src.as<int32_t>(), tp.n_wave, tp.wave_out.as<int32_t>(), d_tebeg.as<int32_t>(), d_ep.as<int32_t>(), d_eq.as<int32_t>(),
                     d_nrec.as<int64_t>(), d_nprod.as<int64_t>(), d_nload.as<int64_t>(), nullptr, nullptr);
  int64_t nrec = 0, nprod = 0, nload = 0;
  if ((st = hip_check(hipMemsetAsync(tp.pstart.p, 0, 8, s), "memset pstart")) ||
      (st = inclusive_scan(d_nrec.as<int64_t>(), tp.pstart.as<int64_t>() + 1, nq, s)) ||
      (st = inclusive_scan(d_nprod.as<int64_t>(), d_nprod.as<int64_t>(), nq, s)) ||
      (st = inclusive_scan(d_nload.as<int64_t>(), d_nload.as<int64_t>(), nq, s)) ||
      (st = hip_check(hipMemcpyAsync(&nrec, tp.pstart.as<int64_t>() + nq, 8, hipMemcpyDeviceToHost, s), "D2H records")) ||
      (st = hip_check(hipMemcpyAsync(&nprod, d_nprod.as<int64_t>() + nq - 1, 8, hipMemcpyDeviceToHost, s), "D2H products")) ||
      (st = hip_check(hipMemcpyAsync(&nload, d_nload.as<int64_t>() + nq - 1, 8, hipMemcpyDeviceToHost, s), "D2H loads")) ||
      (st = hip_check(hipStreamSynchronize(s), "entry records")))
    return st;
  tp.n_prod = nprod;
  tp.n_loads = nload;
  if (nprod != n)
    return set_errorf(CQMM_ERR_STATE, "tile plan: %lld listed products for %lld triplets", (long long)nprod,
                      (long long)n);
  // The kernels read 64 words at a time, k_quad4 64 ahead (no block: -1).
  if ((st = tp.prod.alloc(((size_t)nrec + kWavePad) * 4))) return st;
  if ((st = hip_check(hipMemsetAsync(tp.prod.as<uint32_t>() + nrec, 0xff, kWavePad * 4, s), "memset records tail"))) return st;
  auto *fill = tp.dense ? &k_wave_records<true, true> : &k_wave_records<true, false>;
  hipLaunchKernelGGL(fill, grid, dim3(256), 0, s, d_src.as<int32_t>(), tp.n_wave, tp.wave_out.as<int32_t>(), d_tebeg.as<int32_t>(), d_ep.as<int32_t>(), d_eq.as<int32_t>(),
                     nullptr, nullptr, nullptr, tp.pstart.as<int64_t>(), tp.prod.as<uint32_t>());
  if ((st = hip_check(hipGetLastError(), "tile builder launch"))) return st;
  st = work_parts(tp.pstart.as<int64_t>(), nullptr, tp.n_wave, tp, s);
  pt.mark("  tiles: entry records");
  return st;
}

int launch_tile_products(const TilePlan &tp, bool q_trans, const double *P, const double *Q, double *O,
                         hipStream_t s) {
  if (tp.n_tiles == 0) return CQMM_OK;
  return launch_tile_args(tp, q_trans, 0, tile_launch_args(tp, P, Q, O), s);
}

// Mixed block sizes: the uniform builder's steps with element offsets and
// per-row/column/contraction dimensions (see the kernels above).
int build_tiles_mixed(const TileBuildInput &in, TilePlan &tp, hipStream_t s) {
  const int64_t n = in.n_trip;
  const int32_t cap = stage_elems(in.maxn);
  int st;
  tp = TilePlan();
  tp.nsf = 0;
  tp.maxn = in.maxn;
  tp.n_tiles = in.n_tiles;
  DevBuf d_owner, d_rdim, d_cdim, d_xdim;
  tp.dense = in.maxn <= kDenseNsf;
  tp.quad = !tp.dense && in.class_uniform;
  if (tp.dense || tp.quad) {
    // Blocks of at most 4x4: wavefront w computes quadrant (w / 2, w % 2) of
    // the tile (k_tile_dense_mx); wave_out64 holds its blocks' element offsets.
    const size_t ns = (size_t)in.n_tiles * 64;
    std::vector<int64_t> wave_out(ns, -1);
    parallel_for(in.n_tiles, [&](int64_t b, int64_t e) {
      for (int64_t t = b; t < e; ++t)
        for (int u = 0; u < 8; ++u)
          for (int c = 0; c < 8; ++c)
            wave_out[(t * kWaves + (u >> 2) * 2 + (c >> 2)) * 16 + (u & 3) * 4 + (c & 3)] = in.tile_out[t * 64 + u * 8 + c];
    });
    if ((st = tp.wave_out64.alloc(ns * 8)) || (st = d_rdim.alloc((size_t)in.n_tiles * 8)) ||
        (st = d_cdim.alloc((size_t)in.n_tiles * 8)) || (st = d_xdim.alloc((size_t)std::max<int64_t>(in.nx, 1))))
      return st;
    if ((st = hip_check(hipMemcpyAsync(tp.wave_out64.p, wave_out.data(), ns * 8, hipMemcpyHostToDevice, s),
                        "H2D wave_out")) ||
        (st = hip_check(hipMemcpyAsync(d_rdim.p, in.tile_rdim, (size_t)in.n_tiles * 8, hipMemcpyHostToDevice, s),
                        "H2D rdim")) ||
        (st = hip_check(hipMemcpyAsync(d_cdim.p, in.tile_cdim, (size_t)in.n_tiles * 8, hipMemcpyHostToDevice, s),
                        "H2D cdim")) ||
        (st = hip_check(hipMemcpyAsync(d_xdim.p, in.xdim, (size_t)in.nx, hipMemcpyHostToDevice, s), "H2D xdim")) ||
        (st = hip_check(hipStreamSynchronize(s), "dense tile data")))
      return st;
  } else {
    // Slot owners on the device (from which output blocks exist), then the
    // per-wavefront element offsets and block shapes on the host.
    const size_t ns = (size_t)in.n_tiles * 64;
    std::vector<int32_t> exists(ns);
    parallel_for((int64_t)ns, [&](int64_t b, int64_t e) {
      for (int64_t k = b; k < e; ++k) exists[k] = in.tile_out[k] < 0 ? -1 : 0;
    });
    std::vector<uint8_t> owner(ns);
    {
      DevBuf d_exists, d_wo;
      if ((st = d_exists.alloc(ns * 4))) return st;
      if ((st = hip_check(hipMemcpyAsync(d_exists.p, exists.data(), ns * 4, hipMemcpyHostToDevice, s), "H2D exists")))
        return st;
      if ((st = assign_slots(in, d_exists.as<int32_t>(), d_owner, d_wo, s))) return st;
      if ((st = hip_check(hipMemcpyAsync(owner.data(), d_owner.p, ns, hipMemcpyDeviceToHost, s), "D2H owner")) ||
          (st = hip_check(hipStreamSynchronize(s), "owner")))
        return st;
    }
    std::vector<int64_t> wave_out(ns, -1);
    std::vector<uint8_t> wave_dim(ns, 0);
    for (int64_t t = 0; t < in.n_tiles; ++t)
      for (int sl = 0; sl < 64; ++sl) {
        const uint8_t o = owner[t * 64 + sl];
        if (o == 0xff) continue;
        const int64_t k = t * 64 + o;
        wave_out[k] = in.tile_out[t * 64 + sl];
        const int nr = in.tile_rdim[t * 8 + (sl >> 3)], nc = in.tile_cdim[t * 8 + (sl & 7)];
        if (nr < 1 || nr > 16 || nc < 1 || nc > 16)
          return set_errorf(CQMM_ERR_STATE, "tile plan: output block %d x %d outside 1..16", nr, nc);
        wave_dim[k] = (uint8_t)((nr - 1) | (nc - 1) << 4);
      }
    if ((st = tp.wave_out64.alloc(wave_out.size() * 8)) ||
        (st = tp.wave_dim.alloc(wave_dim.size())) || (st = d_rdim.alloc((size_t)in.n_tiles * 8)) ||
        (st = d_cdim.alloc((size_t)in.n_tiles * 8)) || (st = d_xdim.alloc((size_t)std::max<int64_t>(in.nx, 1))))
      return st;
    if ((st = hip_check(hipMemcpyAsync(tp.wave_out64.p, wave_out.data(), wave_out.size() * 8, hipMemcpyHostToDevice, s),
                        "H2D wave_out")) ||
        (st = hip_check(hipMemcpyAsync(tp.wave_dim.p, wave_dim.data(), wave_dim.size(), hipMemcpyHostToDevice, s),
                        "H2D wave_dim")) ||
        (st = hip_check(hipMemcpyAsync(d_rdim.p, in.tile_rdim, (size_t)in.n_tiles * 8, hipMemcpyHostToDevice, s),
                        "H2D rdim")) ||
        (st = hip_check(hipMemcpyAsync(d_cdim.p, in.tile_cdim, (size_t)in.n_tiles * 8, hipMemcpyHostToDevice, s),
                        "H2D cdim")) ||
        (st = hip_check(hipMemcpyAsync(d_xdim.p, in.xdim, (size_t)in.nx, hipMemcpyHostToDevice, s), "H2D xdim")) ||
        (st = hip_check(hipStreamSynchronize(s), "owner")))
      return st;
  }
  // Sort the products by (tile, contraction atom).
  unsigned end_bit = 1;
  const uint64_t kmax = (uint64_t)in.n_tiles * (uint64_t)in.nx;
  while (end_bit < 64 && ((uint64_t)1 << end_bit) < kmax) ++end_bit;
  DevBuf d_perm, d_key2, d_perm2, d_tmp;
  if ((st = d_perm.alloc(n * 4)) || (st = d_key2.alloc(n * 8)) || (st = d_perm2.alloc(n * 4))) return st;
  hipLaunchKernelGGL(k_iota32, dim3(grid1(n, 256)), dim3(256), 0, s, d_perm.as<int32_t>(), n);
  size_t bytes = 0;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, bytes, in.key, d_key2.as<uint64_t>(), d_perm.as<int32_t>(),
                                           d_perm2.as<int32_t>(), (size_t)n, 0, end_bit, s);
  if ((st = hip_check(e, "radix_sort_pairs (tiles, size)"))) return st;
  if ((st = d_tmp.alloc(bytes))) return st;
  e = rocprim::radix_sort_pairs(d_tmp.p, bytes, in.key, d_key2.as<uint64_t>(), d_perm.as<int32_t>(),
                                d_perm2.as<int32_t>(), (size_t)n, 0, end_bit, s);
  if ((st = hip_check(e, "radix_sort_pairs (tiles)"))) return st;
  if ((st = hip_check(hipStreamSynchronize(s), "tile sort"))) return st;
  d_tmp.release();
  d_perm.release();
  DevBuf d_flag, d_eid;
  if ((st = d_flag.alloc(n * 4)) || (st = d_eid.alloc(n * 4))) return st;
  hipLaunchKernelGGL(k_entry_flags, dim3(grid1(n, 256)), dim3(256), 0, s, d_key2.as<uint64_t>(), n, d_flag.as<int32_t>());
  if ((st = inclusive_scan(d_flag.as<int32_t>(), d_eid.as<int32_t>(), (size_t)n, s))) return st;
  d_flag.release();
  int32_t ne32 = 0;
  if ((st = hip_check(hipMemcpyAsync(&ne32, d_eid.as<int32_t>() + (n - 1), 4, hipMemcpyDeviceToHost, s), "D2H entries")) ||
      (st = hip_check(hipStreamSynchronize(s), "entry count")))
    return st;
  const int64_t ne = ne32;
  tp.n_entries = ne;
  DevBuf d_ep, d_eq, d_etile, d_ex, d_cnt, d_emask, d_esz, d_elbeg, d_ecoff;
  if ((st = d_ep.alloc(ne * 8 * 8)) || (st = d_eq.alloc(ne * 8 * 8)) || (st = d_etile.alloc(ne * 4)) ||
      (st = d_ex.alloc(ne * 4)) || (st = d_cnt.alloc(ne * 8)))
    return st;
  if ((st = hip_check(hipMemsetAsync(d_ep.p, 0xff, ne * 8 * 8, s), "memset ep")) ||
      (st = hip_check(hipMemsetAsync(d_eq.p, 0xff, ne * 8 * 8, s), "memset eq")))
    return st;
  hipLaunchKernelGGL(k_entry_fill_mx, dim3(grid1(n, 256)), dim3(256), 0, s, d_key2.as<uint64_t>(), d_perm2.as<int32_t>(),
                     d_eid.as<int32_t>(), in.slot, in.p, in.q, n, in.nx, d_ep.as<int64_t>(), d_eq.as<int64_t>(),
                     d_etile.as<int32_t>(), d_ex.as<int32_t>());
  d_eid.release();
  d_perm2.release();
  d_key2.release();
  if ((st = d_emask.alloc(ne * 4)) || (st = d_esz.alloc(ne * 4)) || (st = d_elbeg.alloc((ne + 1) * 8))) return st;
  hipLaunchKernelGGL(k_entry_mask_mx, dim3(grid1(ne, 256)), dim3(256), 0, s, d_ep.as<int64_t>(), d_eq.as<int64_t>(),
                     d_etile.as<int32_t>(), d_ex.as<int32_t>(), d_rdim.as<uint8_t>(), d_cdim.as<uint8_t>(),
                     d_xdim.as<uint8_t>(), ne, d_emask.as<uint32_t>(), d_esz.as<int32_t>(), d_cnt.as<int64_t>());
  if ((st = hip_check(hipMemsetAsync(d_elbeg.p, 0, 8, s), "memset lbeg"))) return st;
  if ((st = inclusive_scan(d_cnt.as<int64_t>(), d_elbeg.as<int64_t>() + 1, (size_t)ne, s))) return st;
  int64_t nl = 0;
  if ((st = hip_check(hipMemcpyAsync(&nl, d_elbeg.as<int64_t>() + ne, 8, hipMemcpyDeviceToHost, s), "D2H loads")) ||
      (st = hip_check(hipStreamSynchronize(s), "load count")))
    return st;
  tp.n_loads = nl;
  DevBuf d_lsz;
  if ((st = tp.list64.alloc(nl * 8)) || (st = d_lsz.alloc(nl * 2)) || (st = tp.listls.alloc(nl * 4))) return st;
  hipLaunchKernelGGL(k_list_fill_mx, dim3(grid1(ne, 256)), dim3(256), 0, s, d_ep.as<int64_t>(), d_eq.as<int64_t>(),
                     d_etile.as<int32_t>(), d_ex.as<int32_t>(), d_rdim.as<uint8_t>(), d_cdim.as<uint8_t>(),
                     d_xdim.as<uint8_t>(), d_elbeg.as<int64_t>(), ne, tp.list64.as<uint64_t>(), d_lsz.as<uint16_t>());
  d_ep.release();
  d_eq.release();
  // Chunks.
  DevBuf d_tebeg, d_nch;
  if ((st = d_tebeg.alloc(((size_t)in.n_tiles + 1) * 4)) || (st = d_nch.alloc((size_t)in.n_tiles * 4))) return st;
  hipLaunchKernelGGL(k_tile_ebeg, dim3(grid1((int64_t)in.n_tiles + 1, 256)), dim3(256), 0, s, d_etile.as<int32_t>(), ne,
                     in.n_tiles, d_tebeg.as<int32_t>());
  const int32_t max_entries = tp.dense ? kDenseEntries : kChunkEntries;
  hipLaunchKernelGGL((k_chunks_mx<false>), dim3(grid1(in.n_tiles, 256)), dim3(256), 0, s, d_tebeg.as<int32_t>(),
                     d_emask.as<uint32_t>(), d_esz.as<int32_t>(), d_owner.as<uint8_t>(), in.n_tiles, cap, max_entries,
                     nullptr, d_nch.as<int32_t>());
  if ((st = tp.tile_chunk.alloc(((size_t)in.n_tiles + 1) * 4))) return st;
  if ((st = hip_check(hipMemsetAsync(tp.tile_chunk.p, 0, 4, s), "memset tile_chunk"))) return st;
  if ((st = inclusive_scan(d_nch.as<int32_t>(), tp.tile_chunk.as<int32_t>() + 1, (size_t)in.n_tiles, s))) return st;
  int32_t nch = 0;
  if ((st = hip_check(hipMemcpyAsync(&nch, tp.tile_chunk.as<int32_t>() + in.n_tiles, 4, hipMemcpyDeviceToHost, s),
                      "D2H chunks")) ||
      (st = hip_check(hipStreamSynchronize(s), "chunk count")))
    return st;
  tp.n_chunks = nch;
  DevBuf d_centry;
  if ((st = d_centry.alloc(((size_t)nch + 1) * 4))) return st;
  hipLaunchKernelGGL((k_chunks_mx<true>), dim3(grid1(in.n_tiles, 256)), dim3(256), 0, s, d_tebeg.as<int32_t>(),
                     d_emask.as<uint32_t>(), d_esz.as<int32_t>(), d_owner.as<uint8_t>(), in.n_tiles, cap, max_entries,
                     tp.tile_chunk.as<int32_t>(), d_centry.as<int32_t>());
  if ((st = hip_check(hipMemcpyAsync(d_centry.as<int32_t>() + nch, &ne32, 4, hipMemcpyHostToDevice, s),
                      "H2D chunk end")))
    return st;
  if ((st = tp.chunk_lbeg.alloc(((size_t)nch + 1) * 8))) return st;
  hipLaunchKernelGGL(k_chunk_lbeg, dim3(grid1((int64_t)nch + 1, 256)), dim3(256), 0, s, d_centry.as<int32_t>(),
                     d_elbeg.as<int64_t>(), (int64_t)nch + 1, tp.chunk_lbeg.as<int64_t>());
  if ((st = d_ecoff.alloc((size_t)ne * 4))) return st;
  hipLaunchKernelGGL(k_entry_coff_mx, dim3(grid1((int64_t)nch, 256)), dim3(256), 0, s, d_centry.as<int32_t>(),
                     d_esz.as<int32_t>(), (int64_t)nch, d_ecoff.as<int32_t>());
  hipLaunchKernelGGL(k_list_lds_mx, dim3(grid1((int64_t)nch, 256)), dim3(256), 0, s, tp.chunk_lbeg.as<int64_t>(),
                     d_lsz.as<uint16_t>(), (int64_t)nch, tp.listls.as<uint32_t>());
  if (tp.dense || tp.quad) {
    // The dense and class-tile kernels read the entries and the tile block
    // shapes; no product lists.
    tp.chunk_entry = std::move(d_centry);
    tp.entry_mask = std::move(d_emask);
    tp.entry_coff = std::move(d_ecoff);
    tp.tile_rdim = std::move(d_rdim);
    tp.tile_cdim = std::move(d_cdim);
    tp.n_prod = n;
    if ((st = hip_check(hipGetLastError(), "tile builder launch"))) return st;
    return work_parts(tp.chunk_entry.as<int32_t>(), tp.tile_chunk.as<int32_t>(), tp.n_tiles, tp, s);
  }
  // Product lists.
  DevBuf d_ctile, d_np, d_pbase, d_work;
  if ((st = d_ctile.alloc((size_t)std::max(nch, 1) * 4)) || (st = d_np.alloc((size_t)std::max(nch, 1) * 8)) ||
      (st = d_pbase.alloc(((size_t)nch + 1) * 8)) || (st = d_work.alloc(((size_t)nch + 1) * 8)))
    return st;
  hipLaunchKernelGGL(k_chunk_tile, dim3(grid1(in.n_tiles, 256)), dim3(256), 0, s, tp.tile_chunk.as<int32_t>(),
                     in.n_tiles, d_ctile.as<int32_t>());
  hipLaunchKernelGGL((k_chunk_prods_mx<false>), dim3(grid1(std::max(nch, 1), 256)), dim3(256), 0, s, nch,
                     d_centry.as<int32_t>(), d_ctile.as<int32_t>(), d_emask.as<uint32_t>(), d_ecoff.as<int32_t>(),
                     d_ex.as<int32_t>(), d_owner.as<uint8_t>(), d_rdim.as<uint8_t>(), d_cdim.as<uint8_t>(),
                     d_xdim.as<uint8_t>(), d_np.as<int64_t>(), d_work.as<int64_t>() + 1, nullptr, nullptr, nullptr,
                     nullptr);
  if ((st = hip_check(hipMemsetAsync(d_pbase.p, 0, 8, s), "memset pbase"))) return st;
  if ((st = inclusive_scan(d_np.as<int64_t>(), d_pbase.as<int64_t>() + 1, (size_t)nch, s))) return st;
  if ((st = hip_check(hipMemsetAsync(d_work.p, 0, 8, s), "memset work"))) return st;
  if ((st = inclusive_scan(d_work.as<int64_t>() + 1, d_work.as<int64_t>() + 1, (size_t)nch, s))) return st;
  int64_t nprod = 0;
  if ((st = hip_check(hipMemcpyAsync(&nprod, d_pbase.as<int64_t>() + nch, 8, hipMemcpyDeviceToHost, s), "D2H products")) ||
      (st = hip_check(hipStreamSynchronize(s), "product count")))
    return st;
  tp.n_prod = nprod;
  if (nprod != n)
    return set_errorf(CQMM_ERR_STATE, "tile plan: %lld listed products for %lld triplets", (long long)nprod,
                      (long long)n);
  if ((st = tp.pstart.alloc(((size_t)nch + 1) * kWaves * 8)) || (st = tp.pcnt.alloc(((size_t)nch + 1) * kWaves * 8)) ||
      (st = tp.prod.alloc(((size_t)nprod + kWaveProducts) * 4)))
    return st;
  std::vector<int64_t> tail_start(kWaves, nprod);
  if ((st = hip_check(hipMemsetAsync(tp.pcnt.as<uint64_t>() + (size_t)nch * kWaves, 0, kWaves * 8, s), "memset pcnt")) ||
      (st = hip_check(hipMemcpyAsync(tp.pstart.as<int64_t>() + (size_t)nch * kWaves, tail_start.data(), kWaves * 8,
                                     hipMemcpyHostToDevice, s), "H2D pstart tail")) ||
      (st = hip_check(hipMemsetAsync(tp.prod.as<uint32_t>() + nprod, 0, kWaveProducts * 4, s), "memset prod tail")))
    return st;
  hipLaunchKernelGGL((k_chunk_prods_mx<true>), dim3(grid1(std::max(nch, 1), 256)), dim3(256), 0, s, nch,
                     d_centry.as<int32_t>(), d_ctile.as<int32_t>(), d_emask.as<uint32_t>(), d_ecoff.as<int32_t>(),
                     d_ex.as<int32_t>(), d_owner.as<uint8_t>(), d_rdim.as<uint8_t>(), d_cdim.as<uint8_t>(),
                     d_xdim.as<uint8_t>(), nullptr, nullptr, d_pbase.as<int64_t>(), tp.pstart.as<int64_t>(),
                     tp.pcnt.as<uint64_t>(), tp.prod.as<uint32_t>());
  if ((st = hip_check(hipGetLastError(), "mixed tile builder launch"))) return st;
  return work_parts(d_work.as<int64_t>(), tp.tile_chunk.as<int32_t>(), tp.n_tiles, tp, s);
}

}  // namespace cq
