// kx_gemm_tile.h -- one tile of a bf16 or f32 matrix product on the matrix cores, y[t][r] = sum_k x[t][k] w[r][k]: the main loop that
// the products of the hybrid decoder (kx_linear.hip) and the dense ones of Kimi-K2 (kx_dense_gemm.hip) share, and the
// hand-over between workgroups that split a tile's columns.  No counterpart in the reference, whose products are mat-vecs
// (src/kimi_exec.cu:272-298).
//
// A workgroup of WM x WN waves owns BM tokens and BN rows; wave (wm, wn) holds MI x NI blocks of 32 x 32
// (v_mfma_f32_32x32x16_bf16; for float v_mfma_f32_32x32x2_f32, products and sums in 32 bits).  Both operands are staged through LDS in blocks of 64 (32) columns by global -> LDS copies, 128-byte rows
// (whole lines: with 64-byte rows the copies cost as much a row and everything 10 to 15 % more) with the 16-byte pieces xor-ed by
// the row, so that row-per-lane reads are free of bank conflicts.
// The LDS is a ring of SLOTS half blocks -- tokens, matrix rows, tokens, ... --, two of the block that is multiplied and the others
// on their way:
//   operands of piece q + 1 are read while piece q is multiplied; between the last two pieces of a block the workgroup waits
//   for the next block (a half that was asked for behind it may still be on its way), passes its one barrier per block
//   -- behind it nobody reads the present block any more, its last operands are in registers --, asks for two more halves
//   in its place and reads the next block's first operands.
// What bounds it: a wave reads (MI + NI) KB of operands for MI NI products of 32 cycles, and LDS gives a CU about 128 bytes a
// cycle: waves of 2 x 2 blocks are at that limit with the copies' writes, and every wave asks for its copies between products.  Where
// the columns are long enough the tiles of kx_gemm_turns.h are sooner, 256 x 256 throughout (2048 x 7168 x 8192 231 us as this loop, 171).
// A fifth slot, which keeps the queue of copies from running dry, is worth 2 to 8 % to two workgroups per CU with few tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "kx_arrive.h"
#include "kx_lds_copy.h"
#include "kx_tile_share.h"

namespace kxtile {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// 16 bytes of a row, as a lane holds them: lanes 0-31 have piece 2 q of their row, lanes 32-63 piece 2 q + 1; both operands
// alike, so that it does not matter which of the columns meet in one instruction
template <class T> struct Piece;
template <> struct Piece<uint16_t> {
  typedef bf16x8 Type;
  static __device__ __forceinline__ f32x16 multiply(Type x, Type w, f32x16 acc) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, w, acc, 0, 0, 0); }
};
template <> struct Piece<float> {
  typedef f32x4 Type;
  static __device__ __forceinline__ f32x16 multiply(Type x, Type w, f32x16 acc) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], w[e], acc, 0, 0, 0);
    return acc;
  }
};

template <class T, int WM_, int WN_, int MI_, int NI_, int SLOTS_>
struct Tile {
  typedef f32x16 Block;
  static constexpr int V = 16, SIDE = 32;
  typedef Block Sums[MI_][NI_];
  static constexpr int COLS = 128 / sizeof(T);  // columns of a block
  static constexpr int SLOTS = SLOTS_, WM = WM_, WN = WN_, MI = MI_, NI = NI_, WAVES = WM * WN, THREADS = WAVES * 64;
  static constexpr int BM = WM * MI * 32, BN = WN * NI * 32, SLOT = (BM > BN ? BM : BN) * 128, LDS = SLOTS * SLOT;
  static constexpr int PAIR = (BM + BN) * 128, LEAST_LDS = SLOTS == 4 ? 2 * PAIR : LDS;  // with LDS a CU has two workgroups of four waves, with less of it three
  static constexpr int WAVES_PER_SIMD = MI * NI >= 16 ? 1 : 2;
  static constexpr int CX = BM / 8 / WAVES, CW = BN / 8 / WAVES;  // copy instructions of a wave for half a block, 8 rows each
  static constexpr size_t PART = (size_t)BM * BN;          // floats of a part's sums
  static_assert(SLOTS == 4 || SLOTS == 5, "two blocks, and half of a third");
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "the copies of a block are spread evenly over the waves");

  // Where a slot begins: with four, tokens have the even ones and the matrix the odd ones; with five each takes every one in turn.
  static __device__ __forceinline__ int at(int slot) { return SLOTS == 4 ? (slot >> 1) * PAIR + (slot & 1) * (BM * 128) : slot * SLOT; }

  // Columns COLS kb0 .. COLS kb1 - 1 (kb0 < kb1).  row(r): where staged row r begins, tokens 0 .. BM - 1, then BN rows of the
  // matrix; every row has to be readable, what a row past the end holds only reaches sums that are not used.
  template <class Row>
  static __device__ __forceinline__ void run(uint8_t *lds, int kb0, int kb1, Row row, f32x16 (&acc)[MI][NI]) {
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, h = lane >> 5, sub = lane >> 3, n = kb1 - kb0;
    const T *src[CX + CW];
#pragma unroll
    for (int i = 0; i < CX + CW; ++i)
      src[i] = row(i < CX ? (i * WAVES + wave) * 8 + sub : BM + ((i - CX) * WAVES + wave) * 8 + sub) + kb0 * COLS + ((lane & 7) ^ sub) * (COLS / 8);
    auto copy_x = [&](int b, int slot) {
#pragma unroll
      for (int i = 0; i < CX; ++i) kx_copy16_to_lds(src[i] + b * COLS, __builtin_amdgcn_readfirstlane(lds0 + at(slot) + (i * WAVES + wave) * 1024));
    };
    auto copy_w = [&](int b, int slot) {
#pragma unroll
      for (int i = 0; i < CW; ++i) kx_copy16_to_lds(src[CX + i] + b * COLS, __builtin_amdgcn_readfirstlane(lds0 + at(slot) + (i * WAVES + wave) * 1024));
    };
    struct Frag {
      typename Piece<T>::Type x[MI], w[NI];
    };
    const uint8_t *const xs = lds + (wm * MI * 32 + lr) * 128, *const ws = lds + (wn * NI * 32 + lr) * 128;
    int sx = 0, sw = 1;  // slots of the present block
    auto next = [](int slot) { return slot >= SLOTS - 2 ? slot - (SLOTS - 2) : slot + 2; };
    auto read = [&](Frag &f, int q) {
      const int p = ((2 * q + h) ^ (lr & 7)) * 16;
#pragma unroll
      for (int i = 0; i < MI; ++i) f.x[i] = *(const typename Piece<T>::Type *)(xs + at(sx) + p + i * 4096);
#pragma unroll
      for (int j = 0; j < NI; ++j) f.w[j] = *(const typename Piece<T>::Type *)(ws + at(sw) + p + j * 4096);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Frag &f) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = Piece<T>::multiply(f.x[i], f.w[j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    Frag f0, f1;
    copy_x(0, 0);
    copy_w(0, 1);
    if (n > 1) {
      copy_x(1, 2);
      copy_w(1, 3);
    }
    if (SLOTS == 5 && n > 2) {
      copy_x(2, 4);
      kx_wait_copies<CX + CW + CX>();
    } else if (n > 1) {
      kx_wait_copies<CX + CW>();
    } else {
      kx_wait_copies<0>();
    }
    kx_lds_barrier();
    read(f0, 0);
    for (int b = 0; b < n; ++b) {
      read(f1, 1);
      multiply(f0);
      read(f0, 2);
      multiply(f1);
      read(f1, 3);
      multiply(f0);
      if (b + 1 < n) {
        if (SLOTS == 5 && b + 2 < n) kx_wait_copies<CX>();  // the tokens of block b + 2 are behind block b + 1
        else kx_wait_copies<0>();
        kx_lds_barrier();
        if (SLOTS == 5) {
          if (b + 2 < n) copy_w(b + 2, sx);
          if (b + 3 < n) copy_x(b + 3, sw);
        } else if (b + 2 < n) {
          copy_x(b + 2, sx);
          copy_w(b + 2, sw);
        }
        sx = next(sx);
        sw = next(sw);
        read(f0, 0);
      }
      multiply(f1);
    }
  }
  // Element v of block (i, j) of the present lane: matrix row col(j) and token row(i, v) of the tile.
  static __device__ __forceinline__ int col(int j) { return (((int)threadIdx.x >> 6) % WN * NI + j) * 32 + (threadIdx.x & 31); }
  static __device__ __forceinline__ int row(int i, int v) {
    return (((int)threadIdx.x >> 6) / WN * MI + i) * 32 + 8 * (v >> 2) + 4 * (threadIdx.x >> 5 & 1) + (v & 3);
  }

};

// The sums of `parts` workgroups that hold a part of the columns each, added in the parts' order by the one that arrives last
// (kx_arrive.h); false for the others.  part: parts * PART floats of this tile; arrived: its counter.
template <class TL>
__device__ __forceinline__ bool gather(uint8_t *lds, typename TL::Sums &acc, float *part, int *arrived, int parts, int p) {
  int &last = *(int *)lds;  // behind the barrier below nobody reads operands any more
  uint64_t *at = (uint64_t *)part;
  constexpr size_t PER = TL::PART / 2;
  constexpr int H = TL::V / 2, RUN = 8 / H;  // pairs of a block; blocks whose parts are asked for together
#pragma unroll
  for (int i = 0; i < TL::MI; ++i)
#pragma unroll
    for (int j = 0; j < TL::NI; ++j)
#pragma unroll
      for (int q = 0; q < H; ++q) {
        const float a = acc[i][j][2 * q], b = acc[i][j][2 * q + 1];
        kx_arrive_store(at + p * PER + ((i * TL::NI + j) * H + q) * TL::THREADS + threadIdx.x,
                        (uint64_t)__builtin_bit_cast(uint32_t, a) | (uint64_t)__builtin_bit_cast(uint32_t, b) << 32);
      }
  kx_arrive_writes_done();
  __syncthreads();
  if (threadIdx.x == 0) last = kx_arrive_is_last(arrived, parts);
  __syncthreads();
  if (!last) return false;
  if (threadIdx.x == 0) kx_arrive_reset(arrived);
#pragma unroll
  for (int i = 0; i < TL::MI; ++i)
#pragma unroll
    for (int j0 = 0; j0 < TL::NI; j0 += RUN)
      for (int s = 0; s < parts; ++s) {
        uint64_t y[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) y[q] = kx_arrive_load(at + s * PER + ((i * TL::NI + j0) * H + q) * TL::THREADS + threadIdx.x);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float a = __builtin_bit_cast(float, (uint32_t)y[q]), b = __builtin_bit_cast(float, (uint32_t)(y[q] >> 32));
          auto &block = acc[i][j0 + q / H];
          const int v = 2 * (q % H);
          block[v] = s ? block[v] + a : a;
          block[v + 1] = s ? block[v + 1] + b : b;
        }
      }
  return true;
}

}  // namespace kxtile
#include "kx_gemm_turns.h"
namespace kxtile {

// Workgroup id -> work item: consecutive ids go to the chip's eight dies in turn, each with its own L2, so every die takes a
// run of consecutive items, which share rows of tokens and of the matrix.
__device__ __forceinline__ int item_of(int id, int n) {
  const int die = id & 7, q = n >> 3, r = n & 7;
  return die * q + min(die, r) + (id >> 3);
}

// Where part `part` of `parts` of `blocks` blocks begins.  In 32 bits (the products that fit a device stay below 2^31): two divisions
// in 64 bits cost a workgroup 0.3 us, 2 % of a product of 16 blocks.
__device__ __forceinline__ int cut(int blocks, int part, int parts) { return (uint32_t)blocks * part / (uint32_t)parts; }

typedef Turns<false> Large;                    // 256 x 256, 8 waves, a CU each
typedef Turns<true> Twin;                      // 128 x 128, 8 waves, a CU each
typedef Tile<uint16_t, 2, 2, 2, 2, 5> Medium;  // 128 x 128, 4 waves, two workgroups per CU

struct Place {
  int tile, part, of;
};
__device__ __forceinline__ Place place_of(int id, int tiles, Share s) {
  const int rest = tiles - s.whole, n = rest * s.parts;
  if (id >= n) return {item_of(id - n, s.whole), 0, 1};
  const int q = item_of(id, n), part = q / rest;
  return {s.whole + q - part * rest, part, s.parts};
}
// The 32-bit tile: 64 x 128, 4 waves, two workgroups per CU.  A piece is 4 products of 64 cycles, so LDS and copies are far
// from their limits and what counts is that every SIMD has a wave as long as any: a CU takes 0.97 us per tile and block of 32 columns
// whether it has one workgroup or two.  777 x 8192 x 1024, 832 tiles, takes 142 us whole (181 with two waves a
// workgroup); 777 x 1024 x 4096 140 us with 104 tiles, 79 with their columns in four parts, 11 x 5120 x 1024 38 and 19.  On the
// vector ALU (64 x 64, 4 x 4 a thread) the first, with its activation, took 260 us and was a little further from the 64-bit result.
typedef Tile<float, 2, 2, 1, 2, 4> Single;

static_assert(Large::BM == LARGE.tokens && Large::BN == LARGE.rows && Medium::BM == MEDIUM.tokens && Medium::BN == MEDIUM.rows && Twin::BM == MEDIUM.tokens && Twin::BN == MEDIUM.rows &&
              Single::BM == SINGLE.tokens && Single::BN == SINGLE.rows, "the rules count other tiles");

}  // namespace kxtile
