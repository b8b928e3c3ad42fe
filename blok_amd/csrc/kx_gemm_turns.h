// kx_gemm_turns.h -- tiles of a bf16 matrix product whose two groups of four waves take turns: while one multiplies (its operands of a
// block of 64 columns are all in registers), the other reads its next operands from LDS and asks for copies.  Included by
// kx_gemm_tile.h, whose rows, layout of a staged row and hand-over of parts these tiles share.  No counterpart in the reference, whose
// products are mat-vecs (src/kimi_exec.cu:272-298).
//
// Every SIMD has a wave of each group, so its matrix core always has one wave that issues nothing but products.  That is what counts:
// a copy holds up the wave that asks for it until the CU's one path for addresses has taken it, 26 cycles each and up to
// four waves in a queue, and a wave that asks for copies between its products leaves the matrix core idle meanwhile (2048 x 7168 x 8192,
// cycles per block of a 256 x 256 tile on a CU, of which 2048 are products: 3300 with a copy between every eight products,
// 2330 with all copies in the reading turns; the products alone 2080).  A turn ends with the workgroup's barrier.
//
//   Whole (256 x 256): both groups multiply every block, group g the matrix rows of half g; wave w of a group has 64 tokens x 128 rows.
//     Operands are 24 x 16 bytes a lane, sums 128 registers.  Group 0 copies the tokens, group 1 the matrix:
//       turn 2 b:     group 0 reads block b and asks for the tokens of block b + 1 (their place: the tokens of b - 1, read for the last
//                     time in turn 2 b - 1); group 1 multiplies block b - 1
//       turn 2 b + 1: group 1 reads block b and asks for its half of the matrix of block b + 1 (place of b - 1, its own) and for group
//                     0's half of b + 2 (place of b, which group 0 read in turn 2 b); group 0 multiplies block b
//   Twin (128 x 128): group g has the blocks of that parity to itself, wave w of a group 64 x 64; the groups' sums meet in LDS
//     and each finishes half of the tile.  Each copies for the other, into the place of the block that was read a turn ago:
//       turn 2 i:     group 0 reads block 2 i, asks for 2 i + 3;  turn 2 i + 1: group 1 reads block 2 i + 1, asks for 2 i + 4
//     One workgroup per CU takes 800 cycles a block where one of four waves (Medium) took 1400 and two of them 1300 each.
//
// v_mfma_f32_16x16x32_bf16: it reads and writes half the sums that the 32 x 32 x 16 form does for as many products, and the chip, which
// lowers its clock under load, holds 2.2 GHz instead of 1.85 with nothing but products running.
#pragma once

namespace kxtile {

// 16 x 16 blocks of sums: element v of block (i, j) is matrix row col(j), token row(i, v).  RI: blocks of tokens of a wave while it
// multiplies; with fewer than four, tiles of 64 RI x 256 for the ends of lists of rows.
template <bool TWIN, int RI = 4>
struct Turns {
  typedef f32x4 Block;
  static constexpr int V = 4, SIDE = 16;
  static constexpr int COLS = 64, THREADS = 512, WAVES_PER_SIMD = 2;
  static_assert(!TWIN || RI == 4, "twin tiles are 128 x 128");
  static constexpr int BM = TWIN ? 128 : 64 * RI, BN = TWIN ? 128 : 256;
  static constexpr int MI = TWIN ? 2 : RI, NI = TWIN ? 4 : 8;      // blocks of a wave when the products are done
  static constexpr int XS = BM * 128, WS = BN * 128, LDS = (TWIN ? 4 : 2) * (XS + WS);  // bytes of a block's tokens, of its rows; four blocks, two
  static constexpr size_t PART = (size_t)BM * BN;
  typedef Block Sums[MI][NI];

  static __device__ __forceinline__ int group() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 8); }
  static __device__ __forceinline__ int member() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6 & 3); }
  static __device__ __forceinline__ int col(int j) { return (TWIN ? (member() & 1) * 64 : group() * 128) + j * 16 + (threadIdx.x & 15); }
  static __device__ __forceinline__ int row(int i, int v) {
    return (TWIN ? (member() >> 1) * 64 + group() * 32 : member() * (16 * RI)) + i * 16 + 4 * (threadIdx.x >> 4 & 3) + v;
  }

  static __device__ __forceinline__ void turn() {
    kx_lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  // as Tile::run
  template <class Row>
  static __device__ __forceinline__ void run(uint8_t *lds, int kb0, int kb1, Row row, Sums &out) {
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const int lane = threadIdx.x & 63, sub = lane >> 3, g = group(), me = member(), lr = lane & 15, kq = lane >> 4, n = kb1 - kb0;
    constexpr int RJ = TWIN ? 4 : 8;        // blocks of rows of a wave while it multiplies
    constexpr int XW = TWIN ? XS : 2 * XS;  // the matrix lies behind the tokens: of the same block, of both
    // the up to eight copies of a wave per block, eight rows each.  Whole: tokens or matrix; Twin: four of the tokens and four of the matrix
    const uint16_t *src[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = (i * 4 + me) * 8 + sub;
      src[i] = row(TWIN ? r : g ? BM + r : RI < 4 ? min(r, BM - 1) : r) + kb0 * COLS + ((lane & 7) ^ sub) * 8;
    }
    auto copy = [&](int b, int base, int i) { kx_copy16_to_lds(src[i] + b * COLS, __builtin_amdgcn_readfirstlane(lds0 + base + (i * 4 + me) * 1024)); };
    const uint8_t *const xs = lds + ((TWIN ? (me >> 1) * 64 : me * (16 * RI)) + lr) * 128, *const ws = lds + XW + ((TWIN ? (me & 1) * 64 : g * 128) + lr) * 128;
    const int p[2] = {(kq ^ (lr & 7)) * 16, ((4 + kq) ^ (lr & 7)) * 16};  // the lane's piece of a row, columns 0 to 31 and 32 to 63
    Block acc[RI][RJ];
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
      for (int j = 0; j < RJ; ++j) acc[i][j] = Block{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 x[2][RI], w[2][RJ];
    auto read = [&](int q, int xo, int wo) {
#pragma unroll
      for (int i = 0; i < RI; ++i) x[q][i] = *(const bf16x8 *)(xs + xo + p[q] + i * 2048);
#pragma unroll
      for (int j = 0; j < RJ; ++j) w[q][j] = *(const bf16x8 *)(ws + wo + p[q] + j * 2048);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&]() {
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
          for (int j = 0; j < RJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[q][i], w[q][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!TWIN) {
      constexpr int HALF = BN / 2 * 128;  // of a block of the matrix
      if (g == 0) {
#pragma unroll
        for (int i = 0; i < 2 * RI; ++i) copy(0, 0, i);
        kx_wait_copies<0>();
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) copy(0, XW, i);
        if (n > 1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) copy(1, XW + WS, i);
          kx_wait_copies<4>();
        } else {
          kx_wait_copies<0>();
        }
      }
      static_assert(HALF == 4 * 4 * 1024, "four copies of a wave are a group's half");
      turn();
      if (g == 1) turn();
      for (int b = 0; b < n; ++b) {
        const int at = b & 1, other = at ^ 1;
        read(0, at * XS, at * WS);
        if (b + 1 < n) {
          if (g == 0) {
#pragma unroll
            for (int i = 0; i < RI; ++i) copy(b + 1, other * XS, i);
          } else {
#pragma unroll
            for (int i = 4; i < 8; ++i) copy(b + 1, XW + other * WS, i);
          }
        }
        read(1, at * XS, at * WS);
        if (g == 0) {
          if (b + 1 < n)
#pragma unroll
            for (int i = RI; i < 2 * RI; ++i) copy(b + 1, other * XS, i);
        } else if (b + 2 < n) {
#pragma unroll
          for (int i = 0; i < 4; ++i) copy(b + 2, XW + at * WS, i);
          kx_wait_copies<8>();  // group 0's half of block b + 1, asked for a block ago, has come
        } else {
          kx_wait_copies<0>();
        }
        turn();
        multiply();
        if (g == 1 && b + 2 < n) kx_wait_copies<4>();  // its own half of block b + 1
        else kx_wait_copies<0>();
        turn();
      }
      if (g == 0) turn();
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) out[i][j] = acc[i][j];
    } else {
      auto ask = [&](int b, int q) {
#pragma unroll
        for (int i = 4 * q; i < 4 * q + 4; ++i) copy(b, (b & 3) * 2 * XS, i);
      };
      if (g == 0) {
        if (n > 1) ask(1, 0), ask(1, 1);
      } else {
        ask(0, 0), ask(0, 1);
        if (n > 2) {
          ask(2, 0), ask(2, 1);
          kx_wait_copies<8>();
        } else {
          kx_wait_copies<0>();
        }
      }
      turn();
      if (g == 1) turn();
      for (int b = g; b < n + g; b += 2) {  // as many turns for group 1, whose last block may be missing
        const int at = (b & 3) * 2 * XS;
        if (b < n) {
          read(0, at, at);
          if (b + 3 < n) ask(b + 3, 0);
          read(1, at, at);
          if (b + 3 < n) ask(b + 3, 1);
        }
        if (b + 3 < n) kx_wait_copies<8>();  // block b + 1 has come
        else kx_wait_copies<0>();
        turn();
        if (b < n) multiply();
        turn();
      }
      if (g == 0) turn();
      // behind the last turn nobody reads operands any more
      Block *const give = (Block *)lds + (g * 4 + me) * (MI * NI * 64) + lane, *const take = (Block *)lds + ((g ^ 1) * 4 + me) * (MI * NI * 64) + lane;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          out[i][j] = g ? acc[i + 2][j] : acc[i][j];
          give[(i * NI + j) * 64] = g ? acc[i][j] : acc[i + 2][j];
        }
      turn();
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const Block o = take[(i * NI + j) * 64];
#pragma unroll
          for (int v = 0; v < V; ++v) out[i][j][v] += o[v];
        }
      __syncthreads();  // the hand-over of parts uses the LDS again
    }
  }
};

}  // namespace kxtile
