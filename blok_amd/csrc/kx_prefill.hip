// kx_prefill.hip -- W4A16 grouped GEMM for prefill chunks through one MoE layer.
//
// The reference has no batched prefill: it runs one decode step per prompt token
// (src/kimi_exec.cu:886) and, inside it, the per-expert loops at :845-870.  For a
// chunk of T tokens this file computes the same per-token quantities -- gate/up
// projections with SwiGLU (:853-862), down projection (:863-869), the routed
// combine (:868,:871), the shared expert (:872-875) and the residual add (:877) --
// with the tokens of each expert gathered into one GEMM.
//
// Per workgroup (8 waves) and tile: one expert, 256 weight rows (of a prompt's down product 512), up to 128 of the
// expert's tokens.  Wave w owns weight rows 32 w .. +31 for all 128 tokens
// (fp32 accumulators of v_mfma_f32_32x32x16_bf16).  Per K step of 64 columns:
//  * INT4 weights reach the lanes through LDS as packed words: for every two K steps the
//    64-byte runs of the 256 rows (of both matrices, or of both halves of the 512) are copied by global -> LDS loads, which
//    take no registers and use every byte they fetch, into a ring of two stages; lane
//    (r, h) = (lane % 32, lane / 32) reads the 16 bytes of row r that hold columns 32 h .. +31
//    of the step -- one quantization group, four packed words -- and dequantizes word j to
//    the reference's values, w = bf((n-8)*scale) (:311-312), which is exactly the B operand
//    of the step's j-th MFMA when that MFMA contracts over columns {8 j .. +7} and
//    {32 + 8 j .. +7} (the contraction order within a step is free, the activation operand
//    uses the same columns).  The 16-byte pieces of a row are stored xor-swizzled by the row
//    so that the lanes' reads are free of bank conflicts.  Group scales are copied to LDS
//    the same way, sixteen K steps at a time: 64 bytes per row and matrix, a whole sector of the row (blocks of
//    eight steps fetched half of every sector twice);
//  * the gathered activation rows go through a double-buffered LDS tile, one barrier per step, copied global -> LDS
//    as well (128-byte rows, pieces xor-swizzled by the row).
//
// Dequant without integer conversion: (w & 0x000F000F) | 0x64006400 is the f16 pair
// (1024+n0, 1024+n4), (w & 0x00F000F0) | 0x64006400 is (1024+16 n1, 1024+16 n5), w >> 8 gives
// n2,n6,n3,n7 the same way; fma(f16, s, -1032 s) = (n-8) s and fma(f16, s/16, -72 s) = (n-8) s
// are exact in fp32 (4-bit times 8-bit significands), and one v_cvt_pk_bf16_f32 rounds two of
// them to nearest-even.
//
// MFMA's internal summation order is not documented, so this path is held to the
// max-rel 1e-2 bar and is never used for the token-identity runs.
#include <algorithm>
#include <atomic>
#include "kx_common.h"
#include "kx_lds_copy.h"
#include "kx_dense.h"
#include "kx_math.h"

#include <type_traits>

namespace {

typedef __bf16 kx_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 kx_bf16x2 __attribute__((ext_vector_type(2)));
typedef float kx_f32x2 __attribute__((ext_vector_type(2)));
typedef float kx_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 kx_h2 __attribute__((ext_vector_type(2)));

constexpr int BN = 256, BK = 64, XT = 128 * BK;  // XT: elements of an activation tile
constexpr int W_STAGE = BN * 64;               // bytes of one matrix's packed words for two K steps
constexpr int SC_BLOCK = 16;                   // K steps per staged block of group scales
constexpr int SC_STRIDE = SC_BLOCK * 4;        // bytes per (row, matrix) of a block: 32 bf16, one 64-byte sector of the row

struct PfArgs {
  const uint32_t *w0, *w1;      // packed i32 [E][N][K/8]
  const uint16_t *s0, *s1;      // bf16 scales [E][N][K/32]
  const uint16_t *x;            // bf16 activation rows of K
  uint16_t *out;                // bf16 [pairs][N]
  const int4 *tiles;            // {expert, first, last, _}: tiles of up to 128 pairs, or experts
  const int *n_tiles;           // how many; nullptr: tiles_max
  int tiles_max, cnt_lo;        // records with fewer pairs are left to another launch
  int row_tiles;                // of 256 rows, WIDE 512
  const int *pairs;             // pair ids sorted by expert
  int N, K, x_div;              // activation row = pair / x_div
  size_t expert_w, expert_s;    // elements between experts (words; scales)
};

__device__ __forceinline__ uint32_t pf_and_or(uint32_t a, uint32_t mask, uint32_t magic) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(magic));
  return r;
}
__device__ __forceinline__ uint32_t pf_pack(float lo, float hi) {
  kx_f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, kx_bf16x2));
}

// The INT4 kernels keep copies and loads in flight across barriers and LDS accesses, and say themselves when
// one has to have landed.  The compiler would not let them: it completes every global -> LDS copy in flight
// (s_waitcnt vmcnt(0)) in front of an LDS access it cannot tell from the copy's target and in front of every
// fenced barrier, and loads complete in order, so a wait for a plain load it issued waits for the copies too.
// Hence: weights and activations both reach LDS by copies issued from inline asm (unknown to the compiler), the
// barrier has no fence, and the waits are explicit and counted.
__device__ __forceinline__ void pf_copy16_to_lds(const void *src, uint32_t lds_base) {
  kx_copy16_to_lds(src, __builtin_amdgcn_readfirstlane(lds_base));
}
template <int N>
__device__ __forceinline__ void pf_wait_copies() { kx_wait_copies<N>(); }
__device__ __forceinline__ void pf_barrier() { kx_lds_barrier(); }

// dequantize one packed word (8 weights) to 8 bf16, columns ascending
__device__ __forceinline__ kx_bf16x8 dequant_word(uint32_t w, float sc, float sc16, float c0, float c1, uint32_t magic) {
  const uint32_t w8 = w >> 8;
  const kx_h2 a = __builtin_bit_cast(kx_h2, pf_and_or(w, 0x000F000Fu, magic));   // n0, n4
  const kx_h2 b = __builtin_bit_cast(kx_h2, pf_and_or(w, 0x00F000F0u, magic));   // 16 n1, 16 n5
  const kx_h2 c = __builtin_bit_cast(kx_h2, pf_and_or(w8, 0x000F000Fu, magic));  // n2, n6
  const kx_h2 d = __builtin_bit_cast(kx_h2, pf_and_or(w8, 0x00F000F0u, magic));  // 16 n3, 16 n7
  const float f0 = __builtin_fmaf((float)a.x, sc, c0), f4 = __builtin_fmaf((float)a.y, sc, c0);
  const float f1 = __builtin_fmaf((float)b.x, sc16, c1), f5 = __builtin_fmaf((float)b.y, sc16, c1);
  const float f2 = __builtin_fmaf((float)c.x, sc, c0), f6 = __builtin_fmaf((float)c.y, sc, c0);
  const float f3 = __builtin_fmaf((float)d.x, sc16, c1), f7 = __builtin_fmaf((float)d.y, sc16, c1);
  return __builtin_bit_cast(kx_bf16x8, make_uint4(pf_pack(f0, f1), pf_pack(f2, f3), pf_pack(f4, f5), pf_pack(f6, f7)));
}

// The tiles of up to 128 pairs of every group with at least cnt_lo pairs, {expert, first, last, -}, those of four 32-token
// blocks first and those of one last (a last round of the short ones ends sooner): tiles of a group in turn, so that workgroups which run at
// the same time read the same weights, through one L2 where the row tiles are a multiple of 8 (gate and up of 2048 rows), through several
// where they are not (14 of a down product with 7168).  One workgroup, a thread per group; n_tiles[0]: how many.
__global__ void __launch_bounds__(1024) grouped_tiles_k(const int4 *__restrict__ work, int n_slots, int cnt_lo, int4 *__restrict__ tiles, int *__restrict__ n_tiles) {
  __shared__ int4 sum[2][1024];
  const int i = threadIdx.x;
  const int4 w = i < n_slots ? work[i] : make_int4(-1, 0, 0, 0);
  const int cnt = w.x >= 0 && w.z - w.y >= cnt_lo ? w.z - w.y : 0;
  const int rest = cnt & 127, cls = rest ? (rest + 31) >> 5 : 0, full = (cnt >> 7) + (cls == 4);
  const int4 own = make_int4(full, cls == 3, cls == 2, cls == 1);
  int cur = 0;
  sum[0][i] = own;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1, cur ^= 1) {  // inclusive sums
    int4 v = sum[cur][i];
    if (i >= d) {
      const int4 u = sum[cur][i - d];
      v = make_int4(v.x + u.x, v.y + u.y, v.z + u.z, v.w + u.w);
    }
    sum[cur ^ 1][i] = v;
    __syncthreads();
  }
  const int4 at = sum[cur][i], all = sum[cur][1023];
  for (int t = 0; t < full; ++t) tiles[at.x - full + t] = make_int4(w.x, w.y + t * 128, min(w.y + t * 128 + 128, w.z), 0);
  const int last = cls == 3 ? all.x + at.y : cls == 2 ? all.x + all.y + at.z : all.x + all.y + all.z + at.w;
  if (cls >= 1 && cls <= 3) tiles[last - 1] = make_int4(w.x, w.z - rest, w.z, 0);
  if (i == 0) *n_tiles = all.x + all.y + all.z + all.w;
}

// 8 waves per workgroup, 32 weight rows each: of two matrices (DUAL), of 256 rows of one (SINGLE), or twice 256 of them (WIDE).  An activation
// operand meets two weight operands in DUAL and WIDE: with one a wave reads a KB of LDS for every product of 32 cycles, all of
// LDS' rate.  7168 rows of 2048 columns, 8 experts of 2048 tokens: 0.80 ms as SINGLE with a workgroup per possible tile, 0.61 as WIDE over a
// list.  Records without a list are SINGLE (a few tokens per expert, beside other kernels): twice as many workgroups, of less LDS.
enum { GG_SINGLE = 0, GG_WIDE = 1, GG_DUAL = 2 };
template <int MODE>
__global__ void __launch_bounds__(512, 1) grouped_gemm_k(PfArgs a) {
  constexpr bool DUAL = MODE == GG_DUAL;
  constexpr int MATS = MODE == GG_SINGLE ? 1 : 2;
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_lds[];
  uint16_t *xs_lds = (uint16_t *)pf_lds;                 // two activation tiles
  uint8_t *w_ring = pf_lds + 2 * XT * 2;                 // [2 stages][MATS][256 rows][4 pieces of 16 B]
  uint8_t *sc_lds = w_ring + 2 * MATS * W_STAGE;         // [2 blocks][MATS][256 rows][SC_STRIDE]
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)w_ring;  // LDS address of the ring
  const uint32_t sc0 = ring0 + 2 * MATS * W_STAGE;                                                  // of the scale blocks
  const uint32_t xs0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)pf_lds;    // and of the activation tiles
  const int nk = a.K / BK;
  const int items = (a.n_tiles ? *a.n_tiles : a.tiles_max) * a.row_tiles;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int n0 = item % a.row_tiles * (MODE == GG_WIDE ? 2 * BN : BN);
    const int4 wk = a.tiles[item / a.row_tiles];
    const int e = __builtin_amdgcn_readfirstlane(wk.x);
    const int p_begin = __builtin_amdgcn_readfirstlane(wk.y), p_end = __builtin_amdgcn_readfirstlane(wk.z);
    if (e < 0 || p_end - p_begin < a.cnt_lo) continue;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what follows from it is not worked out, and spilled, in front of the loop
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 31, lh = lane >> 5;
    const int trow = wave * 32 + lr;                       // this lane's weight row within the tile
    uint32_t magic;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    // row r of matrix m: of the second matrix, or 256 rows further down the same one
    auto row_of = [&](int m, int r) { return min(n0 + r + (DUAL ? 0 : m * BN), a.N - 1); };
    // global -> LDS copies of this wave for one stage: MATS*2 instructions of 64 pieces
    const uint32_t *dma_src[MATS * 2];
    int dma_dst[MATS * 2];
#pragma unroll
    for (int u = 0; u < MATS * 2; ++u) {
      const int g = (wave * MATS * 2 + u) * 64 + lane;     // piece index over [MATS][256 rows][4]
      const int m = g >> 10, sl = g & 1023, row = sl >> 2, ps = sl & 3;
      const int p = ps ^ ((row >> 2) & 3);                 // the piece of the row that lives in slot ps
      dma_src[u] = (DUAL && m ? a.w1 : a.w0) + (size_t)e * a.expert_w + (size_t)row_of(m, row) * (a.K >> 3) + p * 4;
      dma_dst[u] = (wave * MATS * 2 + u) * 1024;           // byte offset within a stage, the same for the whole wave
    }
    auto dma_stage = [&](int ss) {  // packed words of K steps 2 ss, 2 ss + 1 into stage ss % 2
#pragma unroll
      for (int u = 0; u < MATS * 2; ++u) pf_copy16_to_lds(dma_src[u] + ss * 16, ring0 + (ss & 1) * MATS * W_STAGE + dma_dst[u]);
    };
    // group scales: blocks of SC_BLOCK K steps, 64 bytes per row and matrix -- whole sectors -- copied global -> LDS.
    // Instruction c = wave * 2 MATS + i covers pieces 64 c .. +63 of [MATS][256 rows][4 slots]; slot s of row r holds
    // piece s ^ ((r / 2) % 4): a wave reads one 2-byte scale per row at the same offset of 32 consecutive rows, and with
    // the pieces in place (64-byte rows) those fall into two banks; xor-ed by the row they fall into eight.  A last block of
    // half the steps (K / 64 an odd multiple of 8) repeats its two pieces, the copies land in slots that are never read.
    const uint16_t *sc_src[MATS * 2];
#pragma unroll
    for (int i = 0; i < MATS * 2; ++i) {
      const int c = wave * MATS * 2 + i, m = c >> 4, row = (c & 15) * 16 + (lane >> 2);
      sc_src[i] = (DUAL && m ? a.s1 : a.s0) + (size_t)e * a.expert_s + (size_t)row_of(m, row) * (a.K >> 5);
    }
    auto copy_scales = [&](int blk) {
      const int left = (nk - blk * SC_BLOCK) >> 2;  // 16-byte pieces of the row from this block on: 2 or at least 4
      const int piece = min((lane & 3) ^ ((lane >> 3) & 3), left - 1);  // row = 16 (c % 16) + lane / 4
#pragma unroll
      for (int i = 0; i < MATS * 2; ++i)
        pf_copy16_to_lds(sc_src[i] + blk * (SC_BLOCK * 2) + piece * 8, sc0 + (blk & 1) * (BN * MATS * SC_STRIDE) + (wave * MATS * 2 + i) * 1024);
    };
    // Once for a tile of the list.  An expert's record is no tile: where a token has fewer candidates than choices (the others' bias
    // -inf, logits that are no numbers) expert 0 stands for the missing ones, and has more pairs than there are tokens.
    for (int m0 = p_begin; m0 < p_end; m0 += 128) {
      const int nb = (p_end - m0 + 31) >> 5;  // 32-token blocks that hold tokens, of which a tile takes four
      // The activation tile goes global -> LDS like the weights.  A row of a K step is 128 B = 8 pieces;
      // copy instruction ii covers rows 8 ii .. 8 ii + 7, slot (row, p') holding piece p' ^ ((row >> 1) & 7), so that
      // the row-per-lane operand reads are free of bank conflicts without padding.  Rows past the expert's tokens
      // read pair 0: they only feed accumulator rows that are never stored.
      constexpr int XCMAX = 2;  // copy instructions per wave and K step at 128 tokens
      const uint16_t *xc_src[XCMAX];
      int xc_dst[XCMAX];
#pragma unroll
      for (int q = 0; q < XCMAX; ++q) {
        const int ii = wave + 8 * q;
        const int slot = ii * 64 + lane, row = slot >> 3, piece = (slot & 7) ^ ((row >> 1) & 7);
        const int pi = m0 + row;
        const int pair = pi < p_end ? a.pairs[pi] : 0;
        xc_src[q] = a.x + (size_t)(pair / a.x_div) * a.K + piece * 8;
        xc_dst[q] = ii * 1024;
      }

      // the tile with NB token blocks, NB a compile-time constant so that the K loop has no branches
      auto run = [&](auto nb_c) {
        constexpr int NB = decltype(nb_c)::value;
        kx_f32x16 acc[MATS][NB];
#pragma unroll
        for (int m = 0; m < MATS; ++m)
#pragma unroll
          for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][t][i] = 0.0f;
        struct WRaw {
          uint4 q[MATS];  // the group's four packed words
          float sc[MATS];
        };
        constexpr int XC = (NB * 4 + 7) / 8;  // activation copies per wave and K step (every wave issues XC)
        auto copy_x = [&](int ks) {            // activations of K step ks into tile ks % 2
#pragma unroll
          for (int q = 0; q < XC; ++q) pf_copy16_to_lds(xc_src[q] + ks * BK, xs0 + (ks & 1) * XT * 2 + xc_dst[q]);
        };
        // this lane's weights of K step ks, from the LDS ring and the staged scales
        auto fetch_w = [&](WRaw &r, int ks) {
#pragma unroll
          for (int m = 0; m < MATS; ++m) {
            const int q = (ks & 1) * 2 + lh;
            const uint8_t *st = w_ring + ((ks >> 1) & 1) * MATS * W_STAGE + m * W_STAGE;
            r.q[m] = *(const uint4 *)(st + (trow * 4 + (q ^ ((trow >> 2) & 3))) * 16);
            const uint8_t *sb = sc_lds + ((ks / SC_BLOCK) & 1) * (BN * MATS * SC_STRIDE) + (m * BN + trow) * SC_STRIDE;
            const int el = (ks % SC_BLOCK) * 2 + lh;  // the lane's group among the block's 32
            r.sc[m] = kx_bf16_f32(*(const uint16_t *)(sb + (((el >> 3) ^ ((trow >> 1) & 3)) * 8 + (el & 7)) * 2));
          }
        };
        auto dequant_j = [&](const WRaw &r, int j, kx_bf16x8 (&b)[MATS]) {
#pragma unroll
          for (int m = 0; m < MATS; ++m) {
            const float sc = r.sc[m];
            const uint32_t w = j == 0 ? r.q[m].x : j == 1 ? r.q[m].y : j == 2 ? r.q[m].z : r.q[m].w;
            b[m] = dequant_word(w, sc, sc * 0.0625f, -1032.0f * sc, -72.0f * sc, magic);
          }
        };
        auto read_a = [&](const uint16_t *xs, int j, kx_bf16x8 (&av)[NB]) {
          const int off = lr * 128 + (((lh * 4 + j) ^ (lr >> 1)) & 7) * 16;  // 128-byte rows, pieces xor-swizzled by the row
#pragma unroll
          for (int t = 0; t < NB; ++t) av[t] = *(const kx_bf16x8 *)((const uint8_t *)xs + t * 32 * 128 + off);
        };
        constexpr int VPER = (34 * MATS + NB * MATS - 1) / (NB * MATS);  // VALU instructions per MFMA
        auto mfma_group = [&](const kx_bf16x8 (&av)[NB], const kx_bf16x8 (&b)[MATS], auto with_valu) {
#pragma unroll
          for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int m = 0; m < MATS; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[t], b[m], acc[m][t], 0, 0, 0);
          // scheduling: one MFMA, then a share of the VALU work that prepares the next group
#pragma unroll
          for (int i = 0; i < NB * MATS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (decltype(with_valu)::value) __builtin_amdgcn_sched_group_barrier(0x002, VPER, 0);
          }
        };
        // one K step.  MFMA j contracts over columns 8 j .. +7 (lanes 0-31) and 32 + 8 j .. +7 (lanes 32-63); the
        // operands of group j+1 (LDS reads, dequant) are produced while the matrix cores run group j.
        auto step = [&](const WRaw &r, int ks, auto ask_late) {
          const uint16_t *xs = xs_lds + (ks & 1) * XT;
          kx_bf16x8 b0[MATS], b1[MATS], a0[NB], a1[NB];
          dequant_j(r, 0, b0);
          read_a(xs, 0, a0);
          read_a(xs, 1, a1);
          dequant_j(r, 1, b1);
          mfma_group(a0, b0, std::true_type{});
          ask_late();
          read_a(xs, 2, a0);
          dequant_j(r, 2, b0);
          mfma_group(a1, b1, std::true_type{});
          read_a(xs, 3, a1);
          dequant_j(r, 3, b1);
          mfma_group(a0, b0, std::true_type{});
          mfma_group(a1, b1, std::false_type{});
        };

        // A copy holds up the wave that asks for it until the CU's address path has taken it.  In a full tile one wave of each SIMD asks behind
        // the step's first products, so that the other one's products run meanwhile: 8 experts of 2048 tokens, gate and up 1000 -> 950
        // us, down 540 -> 525; tiles with fewer tokens take up to 9 % longer that way, their steps being shorter than the copies' way.
        const bool late = NB == 4 && wave >= 4;
        // prologue: stage 0 of the ring, the first scale block, the first activation tile
        WRaw w0, w1;
        copy_scales(0);
        copy_x(0);
        dma_stage(0);
        pf_wait_copies<0>();
        pf_barrier();
        for (int ks = 0; ks < nk; ks += 2) {
          // even step: the other ring stage and the other activation tile were last read behind a barrier.  Order of
          // issue: activations of the next step, the ring copies, then (every SC_BLOCK steps) the next scale block; the
          // activations have to land by the end of this step, the copies behind them stay in flight until the end of
          // the odd step (a wave's copies complete in the order of issue)
          const bool scales_now = ks % SC_BLOCK == 0 && ks + SC_BLOCK < nk;
          auto ask = [&]() {
            if (ks + 1 < nk) copy_x(ks + 1);
            if (ks + 2 < nk) dma_stage((ks >> 1) + 1);
            if (scales_now) copy_scales(ks / SC_BLOCK + 1);
          };
          if (!late) ask();
          fetch_w(w0, ks);
          step(w0, ks, [&]() {
            if (late) ask();
          });
          if (scales_now) pf_wait_copies<MATS * 4>();
          else if (ks + 2 < nk) pf_wait_copies<MATS * 2>();
          else pf_wait_copies<0>();
          pf_barrier();
          if (ks + 1 < nk) {
            if (!late && ks + 2 < nk) copy_x(ks + 2);
            fetch_w(w1, ks + 1);
            step(w1, ks + 1, [&]() {
              if (late && ks + 2 < nk) copy_x(ks + 2);
            });
            pf_wait_copies<0>();  // this wave's copies (ring stage, activations) have landed
            pf_barrier();
          }
        }
        // epilogue: D[i][j], j = lane % 32 (weight row), i = 8*(v/4) + 4*(lane/32) + v%4 (token of the 32-token block)
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int po = m0 + t * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
            if (po < p_end) {
              uint16_t *out = a.out + (size_t)a.pairs[po] * a.N;
              if constexpr (DUAL) {
                if (n0 + trow < a.N) out[n0 + trow] = kx_bf16_rne(kx_swiglu(kx_bfround(acc[0][t][v]), kx_bfround(acc[MATS - 1][t][v])));
              } else {
#pragma unroll
                for (int m = 0; m < MATS; ++m)
                  if (n0 + m * BN + trow < a.N) out[n0 + m * BN + trow] = kx_bf16_rne(acc[m][t][v]);
              }
            }
          }
      };
      if (nb == 1) run(std::integral_constant<int, 1>{});
      else if (nb == 2) run(std::integral_constant<int, 2>{});
      else if (nb == 3) run(std::integral_constant<int, 3>{});
      else run(std::integral_constant<int, 4>{});
    }
  }
}

// x[t][r] = bf(x + bf(bf(sum_slot eout[t*topk+slot][r] * w[t][slot]) + sy[t][r]))  (:868-877)
// W columns per thread, 8 where rows are whole 16-byte pieces; their rows of all slots are asked for together, up to eight.  Bound by the
// experts' results: 2048 tokens of 8 x 7168 154 us with a column per thread, 57 now.
template <int W>
__global__ void __launch_bounds__(256) moe_combine_k(const uint16_t *__restrict__ eout, const float *__restrict__ rw,
                                                     const uint16_t *__restrict__ sy, uint16_t *__restrict__ x, int hidden,
                                                     int topk, uint32_t flags) {
  struct alignas(W * 2) Cols {
    uint16_t v[W];
  };
  const int t = blockIdx.y, r = (blockIdx.x * blockDim.x + threadIdx.x) * W;
  if (r >= hidden) return;
  const uint16_t *e = eout + (size_t)t * topk * hidden + r;
  const Cols s = *(const Cols *)(sy + (size_t)t * hidden + r);
  Cols *xr = (Cols *)(x + (size_t)t * hidden + r), old = *xr;
  float acc[W] = {};
  for (int k0 = 0; k0 < topk; k0 += 8) {
    Cols y[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) y[k] = *(const Cols *)(e + (size_t)min(k0 + k, topk - 1) * hidden);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k0 + k < topk) {
        const float w = rw[(size_t)t * topk + k0 + k];
#pragma unroll
        for (int c = 0; c < W; ++c) acc[c] = __builtin_fmaf(kx_bf16_f32(y[k].v[c]), w, acc[c]);
      }
  }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    const float down = kx_bfround(kx_bfround(acc[c]) + kx_bf16_f32(s.v[c]));
    old.v[c] = (flags & 1u) ? kx_bf16_rne(down) : kx_bf16_rne(kx_bf16_f32(old.v[c]) + down);
  }
  *xr = old;
}

}  // namespace

int kx_grouped_tiles_launch(const int4 *work, int n_slots, int cnt_lo, int4 *tiles, int *n_tiles, hipStream_t st) {
  KX_REQUIRE(n_slots > 0 && n_slots <= 1024, "kx_grouped_tiles: %d groups", n_slots);
  hipLaunchKernelGGL(grouped_tiles_k, dim3(1), dim3(1024), 0, st, work, n_slots, cnt_lo, tiles, n_tiles);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

int kx_grouped_gemm_launch(bool dual, const void *w0, const uint16_t *s0, const void *w1, const uint16_t *s1, const uint16_t *x, uint16_t *out,
                           const int4 *tiles, const int *n_tiles, const int *pairs, int tiles_max, int N, int K, int x_div, size_t expert_w, size_t expert_s,
                           hipStream_t st, int cnt_lo) {
  KX_REQUIRE(K > 0 && K % 512 == 0, "kx_grouped_gemm: K=%d must be a positive multiple of 512", K);
  KX_REQUIRE(N > 0, "kx_grouped_gemm: N=%d must be positive", N);
  PfArgs a;
  a.w0 = (const uint32_t *)w0; a.w1 = (const uint32_t *)w1; a.s0 = s0; a.s1 = s1; a.x = x; a.out = out; a.tiles = tiles; a.pairs = pairs;
  a.n_tiles = n_tiles;
  a.tiles_max = tiles_max;
  a.cnt_lo = cnt_lo;
  a.N = N; a.K = K; a.x_div = x_div; a.expert_w = expert_w; a.expert_s = expert_s;
  const int mode = dual ? GG_DUAL : n_tiles ? GG_WIDE : GG_SINGLE, mats = mode == GG_SINGLE ? 1 : 2;
  a.row_tiles = kx_cdiv(N, mode == GG_WIDE ? 2 * BN : BN);
  const long items = (long)tiles_max * a.row_tiles;
  KX_REQUIRE(tiles_max > 0 && items < (1L << 31), "kx_grouped_gemm: %d tiles of %d rows", tiles_max, N);
  // With a list a workgroup per CU goes over it, since only the device knows how long it is: a workgroup per possible tile (128
  // tokens of every expert) were 170000 for 2048 tokens to 384 experts, nearly all of them without work and each waiting for a CU of
  // its own, whose registers it takes whole.  A few tokens per expert beside other kernels gain
  // nothing by it (16 tokens 580 us, 583 with a list and its launch).
  const dim3 g((unsigned)(n_tiles ? std::min<long>(items, std::max(1, kx_device_cus())) : items)), b(512);
  const size_t lds = (size_t)2 * XT * 2 + (size_t)2 * mats * W_STAGE + (size_t)2 * BN * mats * SC_STRIDE;
  static std::atomic<bool> attr_set{false};  // setting it twice from two threads is harmless
  if (!attr_set) {  // more than 64 KB of dynamic LDS has to be allowed per kernel
    KX_HIP(hipFuncSetAttribute((const void *)grouped_gemm_k<GG_SINGLE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    KX_HIP(hipFuncSetAttribute((const void *)grouped_gemm_k<GG_WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    KX_HIP(hipFuncSetAttribute((const void *)grouped_gemm_k<GG_DUAL>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    attr_set = true;
  }
  if (mode == GG_DUAL) hipLaunchKernelGGL(grouped_gemm_k<GG_DUAL>, g, b, lds, st, a);
  else if (mode == GG_WIDE) hipLaunchKernelGGL(grouped_gemm_k<GG_WIDE>, g, b, lds, st, a);
  else hipLaunchKernelGGL(grouped_gemm_k<GG_SINGLE>, g, b, lds, st, a);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

int kx_moe_combine_launch(const uint16_t *eout, const float *rw, const uint16_t *sy, uint16_t *x, int tokens, int hidden,
                          int topk, uint32_t flags, hipStream_t st) {
  const bool pieces = hidden % 8 == 0 && (((uintptr_t)eout | (uintptr_t)sy | (uintptr_t)x) & 15) == 0;
  if (pieces) hipLaunchKernelGGL(moe_combine_k<8>, dim3(kx_cdiv(hidden, 8 * 256), tokens), dim3(256), 0, st, eout, rw, sy, x, hidden, topk, flags);
  else hipLaunchKernelGGL(moe_combine_k<1>, dim3(kx_cdiv(hidden, 256), tokens), dim3(256), 0, st, eout, rw, sy, x, hidden, topk, flags);
  KX_LAUNCH_CHECK();
  return KX_OK;
}
