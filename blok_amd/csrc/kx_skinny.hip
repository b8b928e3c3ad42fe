// kx_skinny.hip -- dense projections for decode batches of 5 to 32 sequences: y[t, r] = sum_k x[t, k] w[r, k] with
// bf16 weights [rows, cols] streamed once and the tokens as the other side of a matrix-core product.
//
// Reference: matvec_bf16_k / matvec_bf16_f32_k (src/kimi_exec.cu:272-298) called once per token; the epilogues are
// add_k (:248-251), silu_mul_k (:253-256) and the bf16 rounding of the logits (:718-734).
//
// A GEMV kernel streams the weights once per block of four tokens and is bound by its fma count from about 16 tokens
// on (every weight meets every token on the VALU), and
// the prefill GEMM of kx_dense_gemm.hip, built for tiles of 64 tokens and more, leaves most of the chip idle on one of
// 32.  Here a workgroup of 8 waves takes tiles of 32 weight rows (16 of each of two matrices) and all (up to 32) tokens, the eight waves
// split the columns, and their partial 32 x 32 tiles (v_mfma_f32_32x32x16_bf16) are summed through LDS in wave
// order before the epilogue.
//
// Both operands are staged through LDS.  The operand layout of the matrix cores is one row per lane: loading the
// operands straight from memory makes every load instruction touch 32 rows with 32 bytes each, and that streams at
// 2.3-3 TB/s whatever the number of waves (measured; the lm_head then takes 1.0 ms).  So the columns are walked in
// blocks of 256: a copy instruction (global_load_lds_dwordx4, no registers) moves 512 contiguous bytes of two rows,
// lane (l / 32, l % 32) = (row of the pair, 16-byte slot); the lane fetches piece slot ^ (row % 16) of its row, so
// that the operand reads -- lane (r, h) wants piece p of row r and finds it in slot p ^ (r % 16) -- fall into different
// banks.  Blocks go through a ring of 5 stages (4 with more than 16 tokens), four (three) blocks in flight behind the one being
// multiplied; each wave issues its share of a block's copies, waits for its own by count (they complete in order),
// and one barrier per block makes every wave's copies visible and the stage that is overwritten next free.  Wave w
// multiplies pieces 4w .. 4w+3 of the block.  Matrices of large models are copied nontemporally (kx_read_once.h).
// LDS leaves a CU one workgroup.  Where there are tiles for half of the CUs and more, every CU has one and an equal share of the rows, whose tiles follow each other
// through the ring: the next tile's blocks are on their way while a tile's sums are added.  A workgroup per 32 rows instead was 224 for the 7168
// rows of a down projection and, two matrices at a time, two rounds and a quarter for 18432 rows.  12 tokens, 2 x 18432 x 7168 91.5 us so, 79.3 now; 7168 x
// 8192, 7168 x 18432, 12288 x 1536 (two each) and 32768 x 7168 35.7 on average, 32.2 now; a step through two dense layers and a head 624 -> 568 us.
// The copies are issued from inline asm and the barrier carries no fence: a copy the compiler knows of makes it
// complete everything in flight before every LDS access it cannot tell from the copy's target.
//
// Sums are fp32 over exact bf16 products in another order than the GEMV's: this path is held to the 1e-2 bar, like the
// other matrix-core paths, and serves batches the token-identity checks do not run on.
#include <algorithm>
#include <atomic>
#include "kx_common.h"
#include "kx_lds_copy.h"
#include "kx_dense.h"
#include "kx_math.h"
#include "kx_read_once.h"

namespace {

typedef __bf16 kx_bf16x8 __attribute__((ext_vector_type(8)));
typedef float kx_f32x16 __attribute__((ext_vector_type(16)));

struct SkinnyArgs {
  const uint16_t *w0, *w1;  // bf16 [rows, cols]; w1 for the two-matrix SwiGLU form
  const uint16_t *x;        // bf16 [tokens, x_stride]
  void *out;                // [tokens, out_stride]: bf16, or f32 (see mode)
  int rows, cols, tokens, x_stride, out_stride, mode;
  int share, extra;         // rows of a workgroup, one more for the first `extra`
};

template <int N>
__device__ __forceinline__ void sk_wait_copies() { kx_wait_copies<N>(); }
__device__ __forceinline__ void sk_barrier() { kx_lds_barrier(); }

// FEW: up to 16 tokens, half the copies of tokens and a stage more.  DUAL: a tile is 16 rows of each matrix.  ONCE (of the kernel): matrices are copied nontemporally.
template <bool DUAL, bool FEW>
struct Skinny {
  static constexpr int NS = FEW ? 5 : 4;             // stages
  static constexpr int XC = FEW ? 1 : 2, CPW = 2 + XC;  // copy instructions per wave and block: two of the matrix, XC of the tokens
  static constexpr int ROWS = DUAL ? 16 : 32;        // rows of the result per tile
  static constexpr uint32_t TILE = 32 * 512, STAGE = TILE + (FEW ? 16 : 32) * 512, PART = NS * STAGE;
  static constexpr size_t LDS = PART + 8 * 16 * 32 * sizeof(float);  // the ring, and the waves' sums of 16 tokens
};

template <bool DUAL, bool FEW, bool ONCE>
__global__ void __launch_bounds__(512) skinny_staged_k(SkinnyArgs a) {
  using K = Skinny<DUAL, FEW>;
  constexpr int NS = K::NS, CPW = K::CPW, ROWS = K::ROWS;
  extern __shared__ __attribute__((aligned(16))) uint8_t sk_lds[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)sk_lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int nb = a.cols >> 8;  // blocks of 256 columns
  const int bx = blockIdx.x, row_end = min((bx + 1) * a.share + min(bx + 1, a.extra), a.rows);
  int row0 = bx * a.share + min(bx, a.extra);  // of the tile that is multiplied
  const int total = (row_end - row0 + ROWS - 1) / ROWS * nb;
  // this wave's copies of a block: instruction i moves staged rows 2 i and 2 i + 1
  const uint16_t *wsrc[2], *xsrc[K::XC];
  auto rows_from = [&](int first) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 2 * (u * 8 + wave) + h;
      wsrc[u] = (DUAL && u ? a.w1 : a.w0) + (size_t)min(first + (DUAL ? row & 15 : row), row_end - 1) * a.cols + (r ^ (row & 15)) * 8;
    }
  };
#pragma unroll
  for (int u = 0; u < K::XC; ++u) {
    const int row = 2 * (u * 8 + wave) + h;
    xsrc[u] = a.x + (size_t)min(row, a.tokens - 1) * a.x_stride + (r ^ (row & 15)) * 8;
  }
  int copy_row = row0, copy_block = 0, copy_stage = 0;  // what is asked for next
  rows_from(copy_row);
  auto copy_next = [&]() {
    const uint32_t st = lds0 + (uint32_t)copy_stage * K::STAGE + wave * 1024;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint16_t *const from = wsrc[u] + copy_block * 256;
      const uint32_t to = __builtin_amdgcn_readfirstlane(st + u * 8192);
      if constexpr (ONCE) kx_copy16_to_lds_once(from, to);
      else kx_copy16_to_lds(from, to);
    }
#pragma unroll
    for (int u = 0; u < K::XC; ++u) kx_copy16_to_lds(xsrc[u] + copy_block * 256, __builtin_amdgcn_readfirstlane(st + K::TILE + u * 8192));
    copy_stage = copy_stage == NS - 1 ? 0 : copy_stage + 1;
    if (++copy_block == nb) {
      copy_block = 0;
      rows_from(copy_row += ROWS);
    }
  };
  kx_f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  // operand reads of this lane: piece 4 wave + 2 q + h of row r sits in slot piece ^ (r % 16)
  uint32_t roff[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) roff[q] = (uint32_t)((4 * wave + 2 * q + h) ^ (r & 15)) * 16;
  const uint32_t wrow = (uint32_t)r * 512, xrow = K::TILE + (uint32_t)(FEW ? r & 15 : r) * 512;  // tokens 16 to 31 of FEW: nobody's

#pragma unroll
  for (int k = 0; k < NS - 1; ++k)
    if (k < total) copy_next();
  int stage = 0, block = 0;
  for (int k = 0; k < total; ++k) {
    // this wave's copies of block k have landed when at most those of the blocks behind it are in flight; stores of the last tile's
    // results, which are counted with them, make it wait for more
    const int behind = min(total - 1 - k, NS - 2);
    if (NS > 4 && behind >= 3) sk_wait_copies<3 * CPW>();
    else if (behind >= 2) sk_wait_copies<2 * CPW>();
    else if (behind == 1) sk_wait_copies<CPW>();
    else sk_wait_copies<0>();
    sk_barrier();  // every wave's copies of block k are in LDS; every wave is done with block k - 1
    if (k + NS - 1 < total) copy_next();  // into the stage block k - 1 was read from
    const uint8_t *st = sk_lds + (uint32_t)stage * K::STAGE;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const kx_bf16x8 *)(st + xrow + roff[q]), *(const kx_bf16x8 *)(st + wrow + roff[q]), acc, 0, 0, 0);
    stage = stage == NS - 1 ? 0 : stage + 1;
    if (++block < nb) continue;
    block = 0;
    // the tile's sums, 16 tokens at a time; the barriers of a tile's blocks, two at least, lie between its reads here and the next one's writes
    float(*part)[16][32] = (float(*)[16][32])(sk_lds + K::PART);
#pragma unroll
    for (int p = 0; p < (FEW ? 1 : 2); ++p) {
      if (p) sk_barrier();
#pragma unroll
      for (int v = 0; v < 8; ++v) part[wave][8 * (v >> 2) + 4 * h + (v & 3)][r] = acc[8 * p + v];
      sk_barrier();
      const int rr = threadIdx.x % ROWS, t = threadIdx.x / ROWS, row = row0 + rr, tok = 16 * p + t;
      if (t >= 16 || row >= row_end || tok >= a.tokens) continue;
      auto sum = [&](int c) {
        float y = part[0][t][c];
#pragma unroll
        for (int w = 1; w < 8; ++w) y += part[w][t][c];
        return y;
      };
      const float y = sum(rr);
      const size_t o = (size_t)tok * a.out_stride + row;
      if (DUAL) {
        ((uint16_t *)a.out)[o] = kx_bf16_rne(kx_swiglu(kx_bfround(y), kx_bfround(sum(rr + 16))));
      } else if (a.mode == KX_GG_BF16) {
        ((uint16_t *)a.out)[o] = kx_bf16_rne(y);
      } else if (a.mode == KX_GG_F32) {
        ((float *)a.out)[o] = y;
      } else if (a.mode == KX_GG_F32_OF_BF16) {
        ((float *)a.out)[o] = kx_bfround(y);
      } else {  // x = bf(x + bf(y))  (add_k, :248-251)
        uint16_t *xo = (uint16_t *)a.out + o;
        *xo = kx_bf16_rne(kx_bf16_f32(*xo) + kx_bfround(y));
      }
    }
    row0 += ROWS;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  }
}

template <bool DUAL, bool FEW, bool ONCE>
int skinny(SkinnyArgs a, hipStream_t st) {
  using K = Skinny<DUAL, FEW>;
  static std::atomic<bool> attr{false};  // setting it twice from two threads is harmless
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)skinny_staged_k<DUAL, FEW, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)K::LDS));
    attr = true;
  }
  const int tiles = kx_cdiv(a.rows, K::ROWS), cus = std::max(1, kx_device_cus());
  const int even = std::min(cus, a.rows), grid = 2 * tiles > cus ? even : tiles;
  a.share = grid == even ? a.rows / even : K::ROWS;
  a.extra = grid == even ? a.rows % even : 0;
  hipLaunchKernelGGL((skinny_staged_k<DUAL, FEW, ONCE>), dim3(grid), dim3(512), K::LDS, st, a);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

}  // namespace

// One tile of up to 32 tokens against a bf16 matrix (two for SwiGLU).  Returns KX_OK with *done = false, having
// launched nothing, when the shape is not the kernel's (cols not a multiple of 512, more than 32 tokens).
int kx_skinny_gemm_launch(bool dual, const uint16_t *w0, const uint16_t *w1, const uint16_t *x, int x_stride, void *out,
                          int out_stride, int out_mode, int tokens, int rows, int cols, size_t model_bytes, bool *done, hipStream_t st) {
  *done = false;
  if (tokens < 1 || tokens > 32 || rows < 1 || cols < 512 || cols % 512 || x_stride % 8 || x_stride < cols || (dual && !w1)) return KX_OK;
  KX_REQUIRE(out_mode >= KX_GG_BF16 && out_mode <= KX_GG_RESID && !(dual && out_mode != KX_GG_BF16), "kx_skinny_gemm: out_mode=%d", out_mode);
  SkinnyArgs a;
  a.w0 = w0; a.w1 = w1; a.x = x; a.out = out; a.rows = rows; a.cols = cols; a.tokens = tokens; a.x_stride = x_stride;
  a.out_stride = out_stride; a.mode = out_mode;
  const bool few = tokens <= 16;
  int rc;
  if (kxonce::layers(model_bytes)) rc = dual ? few ? skinny<true, true, true>(a, st) : skinny<true, false, true>(a, st) : few ? skinny<false, true, true>(a, st) : skinny<false, false, true>(a, st);
  else rc = dual ? few ? skinny<true, true, false>(a, st) : skinny<true, false, false>(a, st) : few ? skinny<false, true, false>(a, st) : skinny<false, false, false>(a, st);
  *done = rc == KX_OK;
  return rc;
}
