// kx_dense_gemm.hip -- bf16 products of Kimi-K2 steps of more than 32 tokens: the dense projections, the shared expert, the router's
// logits, W_UV per head, with the epilogues of the mat-vec kernels they stand for (matvec_bf16_k / matvec_bf16_f32_k with
// add_k, silu_mul_k and the rounding of the logits, src/kimi_exec.cu:248-298, :718-734).
//
// The main loops are kx_gemm_tile.h's and kx_gemm_turns.h's.  With two matrices (SwiGLU) a tile's rows are blocks of 32 gate rows and their 32 up rows in
// turn, so that a wave holds both halves of a pair.  Before these tiles the products went through the W4A16 kernel's loop with 64
// tokens a tile and every lane loading its own row of the matrix: 400 TFLOP/s where these reach 1200 (2048 tokens, gate
// and up of 2 x 18432 x 7168 with SwiGLU 2.7 ms then, 0.9 now).
// fp32 sums over exact bf16 products: a tolerance path like every matrix-core path (max-rel 1e-2), not used where tokens
// have to be identical.
#include <atomic>
#include "kx_common.h"
#include "kx_dense.h"
#include "kx_gemm_tile.h"
#include "kx_math.h"

namespace {

typedef kxtile::Tile<uint16_t, 2, 2, 1, 2, 4> Short;  // 64 tokens x 128 rows: up to 64 tokens

template <class TL, int MODE, bool DUAL, bool GROUP>
__global__ void __launch_bounds__(TL::THREADS, TL::WAVES_PER_SIMD) dense_gemm_k(KxDenseArgs a, kxtile::Share share) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int COLS = DUAL ? TL::BN / 2 : TL::BN;  // results per token of a tile
  int m0, m_end, n0;
  kxtile::Place place = {0, 0, 1};
  const uint16_t *w0 = a.w0, *w1 = a.w1;
  if constexpr (GROUP) {
    const int4 g = a.work[blockIdx.y];
    if (g.x < 0) return;
    m0 = g.y + blockIdx.z * TL::BM;
    m_end = g.z;
    if (m0 >= m_end) return;
    n0 = blockIdx.x * COLS;
    w0 += (size_t)g.x * a.group_stride;
  } else {
    const int tm = (a.tokens + TL::BM - 1) / TL::BM;
    place = kxtile::place_of(blockIdx.x, tm * ((a.rows + COLS - 1) / COLS), share);
    m0 = place.tile % tm * TL::BM;
    m_end = a.tokens;
    n0 = place.tile / tm * COLS;
  }
  auto row_of = [&](int i) {
    if constexpr (MODE == KX_GG_KV) return i / a.seq * a.seq_jump + i % a.seq;
    else return GROUP ? a.pairs[i] : i;
  };
  const int nb = a.cols >> 6;
  typename TL::Sums acc;
  TL::run(lds, kxtile::cut(nb, place.part, place.of), kxtile::cut(nb, place.part + 1, place.of), [&](int r) -> const uint16_t * {
    if (r < TL::BM) return a.x + (size_t)row_of(min(m0 + r, m_end - 1)) * a.x_stride;
    r -= TL::BM;
    if constexpr (DUAL) return ((r >> 5 & 1) ? w1 : w0) + (size_t)min(n0 + (r >> 6) * 32 + (r & 31), a.rows - 1) * a.cols;
    else return w0 + (size_t)min(n0 + r, a.rows - 1) * a.cols;
  }, acc);
  if (!GROUP && place.of > 1 &&
      !kxtile::gather<TL>(lds, acc, a.part + (size_t)(place.tile - share.whole) * place.of * TL::PART, a.arrived + place.tile - share.whole, place.of, place.part))
    return;
  // result c (of a tile's COLS) of block (i, j): in row at(v) of out, if there is one
  auto result = [&](int j) { const int c = TL::col(j); return n0 + (DUAL ? (c >> 6) * 32 + (c & 31) : c); };
  auto in = [&](int i, int v) { return m0 + TL::row(i, v) < m_end; };
  auto at = [&](int i, int v, int n) { return (size_t)row_of(min(m0 + TL::row(i, v), m_end - 1)) * a.out_stride + n; };
  constexpr int STEP = DUAL ? 32 / TL::SIDE : 1;  // blocks of gate rows in front of their up rows
#pragma unroll
  for (int i = 0; i < TL::MI; ++i) {
    if constexpr (MODE == KX_GG_RESID && !DUAL) {  // x = bf(x + bf(y))  (add_k, :248-251); 16 are read before the first is written
#pragma unroll
      for (int e0 = 0; e0 < TL::NI * TL::V; e0 += 16) {
        uint16_t old[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) old[u] = ((const uint16_t *)a.out)[at(i, (e0 + u) % TL::V, min(result((e0 + u) / TL::V), a.rows - 1))];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int j = (e0 + u) / TL::V, v = (e0 + u) % TL::V, n = result(j);
          if (in(i, v) && n < a.rows) ((uint16_t *)a.out)[at(i, v, n)] = kx_bf16_rne(kx_bf16_f32(old[u]) + kx_bfround(acc[i][j][v]));
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < TL::NI; ++j) {
        if (DUAL && j / STEP % 2) continue;
        const int n = result(j);
        if (n >= a.rows) continue;
        if constexpr (MODE == KX_GG_KV) {
          const int per = a.k_dim + a.v_dim, hd = n / per, d = n - hd * per;
          const bool key = d < a.k_dim;
          uint16_t *to = key ? (uint16_t *)a.out + d : a.out_v + (d - a.k_dim);
          const int ld = key ? a.k_ld : a.v_ld;
#pragma unroll
          for (int v = 0; v < TL::V; ++v)
            if (in(i, v)) {
              const int t = m0 + TL::row(i, v), b = t / a.seq;
              to[((size_t)(b * a.heads + hd) * a.cap + t - b * a.seq) * ld] = kx_bf16_rne(acc[i][j][v]);
            }
        } else {
#pragma unroll
          for (int v = 0; v < TL::V; ++v)
            if (in(i, v)) {
              if constexpr (DUAL) ((uint16_t *)a.out)[at(i, v, n)] = kx_bf16_rne(kx_swiglu(kx_bfround(acc[i][j][v]), kx_bfround(acc[i][j + STEP][v])));
              else if constexpr (MODE == KX_GG_BF16) ((uint16_t *)a.out)[at(i, v, n)] = kx_bf16_rne(acc[i][j][v]);
              else ((float *)a.out)[at(i, v, n)] = MODE == KX_GG_F32 ? acc[i][j][v] : kx_bfround(acc[i][j][v]);
            }
        }
      }
    }
  }
}

template <class TL, int MODE, bool DUAL, bool GROUP>
int launch_as(const KxDenseArgs &a, kxtile::Share share, hipStream_t st) {
  static std::atomic<bool> attr{false};  // setting it twice from two threads is harmless
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)dense_gemm_k<TL, MODE, DUAL, GROUP>, hipFuncAttributeMaxDynamicSharedMemorySize, TL::LDS));
    attr = true;
  }
  const int tn = kx_cdiv(a.rows, DUAL ? TL::BN / 2 : TL::BN), tm = kx_cdiv(a.tokens, TL::BM);
  const dim3 grid = GROUP ? dim3(tn, a.groups, tm) : dim3(share.grid(tn * tm));
  hipLaunchKernelGGL((dense_gemm_k<TL, MODE, DUAL, GROUP>), grid, dim3(TL::THREADS), TL::LDS, st, a, share);
  KX_LAUNCH_CHECK();
  return KX_OK;
}
template <class TL>
int launch(const KxDenseArgs &a, kxtile::Share share, hipStream_t st) {
  if (a.w1) return launch_as<TL, KX_GG_BF16, true, false>(a, share, st);
  switch (a.mode) {
    case KX_GG_BF16: return launch_as<TL, KX_GG_BF16, false, false>(a, share, st);
    case KX_GG_F32: return launch_as<TL, KX_GG_F32, false, false>(a, share, st);
    case KX_GG_RESID: return launch_as<TL, KX_GG_RESID, false, false>(a, share, st);
    case KX_GG_KV: return launch_as<TL, KX_GG_KV, false, false>(a, share, st);
  }
  return launch_as<TL, KX_GG_F32_OF_BF16, false, false>(a, share, st);
}

}  // namespace

int kx_dense_gemm_launch(const KxDenseArgs &a, hipStream_t st) {
  KX_REQUIRE(a.w0 && a.x && a.out && a.tokens > 0 && a.rows > 0, "kx_dense_gemm: tokens=%d rows=%d", a.tokens, a.rows);
  KX_REQUIRE(a.cols > 0 && a.cols % 128 == 0 && a.x_stride >= a.cols && a.x_stride % 8 == 0, "kx_dense_gemm: cols=%d must be a positive multiple of 128", a.cols);
  KX_REQUIRE(a.mode >= KX_GG_BF16 && a.mode <= KX_GG_KV && !((a.w1 || a.work) && a.mode != KX_GG_BF16) && !(a.w1 && a.work), "kx_dense_gemm: out_mode=%d", a.mode);
  KX_REQUIRE(a.mode != KX_GG_KV || (a.seq > 0 && a.tokens % a.seq == 0 && a.heads > 0 && a.rows == a.heads * (a.k_dim + a.v_dim) && a.cap >= a.seq && a.k_ld >= a.k_dim &&
                                    a.v_ld >= a.v_dim && a.out_v),
             "kx_dense_gemm: %d rows for %d heads, %d tokens", a.rows, a.heads, a.tokens);
  if (a.work) {
    KX_REQUIRE(a.pairs && a.groups > 0 && kx_cdiv(a.tokens, kxtile::Medium::BM) <= 65535, "kx_dense_gemm: %d groups", a.groups);
    return launch_as<kxtile::Medium, KX_GG_BF16, false, true>(a, {0, 1}, st);
  }
  const int cus = kx_device_cus() > 0 ? kx_device_cus() : 1, staged = a.w1 ? 2 * kx_pad32(a.rows) : a.rows, blocks = a.cols >> 6;
  const size_t room = a.part && a.arrived ? a.part_floats : 0;
  if (a.tokens <= Short::BM) {
    const long tiles = kx_cdiv(staged, Short::BN);
    long p = cus / tiles;
    p = p > blocks / 16 ? blocks / 16 : p;
    p = (size_t)p > room / Short::PART / tiles ? (long)(room / Short::PART / tiles) : p;
    if (p < 2 || tiles > a.arrivals) p = 1;
    return launch<Short>(a, {0, (int)p}, st);
  }
  const kxtile::Choice c = kxtile::choose(a.tokens, staged, blocks, room, a.arrivals, cus);
  return c.large ? launch<kxtile::Large>(a, c.s, st) : c.twin ? launch<kxtile::Twin>(a, c.s, st) : launch<kxtile::Medium>(a, c.s, st);
}
