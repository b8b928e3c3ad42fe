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
#include "kx_wave.h"

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
  // Blocks of 16 columns are 32 bytes of a row of bf16 results, a quarter of a line, one result to a lane.  Two lanes exchange theirs of two
  // blocks, so that a store takes 64 bytes of each of its rows (even lanes have two columns of block j, odd lanes two of block j + 1).
  // Keys and values of 64 heads from 512 columns, 3072 x 16384 164 -> 86 us (one by one is what the tile's short products wait for; 32 columns
  // to a block took 127); gate and up 2048 x 36864 x 7168 877 -> 848.  Where pairs are not aligned, one by one.
  if constexpr (TL::SIDE == 16 && !GROUP && (MODE == KX_GG_BF16 || MODE == KX_GG_RESID || MODE == KX_GG_KV)) {
    if (MODE == KX_GG_KV || a.pairs_aligned) {
      const uint32_t odd = threadIdx.x & 1, order = odd ? 0x03020706u : 0x05040100u;
      auto pack = [](float lo, float hi) { return (uint32_t)kx_bf16_rne(lo) | (uint32_t)kx_bf16_rne(hi) << 16; };
      auto exchanged = [&](float lo, float hi) {  // of blocks j and j + 1
        const uint32_t p = pack(lo, hi), q = kx_f32_bits(kxw::dpp_f<kxw::DPP_QUAD_XOR1>(kx_bits_f32(p)));
        return __builtin_amdgcn_perm(q, p, order);
      };
      constexpr int PAIRS = DUAL ? TL::NI / 4 : TL::NI / 2;
      auto block = [](int u) { return DUAL ? 4 * u : 2 * u; };
      int n[PAIRS];
#pragma unroll
      for (int u = 0; u < PAIRS; ++u) n[u] = odd ? result(block(u) + 1) - 1 : result(block(u));
      if constexpr (MODE == KX_GG_KV) {
        uint16_t *to[PAIRS];
        int ld[PAIRS];
#pragma unroll
        for (int u = 0; u < PAIRS; ++u) {
          const int per = a.k_dim + a.v_dim, c = min(n[u], a.rows - 2), hd = c / per, d = c - hd * per;
          const bool key = d < a.k_dim;
          ld[u] = key ? a.k_ld : a.v_ld;
          to[u] = (key ? (uint16_t *)a.out + d : a.out_v + (d - a.k_dim)) + (size_t)hd * a.cap * ld[u];
        }
#pragma unroll
        for (int i = 0; i < TL::MI; ++i)
#pragma unroll
          for (int v = 0; v < TL::V; ++v) {
            const int t = m0 + TL::row(i, v), b = t / a.seq;
            const size_t row = (size_t)b * a.heads * a.cap + t - b * a.seq;
#pragma unroll
            for (int u = 0; u < PAIRS; ++u) {
              const uint32_t y = exchanged(acc[i][2 * u][v], acc[i][2 * u + 1][v]);
              if (in(i, v) && n[u] < a.rows) *(uint32_t *)(to[u] + row * ld[u]) = y;
            }
          }
      } else {
#pragma unroll
        for (int i = 0; i < TL::MI; ++i) {
          uint32_t old[TL::V][PAIRS];
          if constexpr (MODE == KX_GG_RESID) {  // x = bf(x + bf(y))  (add_k, :248-251); a block's are read before the first is written
#pragma unroll
            for (int v = 0; v < TL::V; ++v)
#pragma unroll
              for (int u = 0; u < PAIRS; ++u) old[v][u] = *(const uint32_t *)((const uint16_t *)a.out + at(i, v, min(n[u], a.rows - 2)));
          }
#pragma unroll
          for (int v = 0; v < TL::V; ++v)
#pragma unroll
            for (int u = 0; u < PAIRS; ++u) {
              const int j = block(u);
              uint32_t y;
              if constexpr (DUAL)
                y = exchanged(kx_swiglu(kx_bfround(acc[i][j][v]), kx_bfround(acc[i][j + 2][v])), kx_swiglu(kx_bfround(acc[i][j + 1][v]), kx_bfround(acc[i][j + 3][v])));
              else y = exchanged(acc[i][j][v], acc[i][j + 1][v]);
              if constexpr (MODE == KX_GG_RESID)
                y = pack(kx_bits_f32(old[v][u] << 16) + kx_bits_f32(y << 16), kx_bits_f32(old[v][u] & 0xffff0000u) + kx_bits_f32(y & 0xffff0000u));
              if (in(i, v) && n[u] < a.rows) *(uint32_t *)((uint16_t *)a.out + at(i, v, n[u])) = y;
            }
        }
      }
      return;
    }
  }
  // One by one, block by block; row by row where blocks have 16 columns and share a line.  Where a row's results lie, and which lanes have one of
  // it, is worked out in front of the conditions: behind them the compiler does both again for each result, and a chain of 64 comparisons
  // is 0.4 us of a product of 8 us.
#pragma unroll
  for (int i = 0; i < TL::MI; ++i) {
    size_t row[TL::V];
    uint64_t lanes[TL::V];
#pragma unroll
    for (int v = 0; v < TL::V; ++v) {
      if constexpr (MODE == KX_GG_KV) {
        const int t = m0 + TL::row(i, v), b = t / a.seq;
        row[v] = (size_t)b * a.heads * a.cap + t - b * a.seq;
      } else {
        row[v] = at(i, v, 0);
      }
      lanes[v] = __builtin_amdgcn_ballot_w64(in(i, v));
      asm volatile("" : "+s"(lanes[v]));
    }
    if constexpr (MODE == KX_GG_RESID) {  // x = bf(x + bf(y))  (add_k, :248-251); 16 are read before the first is written
      uint16_t *const out = (uint16_t *)a.out;
#pragma unroll
      for (int e0 = 0; e0 < TL::NI * TL::V; e0 += 16) {
        uint16_t old[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) old[u] = out[row[(e0 + u) % TL::V] + min(result((e0 + u) / TL::V), a.rows - 1)];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int j = (e0 + u) / TL::V, v = (e0 + u) % TL::V, n = result(j);
          if (n < a.rows && __builtin_amdgcn_inverse_ballot_w64(lanes[v])) out[row[v] + n] = kx_bf16_rne(kx_bf16_f32(old[u]) + kx_bfround(acc[i][j][v]));
        }
      }
    } else if constexpr (MODE == KX_GG_KV) {
#pragma unroll
      for (int j = 0; j < TL::NI; ++j) {
        const int n = result(j), per = a.k_dim + a.v_dim, hd = n / per, d = n - hd * per;
        if (n >= a.rows) continue;
        const bool key = d < a.k_dim;
        const int ld = key ? a.k_ld : a.v_ld;
        uint16_t *to = (key ? (uint16_t *)a.out + d : a.out_v + (d - a.k_dim)) + (size_t)hd * a.cap * ld;
#pragma unroll
        for (int v = 0; v < TL::V; ++v)
          if (__builtin_amdgcn_inverse_ballot_w64(lanes[v])) to[row[v] * ld] = kx_bf16_rne(acc[i][j][v]);
      }
    } else {
      auto put = [&](int v, int j) {
        const size_t to = row[v] + result(j);
        if constexpr (DUAL) ((uint16_t *)a.out)[to] = kx_bf16_rne(kx_swiglu(kx_bfround(acc[i][j][v]), kx_bfround(acc[i][j + STEP][v])));
        else if constexpr (MODE == KX_GG_BF16) ((uint16_t *)a.out)[to] = kx_bf16_rne(acc[i][j][v]);
        else ((float *)a.out)[to] = MODE == KX_GG_F32 ? acc[i][j][v] : kx_bfround(acc[i][j][v]);
      };
      if constexpr (TL::SIDE == 16) {
#pragma unroll
        for (int v = 0; v < TL::V; ++v)
#pragma unroll
          for (int j = 0; j < TL::NI; ++j)
            if (!(DUAL && j / STEP % 2) && result(j) < a.rows && __builtin_amdgcn_inverse_ballot_w64(lanes[v])) put(v, j);
      } else {
#pragma unroll
        for (int j = 0; j < TL::NI; ++j) {
          if ((DUAL && j / STEP % 2) || result(j) >= a.rows) continue;
#pragma unroll
          for (int v = 0; v < TL::V; ++v)
            if (__builtin_amdgcn_inverse_ballot_w64(lanes[v])) put(v, j);
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

int kx_dense_gemm_launch(const KxDenseArgs &args, hipStream_t st) {
  KxDenseArgs a = args;
  KX_REQUIRE(a.w0 && a.x && a.out && a.tokens > 0 && a.rows > 0, "kx_dense_gemm: tokens=%d rows=%d", a.tokens, a.rows);
  KX_REQUIRE(a.cols > 0 && a.cols % 128 == 0 && a.x_stride >= a.cols && a.x_stride % 8 == 0, "kx_dense_gemm: cols=%d must be a positive multiple of 128", a.cols);
  KX_REQUIRE(a.mode >= KX_GG_BF16 && a.mode <= KX_GG_KV && !((a.w1 || a.work) && a.mode != KX_GG_BF16) && !(a.w1 && a.work), "kx_dense_gemm: out_mode=%d", a.mode);
  KX_REQUIRE(a.mode != KX_GG_KV || (a.seq > 0 && a.tokens % a.seq == 0 && a.heads > 0 && a.rows == a.heads * (a.k_dim + a.v_dim) && a.cap >= a.seq && a.k_ld >= a.k_dim &&
                                    a.v_ld >= a.v_dim && a.out_v),
             "kx_dense_gemm: %d rows for %d heads, %d tokens", a.rows, a.heads, a.tokens);
  a.pairs_aligned = a.rows % 2 == 0 && (uintptr_t)a.out % 4 == 0 &&
                    (a.mode == KX_GG_KV ? (a.k_dim | a.v_dim | a.k_ld | a.v_ld) % 2 == 0 && (uintptr_t)a.out_v % 4 == 0 : a.out_stride % 2 == 0);
  KX_REQUIRE(a.mode != KX_GG_KV || a.pairs_aligned, "kx_dense_gemm: keys of %d and values of %d in rows of %d and %d", a.k_dim, a.v_dim, a.k_ld, a.v_ld);
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
