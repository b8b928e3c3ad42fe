// kx_linear.hip -- matrix products of the hybrid decoder, y[t][r] = sum_k x[t][k] w[r][k].
//
// The counterpart of matvec_bf16_k / matvec_bf16_f32_k and the kernels around them (src/kimi_exec.cu:248-298) for a
// decoder whose shapes come from its config.json: nothing here asks for a multiple of 512 columns.
//
// lin_gemv_k (up to 4 tokens): a workgroup of 8 waves builds the activation rows in LDS (kx_rows.h: residual streams
// and norm, or the gated read-out of the delta rule; of several tokens a launch in front does) while the first weight loads are under way, then every wave
// streams two rows of the matrix at a time, 8 columns per lane and load, the next pieces in flight while the present
// ones are multiplied; the epilogue stores the product, forms the gated activation of a (gate, up) pair, or updates
// all residual streams of the row.
// lin_narrow_k (bf16, up to 64 tokens): all tokens against up to 64 rows, the columns split over waves and workgroups.
// lin_gemm_k (bf16, more tokens): tiles of 256 x 256 or 128 x 128 on the matrix cores (kx_gemm_tile.h, kx_gemm_turns.h).
// In f32 from 5 tokens on tiles of 64 x 128 on the 32-bit matrix instructions; true 32-bit products.
//
// Products with experts: up to 4 tokens lin_gemv_k with a matrix per (token, choice), the routing in its prologue, and with
// the residual update's own product and the chosen experts' as one sum over consecutive segments of columns; beyond that
// the GEMMs with tiles of slots sorted by expert.
#include <algorithm>
#include <atomic>
#include "kx_common.h"
#include "kx_experts.h"
#include "kx_gemm_tile.h"
#include "kx_linear.h"
#include "kx_read_once.h"
#include "kx_rows.h"

namespace {

using kxr::Elem;
using kxtile::bf16x8;
using kxtile::f32x16;

// ---- epilogues, one output element (or pair) at a time ----
template <class T>
__device__ __forceinline__ void put_glu(const KxLinArgs &a, int t, int col, float g, float u, float weight = 1.0f) {
  g = fminf(g, a.limit);
  u = fminf(fmaxf(u, -a.limit), a.limit);
  ((T *)a.mid)[(size_t)t * a.mid_ld + col] = Elem<T>::make(g * kxr::sigmoid_for<T>(a.alpha * g) * (u + a.bias) * weight);
}
// 0.5 z (1 + tanh(y)) = z sigmoid(2 y)
template <class T>
__device__ __forceinline__ float gelu(float z) {
  return z * kxr::sigmoid_for<T>(1.5957691216057308f * __builtin_fmaf(0.044715f * z * z, z, z));
}
template <class T>
__device__ __forceinline__ void put_f32(const KxLinArgs &a, int t, int r, float y) {
  if (r < a.act_from) a.out[(size_t)t * a.out_ld + r] = y;
  else ((T *)a.mid)[(size_t)t * a.mid_ld + r - a.act_from] = Elem<T>::make(gelu<T>(y));
}
// place of matrix row r behind its token's in mid
__device__ __forceinline__ size_t head_place(const KxLinArgs &a, int r) {
  const int h = r / a.head_dim;
  return h * a.head_stride + r - h * a.head_dim;
}
template <class T>
__device__ __forceinline__ void put_head(const KxLinArgs &a, int t, int r, float y) {
  ((T *)a.mid)[(size_t)t * a.mid_ld + head_place(a, r)] = Elem<T>::make(y);
}
// variant of the activation rows that matrix rows from r on meet
__device__ __forceinline__ int variant_of(const KxLinArgs &a, int r) {
  int v = 0;
  for (int i = 1; i < a.n_var; ++i) v += r >= a.var_row[i];
  return v;
}
// EPI of the kernels: KX_LIN_F32, KX_LIN_GLU, or KX_LIN_STREAMS + number of streams (streams_any: up to KX_MAX_STREAMS)
constexpr int STREAMS_ANY = KX_LIN_STREAMS + KX_MAX_STREAMS;
__host__ __device__ constexpr int most_streams(int epi) { return epi > KX_LIN_STREAMS ? epi - KX_LIN_STREAMS : 1; }
// The streams of one element of the residual row, read early and written late.  The small matrices come through the scalar
// cache: every lane uses the same numbers and nothing writes them.
typedef const __attribute__((address_space(4))) float *ScalarPtr;
template <int EPI>
struct Streams {
  static constexpr int S = most_streams(EPI);
  float old[S];
  static __device__ __forceinline__ bool has(const KxLinArgs &a, int s) { return EPI != STREAMS_ANY || s < a.n_streams; }
  // place of token t in a.streams
  static __device__ __forceinline__ size_t of(const KxLinArgs &a, int t) { return (size_t)t * a.n_streams * a.m.rows; }
  __device__ __forceinline__ void load(const KxLinArgs &a, size_t at, int r) {
    const float *x = a.streams + at + r;
#pragma unroll
    for (int s = 0; s < S; ++s) old[s] = x[(size_t)(has(a, s) ? s : 0) * a.m.rows];
  }
  __device__ __forceinline__ void store(const KxLinArgs &a, size_t at, int r, float y) const {
    float *x = a.streams + at + r;
    if (!a.mix) {
      *x = old[0] + y;
      return;
    }
    const ScalarPtr mix = (ScalarPtr)a.mix, outw = (ScalarPtr)a.outw;
    const int n = EPI == STREAMS_ANY ? a.n_streams : S;
#pragma unroll
    for (int d = 0; d < S; ++d) {
      if (has(a, d)) {
        float v = outw[d] * y;
#pragma unroll
        for (int s = 0; s < S; ++s)
          if (has(a, s)) v = __builtin_fmaf(mix[s * n + d], old[s], v);
        x[(size_t)d * a.m.rows] = v;
      }
    }
  }
};

// matrix row of half i (0, 1) of unit k: a (gate, up) pair, or two consecutive rows
template <int EPI>
__device__ __forceinline__ int unit_row(int k, int i) {
  return EPI == KX_LIN_GLU ? (k / KX_GLU_BLOCK) * (2 * KX_GLU_BLOCK) + (k % KX_GLU_BLOCK) + i * KX_GLU_BLOCK : 2 * k + i;
}

constexpr int GEMV_WAVES = 8;
constexpr int CHUNK = 64 * 4 * 8;      // columns per pass of a wave; half of them where waves share a unit
__host__ __device__ __forceinline__ int gemv_row(int ld) { return (ld + CHUNK - 1) / CHUNK * CHUNK; }
// what a launch of lin_gemv_k goes over: one matrix for all tokens, the same with several variants of the rows, a matrix per
// (token, choice), or per token one matrix and then the chosen experts'
enum { GV_PLAIN = 0, GV_VARIANTS = 1, GV_EXPERT_IN = 2, GV_EXPERT_OUT = 3 };

// SPLIT > 1: that many waves share a unit, each with every SPLIT-th pass of its columns (gemv_split says where); a workgroup then has
// one block of units.
template <class T, int NT, int EPI, int MODE, int SPLIT>
__global__ void __launch_bounds__(GEMV_WAVES * 64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 2 ? 4 : 2)))
lin_gemv_k(KxLinArgs a, KxExpertArgs x) {
  using E = Elem<T>;
  constexpr bool OWN = MODE >= GV_EXPERT_IN;  // a token of its own per blockIdx.y
  static_assert(!OWN || NT == 1, "one token per workgroup");
  constexpr int UP = SPLIT > 1 ? 2 : 4, PASS = 64 * UP * 8, UNITS = GEMV_WAVES / SPLIT;  // UP: pieces per row of a pass
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ float red[GEMV_WAVES][2 * NT];
  __shared__ int eid[OWN ? KX_MAX_TOP : 1];
  __shared__ float ewt[MODE == GV_EXPERT_IN ? KX_MAX_TOP : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, place = wave / SPLIT, share = wave % SPLIT;  // place: of the wave's unit in its block
  const int ld = a.m.ld, np = ld >> 3, nc0 = gemv_row(ld) / PASS;
  const int nce = MODE == GV_EXPERT_OUT ? gemv_row(x.ld) / PASS : 0, nc = nc0 + (MODE == GV_EXPERT_OUT ? x.top * nce : 0);
  const int xl = nc * PASS;  // a row in LDS, with zeros up to whole passes of the wave
  const int nv = MODE == GV_VARIANTS ? a.n_var : 1;
  T *xs = (T *)lds;                                              // [NT][nv][xl]
  float *u = (float *)(lds + (size_t)NT * nv * xl * sizeof(T));  // row scratch
  const int tokens = OWN ? 1 : a.tokens, pair = MODE == GV_EXPERT_IN ? blockIdx.y : 0;
  const int tok0 = MODE == GV_EXPERT_IN ? pair / x.top : MODE == GV_EXPERT_OUT ? blockIdx.y : 0;
  const int units = (a.m.rows + 1) >> 1, nblk = (units + UNITS - 1) / UNITS;
  const T *w = (const T *)a.m.w;
  float weight = 1.0f;
  if constexpr (MODE == GV_EXPERT_IN) {
    const int choice = pair - tok0 * x.top;
    if (wave == 0) kxe::route_wave(x.logits + (size_t)tok0 * x.logits_ld, x.bias, x.experts, x.top, eid, ewt);
    __syncthreads();
    if (blockIdx.x == 0 && choice == 0 && (int)threadIdx.x < x.top) {
      x.ids[tok0 * x.top + threadIdx.x] = eid[threadIdx.x];
      x.weights[tok0 * x.top + threadIdx.x] = ewt[threadIdx.x];
    }
    w += (size_t)__builtin_amdgcn_readfirstlane(eid[choice]) * x.stride;
    weight = ewt[choice];
  }
  typename E::Raw bufA[2][UP], bufB[2][UP];
  // Past the last block the first row is asked for once more, by every wave: the number of loads in flight has to be the
  // same on every path, or the compiler waits for all of them.
  auto load = [&](typename E::Raw (&b)[2][UP], int blk, int c) {
    const int k = blk < nblk ? min(blk * UNITS + place, units - 1) : 0;
    if (blk >= nblk) c = 0;
    const T *base = w;
    int bld = ld, bnp = np;
    if constexpr (MODE == GV_EXPERT_OUT) {
      if (c >= nc0) {  // the columns go on with the experts' matrices
        const int j = (c - nc0) / nce;
        c -= nc0 + j * nce;
        base = (const T *)x.w + (size_t)__builtin_amdgcn_readfirstlane(eid[j]) * x.stride;
        bld = x.ld;
        bnp = x.ld >> 3;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const T *wr = base + (size_t)min(unit_row<EPI>(k, i), a.m.rows - 1) * bld;
#pragma unroll
      for (int j = 0; j < UP; ++j) {
        const int p = (c * UP + j) * 64 + lane;
        b[i][j] = E::stream(wr + min(p, bnp - 1) * 8);  // a lane past the row meets zeros
      }
    }
  };
  int blk = blockIdx.x, c = share;
  load(bufA, blk, c);
  if (MODE == GV_EXPERT_OUT && (int)threadIdx.x < x.top) eid[threadIdx.x] = x.ids[tok0 * x.top + threadIdx.x];
  uint32_t need = ~0u;  // variants that this workgroup's rows meet
  if constexpr (MODE == GV_VARIANTS) {
    need = 0;
    for (int k = blockIdx.x; k < nblk; k += gridDim.x) need |= 1u << variant_of(a, 2 * k * UNITS);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (t < tokens) {
      T *row = xs + (size_t)t * nv * xl;
      for (int v = 0; v < nv; ++v)
        for (int y = ld + threadIdx.x; y < nc0 * PASS; y += GEMV_WAVES * 64) row[(size_t)v * xl + y] = E::make(0.0f);
      if constexpr (MODE == GV_EXPERT_OUT) {
        const int el = nce * PASS;
        for (int j = 0; j < x.top; ++j) {
          const T *m = (const T *)x.mid + (size_t)(tok0 * x.top + j) * x.mid_ld;
          for (int y = threadIdx.x; y < el; y += GEMV_WAVES * 64) row[nc0 * PASS + j * el + y] = y < x.ld ? m[y] : E::make(0.0f);
        }
      }
      kxr::build_row<T>(a.row, tok0 + t, row, ld, u, xl, blockIdx.x == 0, need);
    }
  float acc[2 * NT];
#pragma unroll
  for (int v = 0; v < 2 * NT; ++v) acc[v] = 0.0f;
  auto step = [&](typename E::Raw (&cur)[2][UP], typename E::Raw (&nxt)[2][UP]) {  // one pass over columns of one unit per wave
    const bool last = c + SPLIT >= nc;
    const int nblk_ = last ? blk + (SPLIT > 1 ? nblk : (int)gridDim.x) : blk, nc_ = last ? share : c + SPLIT;
    // lane i * NT + t < 2 NT finishes row i of the unit for token t; what it updates is asked for ahead of the next weights
    const int unit = blk * UNITS + place, row = unit_row<EPI>(unit, lane / NT & 1), tok = NT > 1 ? lane % NT : 0;
    const bool finish = (SPLIT == 1 || share == 0) && (EPI == KX_LIN_GLU ? lane < NT && tok < tokens && unit < units : lane < 2 * NT && row < a.m.rows && tok < tokens);
    Streams<EPI> res;
    if (EPI >= KX_LIN_STREAMS && last && finish) res.load(a, Streams<EPI>::of(a, tok0 + tok), row);
    load(nxt, nblk_, nc_);
    __builtin_amdgcn_sched_barrier(0);  // these loads are on their way before the last ones are waited for
    const T *xv = xs + (MODE == GV_VARIANTS ? (size_t)variant_of(a, 2 * blk * UNITS) * xl : 0);
#pragma unroll
    for (int j = 0; j < UP; ++j) {
      const int p = (c * UP + j) * 64 + lane;
      float wf[2][8];
      E::unpack(wf[0], cur[0][j]);
      E::unpack(wf[1], cur[1][j]);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float xf[8];
        E::unpack(xf, E::cached(xv + (size_t)(NT > 1 ? min(t, tokens - 1) : 0) * nv * xl + p * 8));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          acc[t] = __builtin_fmaf(wf[0][e], xf[e], acc[t]);
          acc[NT + t] = __builtin_fmaf(wf[1][e], xf[e], acc[NT + t]);
        }
      }
    }
    if (last) {
      kxw::reduce<2 * NT, 64>(acc, lane);
      if (kxw::reduce_writer<2 * NT, 64>(lane))
#pragma unroll
        for (int j = 0; j < kxw::reduce_out<2 * NT, 64>(); ++j) red[wave][kxw::reduce_index<2 * NT, 64>(lane, j)] = acc[j];
      if constexpr (SPLIT > 1) {
        __syncthreads();
        if (finish)
#pragma unroll
          for (int k = 1; k < SPLIT; ++k) red[wave][lane] += red[wave + k][lane];  // the shares in their order
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave reads its own sums back
      if (finish) {
        if constexpr (EPI == KX_LIN_GLU) put_glu<T>(a, MODE == GV_EXPERT_IN ? pair : tok, unit, red[wave][lane], red[wave][NT + lane], weight);
        else if constexpr (EPI == KX_LIN_F32) put_f32<T>(a, tok, row, red[wave][lane]);
        else if constexpr (EPI == KX_LIN_HEADS) put_head<T>(a, tok, row, red[wave][lane]);
        else res.store(a, Streams<EPI>::of(a, tok0 + tok), row, red[wave][lane]);
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int v = 0; v < 2 * NT; ++v) acc[v] = 0.0f;
    }
    blk = nblk_;
    c = nc_;
  };
  for (;;) {
    step(bufA, bufB);
    if (blk >= nblk) break;
    step(bufB, bufA);
    if (blk >= nblk) break;
  }
}

template <class T, int KIND>
__global__ void __launch_bounds__(512) row_k(KxRowArgs a, T *out, int ld) {
  extern __shared__ float row_lds[];
  kxr::build_row<T, KIND>(a, blockIdx.x, out + (size_t)blockIdx.x * ld, ld, row_lds, (size_t)gridDim.x * ld, true);
}

// ---- bf16 GEMM ----
// Tiles of kx_gemm_tile.h; with GLU rows a wave's blocks are gate and up in turn.  GROUP: blockIdx.y is a tile of slots of one
// expert.
struct Tile {
  int m0, end;  // rows of the result
  size_t w;     // offset of the matrix
  bool alone;   // the matrix is read for this tile only
};
template <bool GROUP>
__device__ __forceinline__ bool tile_of(const KxLinArgs &a, const KxExpertArgs &e, int bm, Tile &t) {
  if constexpr (GROUP) {
    if ((int)blockIdx.y >= *e.n_tiles) return false;
    const int4 r = e.tiles[blockIdx.y];
    t.m0 = r.y;
    t.end = r.y + r.z;
    t.w = (size_t)r.x * e.stride;
    t.alone = r.w == 1;
  } else {
    t.m0 = blockIdx.y * bm;  // bm 0: all tokens
    t.end = a.tokens;
    t.w = 0;
    t.alone = true;
  }
  return true;
}
template <bool GROUP>
__device__ __forceinline__ size_t source_row(const KxExpertArgs &e, const Tile &t, int i) {
  const int s = min(t.m0 + i, t.end - 1);
  return GROUP && e.gather ? e.gather[s] : s;
}
// place of token t of a product of several sequences
__device__ __forceinline__ size_t of_sequence(const KxLinArgs &a, size_t per_seq, size_t per_token, int t) {
  const int b = (uint32_t)t / (uint32_t)a.seq;
  return b * per_seq + (size_t)(t - b * a.seq) * per_token;
}

// one tile, or a part of its columns
template <class T, class TL, int EPI, bool GROUP>
__device__ __forceinline__ void gemm_tile(uint8_t *lds, const KxLinArgs &a, const KxExpertArgs &e, const T *__restrict__ x, int x_ld, const Tile &tl, int n0, kxtile::Place at, int whole) {
  const int nb = a.m.ld / TL::COLS;
  typename TL::Sums acc;
  TL::run(lds, kxtile::cut(nb, at.part, at.of), kxtile::cut(nb, at.part + 1, at.of), [&](int r) {
    if (EPI == KX_LIN_HEADS && !GROUP && a.seq && r < TL::BM) return x + of_sequence(a, a.seq_rows, 1, min(tl.m0 + r, tl.end - 1)) * x_ld;
    return r < TL::BM ? x + source_row<GROUP>(e, tl, r) * x_ld : (const T *)a.m.w + tl.w + (size_t)min(n0 + r - TL::BM, a.m.rows - 1) * a.m.ld;
  }, acc);
  if (!GROUP && at.of > 1 &&
      !kxtile::gather<TL>(lds, acc, a.part + (size_t)(at.tile - whole) * at.of * TL::PART, a.arrived + at.tile - whole, at.of, at.part))
    return;
#pragma unroll
  for (int i = 0; i < TL::MI; ++i) {
    if constexpr (EPI == KX_LIN_GLU) {
      constexpr int STEP = KX_GLU_BLOCK / TL::SIDE;  // blocks of gate rows in front of their up rows
#pragma unroll
      for (int j = 0; j < TL::NI; ++j) {
        if (j / STEP % 2) continue;
        const int r = n0 + TL::col(j);
#pragma unroll
        for (int v = 0; v < TL::V; ++v) {
          const int t = tl.m0 + TL::row(i, v);
          if (t < tl.end && r < a.m.rows)
            put_glu<T>(a, t, (r >> 6) * KX_GLU_BLOCK + (r & 31), acc[i][j][v], acc[i][j + STEP][v], GROUP ? e.slot_weight[t] : 1.0f);
        }
      }
    } else if constexpr (EPI == KX_LIN_F32) {
#pragma unroll
      for (int j = 0; j < TL::NI; ++j) {
        const int r = n0 + TL::col(j);
#pragma unroll
        for (int v = 0; v < TL::V; ++v)
          if (tl.m0 + TL::row(i, v) < tl.end && r < a.m.rows) put_f32<T>(a, tl.m0 + TL::row(i, v), r, acc[i][j][v]);
      }
    } else if constexpr (EPI == KX_LIN_HEADS) {
      size_t to[TL::NI];  // in front of the conditions, or the divisions are made for every result: 128 x 2048 x 512 18.1 us, 11.0 now
#pragma unroll
      for (int j = 0; j < TL::NI; ++j) to[j] = head_place(a, n0 + TL::col(j));
#pragma unroll
      for (int v = 0; v < TL::V; ++v) {
        const int t = tl.m0 + TL::row(i, v);
        T *const row = (T *)a.mid + (a.seq ? of_sequence(a, a.seq_out, a.mid_ld, t) : (size_t)t * a.mid_ld);
#pragma unroll
        for (int j = 0; j < TL::NI; ++j)
          if (t < tl.end && n0 + TL::col(j) < a.m.rows) row[to[j]] = Elem<T>::make(acc[i][j][v]);
      }
    } else {
      size_t row[TL::V];
#pragma unroll
      for (int v = 0; v < TL::V; ++v) row[v] = Streams<EPI>::of(a, min(tl.m0 + TL::row(i, v), a.tokens - 1));
      constexpr int G = most_streams(EPI) > 2 ? 4 : 16;  // elements read before the first is written
      // A token's place is worked out once.  Blocks of 16 columns are half a line: those of a row follow each other (4 streams of 1024 x 1024 x
      // 4096 48.6 us block by block, 40.1 so).
      auto block = [](int x) { return TL::SIDE == 16 ? x % TL::NI : x / TL::V; };
      auto elem = [](int x) { return TL::SIDE == 16 ? x / TL::NI : x % TL::V; };
#pragma unroll
      for (int e0 = 0; e0 < TL::NI * TL::V; e0 += G) {
        Streams<EPI> res[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int j = block(e0 + u), v = elem(e0 + u);
          res[u].load(a, row[v], min(n0 + TL::col(j), a.m.rows - 1));
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int j = block(e0 + u), v = elem(e0 + u), r = n0 + TL::col(j);
          if (tl.m0 + TL::row(i, v) < a.tokens && r < a.m.rows) res[u].store(a, row[v], r, acc[i][j][v]);
        }
      }
    }
  }
}

// Tiles of up to 256 slots of an expert.  Its last one takes the kernel of as many quarters as it fills: 2 of them are as long as two tiles of 128 x 128.
template <class TL>
constexpr bool LISTED_LARGE = false;
template <>
constexpr bool LISTED_LARGE<kxtile::Large> = true;

template <class T, class TL, int EPI, bool GROUP>
__global__ void __launch_bounds__(TL::THREADS, TL::WAVES_PER_SIMD) lin_gemm_k(KxLinArgs a, KxExpertArgs e, const T *__restrict__ x, int x_ld, kxtile::Share share) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  Tile tl;
  if constexpr (GROUP) {
    if (!tile_of<true>(a, e, TL::BM, tl)) return;
    const int n0 = blockIdx.x * TL::BN;
    if constexpr (LISTED_LARGE<TL>) {
      const int n = tl.end - tl.m0;
      if (n <= 64) return gemm_tile<T, kxtile::Turns<false, 1>, EPI, true>(lds, a, e, x, x_ld, tl, n0, {0, 0, 1}, 0);
      if (n <= 128) return gemm_tile<T, kxtile::Turns<false, 2>, EPI, true>(lds, a, e, x, x_ld, tl, n0, {0, 0, 1}, 0);
      if (n <= 192) return gemm_tile<T, kxtile::Turns<false, 3>, EPI, true>(lds, a, e, x, x_ld, tl, n0, {0, 0, 1}, 0);
    }
    gemm_tile<T, TL, EPI, true>(lds, a, e, x, x_ld, tl, n0, {0, 0, 1}, 0);
  } else {
    const int tm = (a.tokens + TL::BM - 1) / TL::BM;
    const kxtile::Place at = kxtile::place_of(blockIdx.x, tm * ((a.m.rows + TL::BN - 1) / TL::BN), share);
    const int n0 = at.tile / tm * TL::BN;
    tl.m0 = at.tile % tm * TL::BM;
    tl.end = a.tokens;
    tl.w = 0;
    gemm_tile<T, TL, EPI, false>(lds, a, e, x + (size_t)variant_of(a, n0) * a.tokens * x_ld, x_ld, tl, n0, at, share.whole);
  }
}

// ---- bf16 products of few tokens ----
// Bound by the stream of the matrix.  A workgroup of 8 waves owns a share of up to 64 rows (kxtile::even_groups; with GLU rows a block of gate and its block of up),
// all tokens, and one of `splits` parts of the columns, so that a matrix of few rows still has a workgroup or two for every CU:
// a tile per 128 rows alone is 16 workgroups for 2048 rows (90 us for 8 tokens against 2048 x 10240; 11 us here).  The columns
// are walked in blocks of 128, each two halves of 64 in the layout of the tiles above, through a ring of NS blocks; wave w
// multiplies 16 columns of each half for row block w % 2, so that four waves hold sums of the same outputs, which meet in LDS.
// With several parts the sums go to memory and the workgroup that arrives last (kx_arrive.h) adds the parts in their order,
// whoever it is, and runs the epilogue: results do not depend on timing.  Token rows past the last are never copied: what the
// LDS holds there only feeds sums that are not stored.  Large matrices are copied nontemporally, whole lines of them (kx_read_once.h).
// Not those of an expert with several tiles, which find its rows in the L2: 40 tokens to the same 4 of 128 experts of 3 x 4096 x 1536 101.8 us so, 88.7 now, 96 tokens 139.5
// and 119.2; 96 tokens spread unevenly 264.6 and 242.3.
constexpr int NARROW_ROWS = 64, NARROW_MAX_SPLITS = 16;
template <int MI, int EPI, bool GROUP>
__global__ void __launch_bounds__(512, MI == 1 ? 4 : 2) lin_narrow_k(KxLinArgs a, KxExpertArgs e, const uint16_t *__restrict__ x, int x_ld, int splits, bool once, int share, int extra) {
  constexpr int ROWS = NARROW_ROWS + 32 * MI, HALF = ROWS * 128, STAGE = 2 * HALF, NS = MI == 1 ? 3 : 4, CPW = 2 + MI;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ int last_one;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31, h = lane >> 5, part = GROUP ? 0 : blockIdx.y;
  // share rows each, the first `extra` workgroups one more (divisions in 64 bits here cost a workgroup 0.5 us)
  const int bx = blockIdx.x, n0 = bx * share + min(bx, extra), n1 = min(n0 + share + (bx < extra), a.m.rows);
  Tile tl;
  if (!tile_of<GROUP>(a, e, 0, tl)) return;
  const int m0 = tl.m0, tokens = tl.end - m0;
  const bool nt = once && tl.alone;
  x += (size_t)variant_of(a, n0) * a.tokens * x_ld;
  const int nh = a.m.ld >> 6, nb = (nh + 1) >> 1;  // halves, blocks
  const int b0 = (int)((long)nb * part / splits), b1 = (int)((long)nb * (part + 1) / splits);
  // copy instructions of a block: 16 of 8 matrix rows, two per wave; then 8 tokens at a time of both halves, MI per wave (the
  // last one again where there are fewer, so that every wave waits for the same number)
  const uint16_t *src[CPW];
  uint32_t dst[CPW];
  int half[CPW];
  const int groups = (tokens + 7) >> 3, sub = lane >> 3;
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    if (i < 2) {
      const int q = wave * 2 + i, row = (q & 7) * 8 + sub;
      half[i] = q >> 3;
      src[i] = (const uint16_t *)a.m.w + tl.w + (size_t)min(n0 + row, n1 - 1) * a.m.ld + ((lane & 7) ^ sub) * 8;
      dst[i] = half[i] * HALF + (q & 7) * 1024;
    } else {
      const int q = min(wave + 8 * (i - 2), 2 * groups - 1);
      half[i] = q >= groups;
      const int g = q - half[i] * groups;
      src[i] = x + source_row<GROUP>(e, tl, g * 8 + sub) * x_ld + ((lane & 7) ^ sub) * 8;
      dst[i] = half[i] * HALF + NARROW_ROWS * 128 + g * 1024;
    }
  }
  auto copy = [&](int b, int stage) {
    const uint32_t st = lds0 + stage * STAGE;
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const uint16_t *const from = src[i] + min(2 * b + half[i], nh - 1) * 64;
      const uint32_t to = __builtin_amdgcn_readfirstlane(st + dst[i]);
      if (i < 2 && nt) kx_copy16_to_lds_once(from, to);  // the matrix
      else kx_copy16_to_lds(from, to);
    }
  };
  f32x16 acc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
  const int p = ((2 * (wave >> 1) + h) ^ (lr & 7)) * 16, wrow = ((wave & 1) * 32 + lr) * 128 + p, xrow = (NARROW_ROWS + lr) * 128 + p;
#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    if (b0 + i < b1) copy(b0 + i, i);
  int stage = 0;
  for (int b = b0; b < b1; ++b) {
    const int behind = min(b1 - 1 - b, NS - 2);  // blocks asked for after this one
    if (behind >= 2) kx_wait_copies<2 * CPW>();
    else if (behind == 1) kx_wait_copies<CPW>();
    else kx_wait_copies<0>();
    kx_lds_barrier();  // block b is in LDS for every wave, and every wave is done with block b - 1
    if (b + NS - 1 < b1) copy(b + NS - 1, stage == 0 ? NS - 1 : stage - 1);
    const uint8_t *st = lds + stage * STAGE;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (2 * b + u < nh) {
        const bf16x8 wb = *(const bf16x8 *)(st + u * HALF + wrow);
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)(st + u * HALF + xrow + i * 32 * 128), wb, acc[i], 0, 0, 0);
      }
    }
    stage = stage == NS - 1 ? 0 : stage + 1;
  }
  kx_lds_barrier();  // the ring takes the sums: [wave][token][row of the wave's block]
  float *sums = (float *)lds;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) sums[(wave * MI * 32 + i * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * 32 + lr] = acc[i][v];
  __syncthreads();
  auto own = [&](int t, int r) {  // this workgroup's sum for token t and its row r
    const float *s = sums + (((r >> 5) * MI * 32 + t) * 32 + (r & 31));
    return ((s[0] + s[2 * MI * 1024]) + s[4 * MI * 1024]) + s[6 * MI * 1024];
  };
  const int outs = tokens * NARROW_ROWS;
  float *mine = a.part + (size_t)blockIdx.x * splits * outs;
  if (splits > 1) {
    for (int i = threadIdx.x; i < outs; i += 512) kx_arrive_store(mine + (size_t)part * outs + i, own(i >> 6, i & 63));
    kx_arrive_writes_done();
    __syncthreads();
    if (threadIdx.x == 0) last_one = kx_arrive_is_last(a.arrived + blockIdx.x, splits);
    __syncthreads();
    if (!last_one) return;
    if (threadIdx.x == 0) kx_arrive_reset(a.arrived + blockIdx.x);
  }
  auto value = [&](int t, int r) {
    if (splits == 1) return own(t, r);
    float v[NARROW_MAX_SPLITS];
#pragma unroll
    for (int s = 0; s < NARROW_MAX_SPLITS; ++s) v[s] = s < splits ? kx_arrive_load(mine + (size_t)s * outs + t * NARROW_ROWS + r) : 0.0f;
    float y = v[0];
#pragma unroll
    for (int s = 1; s < NARROW_MAX_SPLITS; ++s) y += v[s];
    return y;
  };
  if constexpr (EPI == KX_LIN_GLU) {
    for (int i = threadIdx.x; i < tokens * 32; i += 512) {
      const int t = i >> 5, c = i & 31;
      if (n0 + c < a.m.rows) put_glu<uint16_t>(a, m0 + t, n0 / 2 + c, value(t, c), value(t, 32 + c), GROUP ? e.slot_weight[m0 + t] : 1.0f);
    }
  } else {
    for (int i = threadIdx.x; i < outs; i += 512) {
      const int t = m0 + (i >> 6), r = n0 + (i & 63);
      if (r >= n1) continue;
      Streams<EPI> res;
      if constexpr (EPI >= KX_LIN_STREAMS) res.load(a, Streams<EPI>::of(a, t), r);
      const float y = value(i >> 6, i & 63);
      if constexpr (EPI == KX_LIN_F32) put_f32<uint16_t>(a, t, r, y);
      else if constexpr (EPI == KX_LIN_HEADS) put_head<uint16_t>(a, t, r, y);
      else res.store(a, Streams<EPI>::of(a, t), r, y);
    }
  }
}

constexpr size_t GEMV_LDS = 150 * 1024;

// Waves per unit of two rows: a workgroup has 16 rows with one, 8 with two, 4 with four.  As many as let the CU with the most rows have
// the fewest, without more workgroups than run at once and with a pass for every wave.  2048 x 2048 and 2048 x 8192, one token, are 128
// workgroups of 16 rows: 8.0 us on average, 7.1 as 256 of 8.
int gemv_split(int rows, int passes, int grid_y) {
  const long cus = std::max(1, kx_device_cus());
  long best = 1, least = 0;
  for (int s = 1; s <= 4; s *= 2) {
    const long groups = (long)kx_cdiv((rows + 1) / 2, GEMV_WAVES / s) * grid_y, most = (groups + cus - 1) / cus * (16 / s);
    if (s > 1 && (groups > 2 * cus || passes < s)) break;
    if (s == 1 || most < least) best = s, least = most;
  }
  return (int)best;
}
// `lds` bytes of the dynamic part; grid_y: 1, or the tokens or (token, choice) pairs
template <class T, int NT, int EPI, int MODE, int SPLIT = 1>
int gemv_launch(const KxLinArgs &a, const KxExpertArgs &x, size_t lds, int grid_y, hipStream_t st) {
  if constexpr (SPLIT == 1 && EPI >= KX_LIN_STREAMS) {
    const int split = gemv_split(a.m.rows, kx_cdiv(a.m.ld, CHUNK / 2), grid_y);
    if (split == 2) return gemv_launch<T, NT, EPI, MODE, 2>(a, x, lds, grid_y, st);
    if (split == 4) return gemv_launch<T, NT, EPI, MODE, 4>(a, x, lds, grid_y, st);
  }
  static std::atomic<bool> attr{false};  // setting it twice from two threads is harmless
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)lin_gemv_k<T, NT, EPI, MODE, SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)GEMV_LDS));
    attr = true;
  }
  const int nblk = kx_cdiv((a.m.rows + 1) / 2, GEMV_WAVES / SPLIT), most = SPLIT > 1 ? nblk : std::max(1, 2 * std::max(1, kx_device_cus()) / grid_y);
  hipLaunchKernelGGL((lin_gemv_k<T, NT, EPI, MODE, SPLIT>), dim3(std::min(nblk, most), grid_y), dim3(GEMV_WAVES * 64), lds, st, a, x);
  KX_LAUNCH_CHECK();
  return KX_OK;
}
template <class T, int NT, int EPI>
int gemv_nt(const KxLinArgs &a, size_t lds, hipStream_t st) {
  if constexpr (EPI == KX_LIN_F32)
    if (a.row.kind == KX_ROW_SHIFT) return gemv_launch<T, NT, EPI, GV_VARIANTS>(a, KxExpertArgs(), lds, 1, st);
  return gemv_launch<T, NT, EPI, GV_PLAIN>(a, KxExpertArgs(), lds, 1, st);
}

template <class T, int KIND>
int rows_kind(const KxRowArgs &r, int tokens, T *out, int ld, hipStream_t st) {
  const size_t scratch = (size_t)kx_row_scratch(r) * 4;
  KX_REQUIRE(out && scratch <= 160 * 1024 - 1024, "kx_linear: rows of %d columns do not fit a workgroup", r.cols);
  static std::atomic<bool> attr{false};
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)row_k<T, KIND>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 1024));
    attr = true;
  }
  // a workgroup per token: twice the threads where the tokens do not fill the chip
  hipLaunchKernelGGL((row_k<T, KIND>), dim3(tokens), dim3(tokens <= 256 ? 512 : 256), scratch, st, r, out, ld);
  KX_LAUNCH_CHECK();
  return KX_OK;
}
template <class T>
int rows_launch(const KxRowArgs &r, int tokens, T *out, int ld, hipStream_t st) {
  switch (r.kind) {
    case KX_ROW_NORM: return rows_kind<T, KX_ROW_NORM>(r, tokens, out, ld, st);
    case KX_ROW_GATED: return rows_kind<T, KX_ROW_GATED>(r, tokens, out, ld, st);
    case KX_ROW_SHIFT: return rows_kind<T, KX_ROW_SHIFT>(r, tokens, out, ld, st);
    case KX_ROW_TANH: return rows_kind<T, KX_ROW_TANH>(r, tokens, out, ld, st);
  }
  return rows_kind<T, KX_ROW_PLAIN>(r, tokens, out, ld, st);
}

// Parts of the columns so that about two workgroups per CU run at once, each of at least 512 columns, as the scratch allows.
int narrow_splits(const KxLinArgs &a, int groups) {
  if (!a.part || !a.arrived) return 1;
  const int blocks = kx_cdiv(a.m.ld, 128);
  int s = std::min({2 * std::max(1, kx_device_cus()) / groups, blocks / 4, NARROW_MAX_SPLITS});
  s = (int)std::min<size_t>(s, a.part_floats / ((size_t)groups * NARROW_ROWS * a.tokens));
  return s < 2 || groups > a.arrivals ? 1 : s;
}
template <int EPI, bool GROUP>
int narrow_launch(const KxLinArgs &a, const KxExpertArgs &e, const uint16_t *x, int x_ld, hipStream_t st) {
  static std::atomic<bool> attr{false};
  constexpr size_t lds[2] = {3 * 2 * (NARROW_ROWS + 32) * 128, 4 * 2 * (NARROW_ROWS + 64) * 128};
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)lin_narrow_k<1, EPI, GROUP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds[0]));
    if constexpr (!GROUP) KX_HIP(hipFuncSetAttribute((const void *)lin_narrow_k<2, EPI, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds[1]));
    attr = true;
  }
  int groups = kx_cdiv(a.m.rows, NARROW_ROWS);
  const int splits = GROUP ? 1 : narrow_splits(a, groups);
  int share = NARROW_ROWS, extra = 0;  // rows of a workgroup
  if (!GROUP && EPI != KX_LIN_GLU && a.n_var == 1) {  // GLU: blocks of gate and up; variants begin at multiples of 128 rows
    const bool parts = splits > 1;
    const int even = kxtile::even_groups(a.m.rows, a.m.ld, groups, splits, parts ? a.part_floats / ((size_t)NARROW_ROWS * a.tokens) : (size_t)-1, parts ? a.arrivals : a.m.rows,
                                         std::max(1, kx_device_cus()));
    if (even > groups) groups = even, share = a.m.rows / even, extra = a.m.rows % even;
  }
  const dim3 grid(groups, GROUP ? e.max_tiles : splits);
  const bool once = GROUP ? kxonce::experts((size_t)e.experts * e.stride * 2, (size_t)a.model_mb << 20) : kxonce::matrix((size_t)a.m.rows * a.m.ld * 2, (size_t)a.model_mb << 20);
  if constexpr (GROUP) hipLaunchKernelGGL((lin_narrow_k<1, EPI, true>), grid, dim3(512), lds[0], st, a, e, x, x_ld, splits, once, share, extra);
  else if (a.tokens <= 32) hipLaunchKernelGGL((lin_narrow_k<1, EPI, false>), grid, dim3(512), lds[0], st, a, e, x, x_ld, splits, once, share, extra);
  else hipLaunchKernelGGL((lin_narrow_k<2, EPI, false>), grid, dim3(512), lds[1], st, a, e, x, x_ld, splits, once, share, extra);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

// 64 slots of an expert.  Three workgroups per CU, or two by asking for more LDS where even routing then ends sooner: bound by the
// stream of the matrices, a round of workgroups takes as long as there are of them per CU.  Experts of 3 x 2048 x 1024, 64
// and 128 tokens to 8 of 64, which make 1024 tiles: 228 and 251 us with two, 244 and 268 with three; 3 x 1536 x 768, 768 tiles: 149 and 138.
// Where few experts have the tokens three are better throughout (1000 tokens to 4 of 128, all among 8: 422 with two, 375 with
// three), but that is known on the device alone.  How many tiles there are is only certain while nearly every expert makes do
// with one: with more than 16 pairs per expert two are not taken (256 tokens, even 262 with two, 281 with three, a few experts with more
// tokens 293 and 277; 760 tokens 343 and 327).
typedef kxtile::Tile<uint16_t, 2, 2, 1, 2, 4> SmallSlots;
int small_slots_lds(const KxLinArgs &a, const KxExpertArgs &e) {
  const long pairs = (long)a.tokens * e.top, used = std::min<long>(pairs, e.experts), cus = std::max(1, kx_device_cus());
  if (pairs > 16 * used) return SmallSlots::LEAST_LDS;
  const long tiles = used * kx_cdiv(a.m.rows, SmallSlots::BN);
  const long two = (tiles + 2 * cus - 1) / (2 * cus) * 2, three = (tiles + 3 * cus - 1) / (3 * cus) * 3;
  return two < three ? SmallSlots::LDS : SmallSlots::LEAST_LDS;
}
template <class T, class TL, int EPI, bool GROUP>
int tile_launch(const KxLinArgs &a, const KxExpertArgs &e, const T *x, int x_ld, kxtile::Share share, hipStream_t st, int lds = TL::LDS) {
  static std::atomic<bool> attr{false};
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)lin_gemm_k<T, TL, EPI, GROUP>, hipFuncAttributeMaxDynamicSharedMemorySize, TL::LDS));
    attr = true;
  }
  const int tn = kx_cdiv(a.m.rows, TL::BN);
  const dim3 grid = GROUP ? dim3(tn, e.max_tiles) : dim3(share.grid(tn * kx_cdiv(a.tokens, TL::BM)));
  hipLaunchKernelGGL((lin_gemm_k<T, TL, EPI, GROUP>), grid, dim3(TL::THREADS), lds, st, a, e, x, x_ld, share);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

// GEMM over rows in memory; GROUP: e.max_tiles tiles of slots
template <class T, int EPI, bool GROUP>
int gemm_launch(const KxLinArgs &a, const KxExpertArgs &e, const T *x, int x_ld, hipStream_t st) {
  KX_REQUIRE(x && x_ld >= a.m.ld, "kx_linear: activation rows of %d, the matrix has %d", x_ld, a.m.ld);
  if constexpr (sizeof(T) == 2 && GROUP)
    if (e.tile_slots <= 32) return narrow_launch<EPI, true>(a, e, x, x_ld, st);
  const size_t room = a.part ? a.part_floats : 0;
  const int arrivals = a.arrived ? a.arrivals : 0, cus = std::max(1, kx_device_cus());
  if constexpr (sizeof(T) == 4) {
    const kxtile::Share s = GROUP ? kxtile::Share{0, 1} : kxtile::choose_single(a.tokens, a.m.rows, a.m.ld / kxtile::Single::COLS, room, arrivals, cus);
    return tile_launch<float, kxtile::Single, EPI, GROUP>(a, e, x, x_ld, s, st);
  } else if constexpr (GROUP) {
    if (e.tile_slots > 128) return tile_launch<uint16_t, kxtile::Large, EPI, true>(a, e, x, x_ld, {0, 1}, st);
    return e.tile_slots > 64 ? tile_launch<uint16_t, kxtile::Medium, EPI, true>(a, e, x, x_ld, {0, 1}, st) : tile_launch<uint16_t, SmallSlots, EPI, true>(a, e, x, x_ld, {0, 1}, st, small_slots_lds(a, e));
  } else {
    const kxtile::Choice c = kxtile::choose(a.tokens, a.m.rows, a.m.ld >> 6, room, arrivals, cus);
    if (c.large && a.n_var == 1) return tile_launch<uint16_t, kxtile::Large, EPI, false>(a, e, x, x_ld, c.s, st);  // variants begin at multiples of 128 rows
    // with variants a choice of large tiles is taken as medium ones, whole
    const kxtile::Share whole = {kx_cdiv(a.tokens, kxtile::Medium::BM) * kx_cdiv(a.m.rows, kxtile::Medium::BN), 1};
    if (c.twin) return tile_launch<uint16_t, kxtile::Twin, EPI, false>(a, e, x, x_ld, c.s, st);
    return tile_launch<uint16_t, kxtile::Medium, EPI, false>(a, e, x, x_ld, c.large ? whole : c.s, st);
  }
}

template <class T, int EPI>
int linear_epi(const KxLinArgs &a, void *row_buf, hipStream_t st) {
  const size_t scratch = (size_t)kx_row_scratch(a.row) * 4;
  if (a.tokens <= KX_GEMV_TOKENS) {
    const int nt = a.tokens > 2 ? 4 : a.tokens;
    const size_t lds = (size_t)nt * kx_row_variants(a.row) * gemv_row(a.m.ld) * sizeof(T) + scratch;
    if (lds <= GEMV_LDS) {
      // Rows of several tokens are built by a launch of their own, a workgroup per token: in the product's, where a workgroup builds them one after the other, each takes 3
      // us that the matrix waits.  The rows are the same.  us, before / now: 4 tokens of two normed streams 16384 x 2048 26.9 / 20.2, 6208 x
      // 2048 21.6 / 13.9, 4096 x 1024 14.6 / 10.9, a gated read-out 2048 x 2048 13.2 / 10.2; two tokens 19.4 / 18.3, 14.2 / 12.4 and 9.5 / 9.5, but the
      // gated one 8.5 / 9.1.  Small products gain as well, one stream, two tokens and four: 256 x 256 7.7 / 7.5 and 12.7 / 9.4, 768 x 768 8.6 / 8.1 and 13.7 / 9.8, 64 x 2048 9.1 /
      // 8.5 and 14.9 / 10.0; in 32 bits 256 x 256 8.7 / 8.3 and 13.8 / 10.4, 768 x 768 10.2 / 9.9 and 15.5 / 11.6, 8192 x 2048 29.1 / 24.0 and 39.5 / 26.6.
      if (row_buf && (uintptr_t)row_buf % 16 == 0 && ((nt > 1 && a.row.kind == KX_ROW_NORM) || (nt == 4 && a.row.kind == KX_ROW_GATED))) {
        const int rc = rows_launch<T>(a.row, a.tokens, (T *)row_buf, a.m.ld, st);
        if (rc) return rc;
        KxLinArgs b = a;
        b.row = KxRowArgs();
        b.row.cols = a.row.cols; b.row.x = row_buf; b.row.x_ld = a.m.ld;
        const size_t row = gemv_row(a.m.ld) * sizeof(T);
        return nt == 2 ? gemv_nt<T, 2, EPI>(b, 2 * row, st) : gemv_nt<T, 4, EPI>(b, 4 * row, st);
      }
      if (nt == 1) return gemv_nt<T, 1, EPI>(a, lds, st);
      if (nt == 2) return gemv_nt<T, 2, EPI>(a, lds, st);
      return gemv_nt<T, 4, EPI>(a, lds, st);
    }
  }
  const T *x = (const T *)a.row.x;
  int x_ld = a.row.x_ld;
  if (a.row.kind != KX_ROW_PLAIN) {
    int rc = rows_launch<T>(a.row, a.tokens, (T *)row_buf, a.m.ld, st);
    if (rc) return rc;
    x = (const T *)row_buf;
    x_ld = a.m.ld;
  }
  KX_REQUIRE(a.row.kind != KX_ROW_PLAIN || !a.row.rows_map, "kx_linear: mapped rows have to be built");
  KX_REQUIRE(x && x_ld >= a.m.ld, "kx_linear: activation rows of %d, the matrix has %d", x_ld, a.m.ld);
  if constexpr (sizeof(T) == 2 && EPI == STREAMS_ANY) {  // more streams than the matrix-core kernel is built for: a few tokens at a time
    KX_REQUIRE(gemv_row(a.m.ld) * sizeof(T) <= GEMV_LDS, "kx_linear: rows of %d columns with %d streams do not fit a workgroup", a.m.ld, a.n_streams);
    const int most = (size_t)4 * gemv_row(a.m.ld) * sizeof(T) <= GEMV_LDS ? 4 : 1;
    for (int t = 0; t < a.tokens; t += most) {
      KxLinArgs b = a;
      b.row = KxRowArgs();
      b.row.cols = a.row.cols; b.row.x = x + (size_t)t * x_ld; b.row.x_ld = x_ld;
      b.tokens = std::min(most, a.tokens - t);
      b.streams = a.streams + (size_t)t * a.n_streams * a.m.rows;
      const size_t lds = (size_t)most * gemv_row(a.m.ld) * sizeof(T);
      int rc = most == 4 ? gemv_nt<T, 4, EPI>(b, lds, st) : gemv_nt<T, 1, EPI>(b, lds, st);
      if (rc) return rc;
    }
    return KX_OK;
  } else {
    if constexpr (sizeof(T) == 2)
      if (a.tokens <= KX_NARROW_TOKENS) return narrow_launch<EPI, false>(a, KxExpertArgs(), x, x_ld, st);
    return gemm_launch<T, EPI, false>(a, KxExpertArgs(), x, x_ld, st);
  }
}

int check_matrix(const KxLinArgs &a) {
  KX_REQUIRE(a.m.w && a.m.rows > 0 && a.m.cols > 0 && a.m.ld >= a.m.cols && a.m.ld % KX_LD == 0, "kx_linear: matrix of %d x %d (%d)", a.m.rows, a.m.cols, a.m.ld);
  KX_REQUIRE(a.tokens > 0 && a.row.cols == a.m.cols, "kx_linear: tokens=%d, rows of %d for %d columns", a.tokens, a.row.cols, a.m.cols);
  KX_REQUIRE(a.epi != KX_LIN_GLU || a.m.rows % (2 * KX_GLU_BLOCK) == 0, "kx_linear: %d rows are no (gate, up) blocks", a.m.rows);
  KX_REQUIRE(a.n_streams >= 1 && a.n_streams <= KX_MAX_STREAMS && (a.mix || a.n_streams == 1), "kx_linear: %d streams", a.n_streams);
  KX_REQUIRE(a.epi != KX_LIN_F32 || a.act_from >= a.m.rows || (a.mid && a.mid_ld >= a.m.rows - a.act_from), "kx_linear: no room for %d activations", a.m.rows - a.act_from);
  KX_REQUIRE(a.epi != KX_LIN_HEADS || (a.head_dim > 0 && a.mid), "kx_linear: heads of %d", a.head_dim);
  KX_REQUIRE(!a.seq || (a.seq > 0 && a.epi == KX_LIN_HEADS && a.row.kind == KX_ROW_PLAIN && a.tokens > KX_NARROW_TOKENS && a.tokens % a.seq == 0), "kx_linear: %d tokens in sequences of %d",
             a.tokens, a.seq);
  KX_REQUIRE(a.row.kind != KX_ROW_SHIFT || (a.epi == KX_LIN_F32 && a.row.n_streams == 1 && a.row.batch > 0 && a.row.tokens == a.tokens && a.row.prev && a.row.prev_out &&
                                            a.row.prev != a.row.prev_out && a.n_var == a.row.n_mix + 1 && a.n_var <= KX_MAX_VARIANTS),
             "kx_linear: %d mixes of %d tokens", a.row.n_mix, a.row.tokens);
  for (int v = 1; v < a.n_var; ++v) KX_REQUIRE(a.var_row[v] % KX_VARIANT_ROWS == 0, "kx_linear: variant %d from row %d on", v, a.var_row[v]);
  KX_REQUIRE(!a.row.tail || (a.row.kind == KX_ROW_GATED && a.row.head_ld % KX_LD == 0 && a.row.head_ld >= a.row.heads * a.row.vdim && a.row.tail_ld >= a.m.ld - a.row.head_ld),
             "kx_linear: a row of %d and its tail of %d", a.row.head_ld, a.row.tail_ld);
  return KX_OK;
}

template <class T>
int linear(const KxLinArgs &a, void *row_buf, hipStream_t st) {
  int rc = check_matrix(a);
  if (rc) return rc;
  if (a.epi == KX_LIN_F32) return linear_epi<T, KX_LIN_F32>(a, row_buf, st);
  if (a.epi == KX_LIN_GLU) return linear_epi<T, KX_LIN_GLU>(a, row_buf, st);
  if (a.epi == KX_LIN_HEADS) return linear_epi<T, KX_LIN_HEADS>(a, row_buf, st);
  if (a.n_streams == 1) return linear_epi<T, KX_LIN_STREAMS + 1>(a, row_buf, st);
  if (a.n_streams == 2) return linear_epi<T, KX_LIN_STREAMS + 2>(a, row_buf, st);
  if constexpr (sizeof(T) == 2) {
    if (a.n_streams == 3) return linear_epi<T, KX_LIN_STREAMS + 3>(a, row_buf, st);
    if (a.n_streams == 4) return linear_epi<T, KX_LIN_STREAMS + 4>(a, row_buf, st);
  }
  return linear_epi<T, STREAMS_ANY>(a, row_buf, st);
}

template <class T>
size_t expert_in_lds(const KxLinArgs &a) { return (size_t)gemv_row(a.m.ld) * sizeof(T) + (size_t)kx_row_scratch(a.row) * 4; }
template <class T>
size_t expert_out_lds(const KxLinArgs &a, const KxExpertArgs &e) {
  return ((size_t)gemv_row(a.m.ld) + (size_t)e.top * gemv_row(e.ld)) * sizeof(T) + (size_t)kx_row_scratch(a.row) * 4;
}
int check_experts(const KxExpertArgs &e) {
  KX_REQUIRE(e.experts > 0 && e.experts <= KX_MAX_EXPERTS && e.top > 0 && e.top <= e.experts && e.top <= KX_MAX_TOP, "experts: %d of %d", e.top, e.experts);
  return KX_OK;
}
template <class T>
int expert_in(const KxLinArgs &a, const KxExpertArgs &e, hipStream_t st) {
  KX_REQUIRE(a.epi == KX_LIN_GLU && e.logits && e.ids && e.weights && expert_in_lds<T>(a) <= GEMV_LDS, "experts: rows of %d columns", a.m.cols);
  return gemv_launch<T, 1, KX_LIN_GLU, GV_EXPERT_IN>(a, e, expert_in_lds<T>(a), a.tokens * e.top, st);
}
template <class T>
int expert_out(const KxLinArgs &a, const KxExpertArgs &e, hipStream_t st) {
  KX_REQUIRE(a.epi == KX_LIN_STREAMS && a.n_streams == 1 && !a.mix && e.ids && e.w && e.mid && e.mid_ld >= e.ld && e.ld % KX_LD == 0 && expert_out_lds<T>(a, e) <= GEMV_LDS,
             "experts: rows of %d and %d x %d columns", a.m.cols, e.top, e.ld);
  return gemv_launch<T, 1, KX_LIN_STREAMS + 1, GV_EXPERT_OUT>(a, e, expert_out_lds<T>(a, e), a.tokens, st);
}
template <class T>
int expert_gemm(const KxLinArgs &a, const KxExpertArgs &e, const T *x, int x_ld, hipStream_t st) {
  KX_REQUIRE(e.tiles && e.n_tiles && e.max_tiles > 0 && e.max_tiles <= 65535 && a.n_var == 1, "experts: %d tiles", e.max_tiles);
  KX_REQUIRE(e.tile_slots > 0 && e.tile_slots <= (sizeof(T) == 4 ? 64 : 256), "experts: tiles of %d", e.tile_slots);
  KX_REQUIRE(a.epi != KX_LIN_GLU || e.slot_weight, "experts: no weights");
  if (a.epi == KX_LIN_GLU) return gemm_launch<T, KX_LIN_GLU, true>(a, e, x, x_ld, st);
  KX_REQUIRE(a.epi == KX_LIN_F32, "experts: epilogue %d", a.epi);
  return gemm_launch<T, KX_LIN_F32, true>(a, e, x, x_ld, st);
}

}  // namespace

int kx_linear_launch(bool f32, const KxLinArgs &a, void *row_buf, hipStream_t st) {
  return f32 ? linear<float>(a, row_buf, st) : linear<uint16_t>(a, row_buf, st);
}
int kx_rows_launch(bool f32, const KxRowArgs &r, int tokens, void *out, int ld, hipStream_t st) {
  return f32 ? rows_launch<float>(r, tokens, (float *)out, ld, st) : rows_launch<uint16_t>(r, tokens, (uint16_t *)out, ld, st);
}
bool kx_expert_small(bool f32, const KxLinArgs &in, const KxLinArgs &out, const KxExpertArgs &e, int tokens) {
  return tokens <= KX_GEMV_TOKENS && (f32 ? expert_in_lds<float>(in) <= GEMV_LDS && expert_out_lds<float>(out, e) <= GEMV_LDS
                                          : expert_in_lds<uint16_t>(in) <= GEMV_LDS && expert_out_lds<uint16_t>(out, e) <= GEMV_LDS);
}
int kx_expert_in_launch(bool f32, const KxLinArgs &a, const KxExpertArgs &e, hipStream_t st) {
  int rc = check_matrix(a);
  if (rc || (rc = check_experts(e))) return rc;
  return f32 ? expert_in<float>(a, e, st) : expert_in<uint16_t>(a, e, st);
}
int kx_expert_out_launch(bool f32, const KxLinArgs &a, const KxExpertArgs &e, hipStream_t st) {
  int rc = check_matrix(a);
  if (rc || (rc = check_experts(e))) return rc;
  return f32 ? expert_out<float>(a, e, st) : expert_out<uint16_t>(a, e, st);
}
int kx_expert_gemm_launch(bool f32, const KxLinArgs &a, const KxExpertArgs &e, const void *x, int x_ld, hipStream_t st) {
  int rc = check_matrix(a);
  if (rc) return rc;
  return f32 ? expert_gemm<float>(a, e, (const float *)x, x_ld, st) : expert_gemm<uint16_t>(a, e, (const uint16_t *)x, x_ld, st);
}
