// kx_window.hip -- see kx_window.h.
//
// The counterpart of the tiled attention over cached keys and values (attn_tile_* and tiled_attention,
// src/kimi_exec.cu:414-475, :692-716) for a window with pooled blocks; the scores and the softmax are 32-bit.
//
// One token per sequence: win_partial_k<T, true>.  A workgroup takes up to CH keys of one key/value head for one token:
// it norms the query itself, and the workgroup that holds the newest key also norms that key, writes the cache rows
// and, where a block completes, its means.  win_merge_k merges the parts, adds the sink and applies the output gate.
// Steps of several positions: win_prep_k norms the projections and writes queries and cache rows, win_pool_k the
// blocks that complete, and then win_flash_k (bf16) or win_flash_f32_k attend on the matrix cores, or win_partial_k<T, false> +
// win_merge_k where neither takes the shape.
#include <algorithm>
#include <atomic>
#include <type_traits>
#include "kx_common.h"
#include "kx_lds_copy.h"
#include "kx_rows.h"
#include "kx_window.h"
#include "kx_window_choice.h"

namespace {

using kxr::Elem;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr float NEG_INF = -__builtin_inff();
constexpr int RB = 4;            // query heads whose values are summed together in win_partial_k
constexpr int PART_THREADS = 256;
// Rows of keys and of values that a thread of win_partial_k asks for first: all, of 64 keys of 128 columns.  One token is a chain of waits for
// memory on few workgroups; with the rows, the numbers under the norms and the query asked for together it has three left.  16 heads of 128
// on 4 key heads, 384 keys: 13.4 us before and 10.2 now, and win_merge_k, whose sums are asked for ahead of their weights, 4.8 and 3.7.
constexpr int AHEAD_K = 2, AHEAD_V = 4;

__host__ __device__ __forceinline__ int seen_blocks(int p, int size, int pool) {
  return pool > 0 && p - size + 1 > 0 ? (p - size + 1) / pool : 0;
}
__host__ __device__ __forceinline__ int window_lo(int p, int size) { return p - size + 1 > 0 ? p - size + 1 : 0; }

// mean of block b of one head into the pooled rows; the whole workgroup
template <class T>
__device__ __forceinline__ void pool_block(const KxWindowArgs &a, size_t head, int b, int tid, int n) {
  const KxWindowCache &c = a.c;
  const float inv = 1.0f / (float)a.s.pool;
  for (int x = tid; x < c.dp + c.vp; x += n) {
    const bool key = x < c.dp;
    const int col = key ? x : x - c.dp, w = key ? c.dp : c.vp;
    const T *src = (const T *)(key ? c.k : c.v) + head * c.cap * w + col;
    float sum = 0.0f;
    int slot = (int)((long)b * a.s.pool % c.cap);
    for (int j = 0; j < a.s.pool; ++j) {
      sum += Elem<T>::load(src + (size_t)slot * w);
      if (++slot == c.cap) slot = 0;
    }
    ((T *)(key ? c.pk : c.pv))[(head * c.blocks + b) * w + col] = Elem<T>::make(sum * inv);
  }
}

template <class T>
__global__ void __launch_bounds__(256) win_prep_k(KxWindowArgs a) {
  __shared__ float red[4];
  const KxWindowSpec &s = a.s;
  const KxWindowCache &c = a.c;
  const int tok = blockIdx.x, i = tok / a.batch, b = tok - i * a.batch, p = a.pos + i;
  const float *pr = a.proj + (size_t)tok * a.proj_ld;
  const int nq = s.heads * s.dim, nk = s.kv_heads * s.dim;
  float qs = 1.0f, ks = 1.0f;
  if (a.q_norm) {
    float v = 0.0f, w = 0.0f;
    for (int x = threadIdx.x; x < nq; x += 256) v = __builtin_fmaf(pr[a.q_off + x], pr[a.q_off + x], v);
    for (int x = threadIdx.x; x < nk; x += 256) w = __builtin_fmaf(pr[a.k_off + x], pr[a.k_off + x], w);
    qs = kx_rsqrtf(kxr::block_sum(v, red) / (float)nq + a.eps);
    ks = kx_rsqrtf(kxr::block_sum(w, red) / (float)nk + a.eps);
  }
  T *q = (T *)a.q + (size_t)tok * s.heads * c.dp;
  for (int x = threadIdx.x; x < s.heads * c.dp; x += 256) {
    const int h = x / c.dp, d = x - h * c.dp, y = h * s.dim + d;
    q[x] = Elem<T>::make(d < s.dim ? pr[a.q_off + y] * qs * (a.q_norm ? a.q_norm[y] : 1.0f) : 0.0f);
  }
  const int slot = p % c.cap;
  for (int x = threadIdx.x; x < s.kv_heads * c.dp; x += 256) {
    const int g = x / c.dp, d = x - g * c.dp, y = g * s.dim + d;
    ((T *)c.k)[((size_t)(b * s.kv_heads + g) * c.cap + slot) * c.dp + d] =
        Elem<T>::make(d < s.dim ? pr[a.k_off + y] * ks * (a.k_norm ? a.k_norm[y] : 1.0f) : 0.0f);
  }
  for (int x = threadIdx.x; x < s.kv_heads * c.vp; x += 256) {
    const int g = x / c.vp, d = x - g * c.vp;
    ((T *)c.v)[((size_t)(b * s.kv_heads + g) * c.cap + slot) * c.vp + d] = Elem<T>::make(d < s.vdim ? pr[a.v_off + g * s.vdim + d] : 0.0f);
  }
}

template <class T>
__global__ void __launch_bounds__(256) win_pool_k(KxWindowArgs a, int b0) {
  pool_block<T>(a, (size_t)blockIdx.z * a.s.kv_heads + blockIdx.y, b0 + blockIdx.x, threadIdx.x, 256);
}

// Part `blockIdx.x` of the keys of token tok0 + blockIdx.z for key/value head blockIdx.y: up to ch keys, blocks first.
// part: [tokens][parts][heads * vp] sums, then [tokens][parts][heads] maxima, then as many denominators.
// Four waves per SIMD: LDS has room for as many, and with the registers of three long contexts of many sequences are slower (16 sequences of 1000 keys, 16
// heads of 128, 32 bits: 56 us, 52 so).
template <class T, bool FUSED>
__global__ void __launch_bounds__(PART_THREADS, 4) win_partial_k(KxWindowArgs a, int tok0, int ch, float *po, float *pm, float *pz) {
  using E = Elem<T>;
  extern __shared__ __attribute__((aligned(16))) float win_lds[];
  __shared__ float red[2][4];
  const KxWindowSpec &s = a.s;
  const KxWindowCache &c = a.c;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tok = tok0 + blockIdx.z, i = tok / a.batch, b = tok - i * a.batch, p = a.pos + i;
  const int g = blockIdx.y, R = s.heads / s.kv_heads, parts = gridDim.x;
  const int nb = seen_blocks(p, s.size, s.pool), lo = window_lo(p, s.size), total = nb + p - lo + 1;
  const int e0 = blockIdx.x * ch, n = min(ch, total - e0);
  const size_t out0 = (size_t)blockIdx.z * parts + blockIdx.x;
  if (n <= 0) {  // fewer keys than the launch's largest token has
    for (int r = tid; r < R; r += PART_THREADS) {
      pm[out0 * s.heads + g * R + r] = NEG_INF;
      pz[out0 * s.heads + g * R + r] = 0.0f;
    }
    return;
  }
  float *qv = win_lds;                 // [R][dp]
  float *sc = qv + R * c.dp;           // [R][ch]
  float *sum = sc + R * ch;            // [groups][RB][vp]
  const size_t head = (size_t)b * s.kv_heads + g;
  const T *kc = (const T *)c.k + head * c.cap * c.dp, *vc = (const T *)c.v + head * c.cap * c.vp;
  const T *pkc = (const T *)c.pk + head * c.blocks * c.dp, *pvc = (const T *)c.pv + head * c.blocks * c.vp;
  const int base = p / c.cap * c.cap;  // position j of the window: slot j - base, one ring length more below it
  auto slot_of = [&](int e) {
    const int j = lo + e - nb - base;
    return j < 0 ? j + c.cap : j;
  };
  // scores: 8 lanes per key; values: vp / 8 threads per key.  The first rows of both are asked for before anything else.
  const int l8 = lane & 7, tpk = c.vp >> 3, groups = PART_THREADS / tpk, grp = tid / tpk, col = (tid - grp * tpk) * 8;
  struct Keys { typename E::Raw x[2]; };  // 128 columns
  auto key_row = [&](int k0) {
    const int e = e0 + min(k0 + (lane >> 3), n - 1);
    return e < nb ? pkc + (size_t)e * c.dp : kc + (size_t)slot_of(e) * c.dp;
  };
  auto ask_keys = [&](int k0) {
    const T *key = key_row(k0);
    Keys k;
    k.x[0] = E::cached(key + min(l8 * 8, c.dp - 8));
    if (sizeof(T) == 2 || c.dp > 64) k.x[1] = E::cached(key + min(l8 * 8 + 64, c.dp - 8));
    return k;
  };
  auto ask_values = [&](int k) {
    const int e = e0 + min(k, n - 1);
    return E::cached((e < nb ? pvc + (size_t)e * c.vp : vc + (size_t)slot_of(e) * c.vp) + col);
  };
  Keys kr[AHEAD_K];
  typename E::Raw vr[AHEAD_V];
  auto ask_all = [&] {  // in 32 bits, twice the bytes, no row twice: a short context has no second ones
#pragma unroll
    for (int y = 0; y < AHEAD_K; ++y)
      if (sizeof(T) == 2 || y == 0 || 32 * y < n) kr[y] = ask_keys(wave * 8 + 32 * y);
#pragma unroll
    for (int y = 0; y < AHEAD_V; ++y)
      if (sizeof(T) == 2 || y == 0 || groups * y < n) vr[y] = ask_values(grp + groups * y);
  };
  ask_all();
  if (FUSED) {
    const float *pr = a.proj + (size_t)tok * a.proj_ld;
    const int nq = s.heads * s.dim, nk = s.kv_heads * s.dim;
    float qs = 1.0f, ks = 1.0f;
    constexpr int UB = 8, UQ = 4;  // numbers of a thread asked for together
    float qx[UQ], qw[UQ];
#pragma unroll
    for (int k = 0; k < UQ; ++k) {
      const int x = min(tid + k * PART_THREADS, R * c.dp - 1), r = x / c.dp, y = (g * R + r) * s.dim + min(x - r * c.dp, s.dim - 1);
      qx[k] = pr[a.q_off + y];
      qw[k] = a.q_norm ? a.q_norm[y] : 1.0f;
    }
    if (a.q_norm) {
      float u[2][UB], v[2] = {};
      auto ask = [&](int j, int x0) {
#pragma unroll
        for (int k = 0; k < UB; ++k) u[j][k] = pr[(j ? a.k_off : a.q_off) + min(x0 + k * PART_THREADS, (j ? nk : nq) - 1)];
      };
      ask(0, tid);
      ask(1, tid);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        for (int x0 = tid; x0 < (j ? nk : nq); x0 += UB * PART_THREADS) {
          if (x0 > tid) ask(j, x0);
#pragma unroll
          for (int k = 0; k < UB; ++k)
            if (x0 + k * PART_THREADS < (j ? nk : nq)) v[j] = __builtin_fmaf(u[j][k], u[j][k], v[j]);
        }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v[j] = kxr::wave_sum(v[j]);
        if (lane == 0) red[j][wave] = v[j];
      }
      __syncthreads();
      qs = kx_rsqrtf((((red[0][0] + red[0][1]) + red[0][2]) + red[0][3]) / (float)nq + a.eps);
      ks = kx_rsqrtf((((red[1][0] + red[1][1]) + red[1][2]) + red[1][3]) / (float)nk + a.eps);
    }
    auto put = [&](int x, float q, float w) {
      float v = x - x / c.dp * c.dp < s.dim ? q * qs * w : 0.0f;
      if (sizeof(T) == 2) v = kx_bfround(v);  // the query the other kernels read
      qv[x] = v;
    };
#pragma unroll
    for (int k = 0; k < UQ; ++k)
      if (tid + k * PART_THREADS < R * c.dp) put(tid + k * PART_THREADS, qx[k], qw[k]);
    for (int x = tid + UQ * PART_THREADS; x < R * c.dp; x += PART_THREADS) {
      const int r = x / c.dp, y = (g * R + r) * s.dim + min(x - r * c.dp, s.dim - 1);
      put(x, pr[a.q_off + y], a.q_norm ? a.q_norm[y] : 1.0f);
    }
    if (e0 + n == total) {  // this workgroup holds the newest key: it writes the cache
      const int slot = p % c.cap;
      for (int d = tid; d < c.dp; d += PART_THREADS) {
        const int y = g * s.dim + d;
        ((T *)c.k)[(head * c.cap + slot) * c.dp + d] = E::make(d < s.dim ? pr[a.k_off + y] * ks * (a.k_norm ? a.k_norm[y] : 1.0f) : 0.0f);
      }
      for (int d = tid; d < c.vp; d += PART_THREADS)
        ((T *)c.v)[(head * c.cap + slot) * c.vp + d] = E::make(d < s.vdim ? pr[a.v_off + g * s.vdim + d] : 0.0f);
      __threadfence_block();
      __syncthreads();
      if (s.pool > 0 && (p + 1) % s.pool == 0 && p / s.pool < c.blocks) pool_block<T>(a, head, p / s.pool, tid, PART_THREADS);
      ask_all();  // the newest key's rows are there now
    }
  } else {
    const T *q = (const T *)a.q + ((size_t)tok * s.heads + g * R) * c.dp;
    for (int x = tid; x < R * c.dp; x += PART_THREADS) qv[x] = E::load(q + x);
  }
  __syncthreads();
  auto scores = [&](int k0, const Keys &first) {
    const T *key = key_row(k0);
    for (int r0 = 0; r0 < R; r0 += RB) {
      float d[RB] = {};
      auto times = [&](const typename E::Raw &raw, int x) {
        float kf[8];
        E::unpack(kf, raw);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const float *q = qv + min(r0 + r, R - 1) * c.dp + x;
          const float4 qa = *(const float4 *)q, qb = *(const float4 *)(q + 4);
          d[r] = __builtin_fmaf(kf[0], qa.x, d[r]); d[r] = __builtin_fmaf(kf[1], qa.y, d[r]);
          d[r] = __builtin_fmaf(kf[2], qa.z, d[r]); d[r] = __builtin_fmaf(kf[3], qa.w, d[r]);
          d[r] = __builtin_fmaf(kf[4], qb.x, d[r]); d[r] = __builtin_fmaf(kf[5], qb.y, d[r]);
          d[r] = __builtin_fmaf(kf[6], qb.z, d[r]); d[r] = __builtin_fmaf(kf[7], qb.w, d[r]);
        }
      };
#pragma unroll
      for (int y = 0; y < 2; ++y)
        if (l8 * 8 + 64 * y < c.dp) times(first.x[y], l8 * 8 + 64 * y);
      for (int x = l8 * 8 + 128; x < c.dp; x += 64) times(E::cached(key + x), x);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        d[r] += kxw::dpp_f<kxw::DPP_QUAD_XOR1>(d[r]);
        d[r] += kxw::dpp_f<kxw::DPP_QUAD_XOR2>(d[r]);
        d[r] += kxw::dpp_f<kxw::DPP_ROW_HALF_MIRROR>(d[r]);
        if (l8 == 0 && r0 + r < R && k0 + (lane >> 3) < n) sc[(r0 + r) * ch + k0 + (lane >> 3)] = d[r] * s.scale;
      }
    }
  };
#pragma unroll
  for (int y = 0; y < AHEAD_K; ++y)
    if (wave * 8 + 32 * y < n) scores(wave * 8 + 32 * y, kr[y]);
  for (int k0 = wave * 8 + 32 * AHEAD_K; k0 < n; k0 += 32) scores(k0, ask_keys(k0));
  __syncthreads();
  for (int r = wave; r < R; r += 4) {
    float m = NEG_INF, z = 0.0f;
    for (int k = lane; k < n; k += 64) m = fmaxf(m, sc[r * ch + k]);
    m = kxw::wave_max_f32(m);
    for (int k = lane; k < n; k += 64) {
      const float e = kx_expf(sc[r * ch + k] - m);
      sc[r * ch + k] = e;
      z += e;
    }
    z = kxr::wave_sum(z);
    if (lane == 0) {
      pm[out0 * s.heads + g * R + r] = m;
      pz[out0 * s.heads + g * R + r] = z;
    }
  }
  __syncthreads();
  for (int r0 = 0; r0 < R; r0 += RB) {
    float acc[RB][8] = {};
    auto times = [&](const typename E::Raw &raw, int k) {
      float vf[8];
      E::unpack(vf, raw);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const float w = sc[min(r0 + r, R - 1) * ch + k];
#pragma unroll
        for (int x = 0; x < 8; ++x) acc[r][x] = __builtin_fmaf(w, vf[x], acc[r][x]);
      }
    };
    if (grp < groups) {
#pragma unroll
      for (int y = 0; y < AHEAD_V; ++y)
        if (grp + groups * y < n) times(vr[y], grp + groups * y);
      for (int k = grp + groups * AHEAD_V; k < n; k += groups) times(ask_values(k), k);
    }
    if (grp < groups)
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int x = 0; x < 8; ++x) sum[(grp * RB + r) * c.vp + col + x] = acc[r][x];
    __syncthreads();
    for (int x = tid; x < RB * c.vp; x += PART_THREADS) {
      const int r = x / c.vp, d = x - r * c.vp;
      if (r0 + r >= R) continue;
      float v = sum[x];
      for (int y = 1; y < groups; ++y) v += sum[y * RB * c.vp + x];
      po[(out0 * s.heads + g * R + r0 + r) * c.vp + d] = v;
    }
    __syncthreads();
  }
}

// the parts of one head of one token merged, with the sink, times sigmoid(gate); one wave finds the parts' weights
constexpr int MERGE_THREADS = 128;
template <class T>
__global__ void __launch_bounds__(MERGE_THREADS) win_merge_k(KxWindowArgs a, int tok0, int parts, const float *po, const float *pm, const float *pz) {
  extern __shared__ float weight[];  // [parts]
  const KxWindowSpec &s = a.s;
  const int h = blockIdx.x, tok = tok0 + blockIdx.y, tid = threadIdx.x;
  const size_t row = (size_t)blockIdx.y * parts;
  constexpr int UB = 8;  // parts asked for together, the first before their weights are known
  auto ask = [&](float (&x)[UB], int d, int k0) {
#pragma unroll
    for (int k = 0; k < UB; ++k) x[k] = po[((row + min(k0 + k, parts - 1)) * s.heads + h) * a.c.vp + d];
  };
  auto gate_of = [&](int d) { return a.g_off >= 0 ? a.proj[(size_t)tok * a.proj_ld + a.g_off + h * s.vdim + d] : 0.0f; };
  const int d0 = min(tid, s.vdim - 1);
  float x[UB], gate = gate_of(d0);
  ask(x, d0, 0);
  if (tid < 64) {
    const float sink = a.sinks ? a.sinks[h] : 0.0f;
    const float m0 = tid < parts ? pm[(row + tid) * s.heads + h] : NEG_INF, z0 = tid < parts ? pz[(row + tid) * s.heads + h] : 0.0f;
    float m = fmaxf(s.sink ? sink : NEG_INF, m0), z = 0.0f;
    for (int k = tid + 64; k < parts; k += 64) m = fmaxf(m, pm[(row + k) * s.heads + h]);
    m = kxw::wave_max_f32(m);
    for (int k = tid; k < parts; k += 64) {
      const bool first = k == tid;
      const float w = kx_expf((first ? m0 : pm[(row + k) * s.heads + h]) - m);
      weight[k] = w;
      z = __builtin_fmaf(first ? z0 : pz[(row + k) * s.heads + h], w, z);
    }
    const float inv = 1.0f / (kxr::wave_sum(z) + (s.sink ? kx_expf(sink - m) : 0.0f));
    for (int k = tid; k < parts; k += 64) weight[k] *= inv;
  }
  __syncthreads();
  T *out = (T *)a.out + (size_t)tok * a.out_ld + h * s.vdim;
  for (int d = tid; d < s.vdim; d += MERGE_THREADS) {
    if (d > tid) gate = gate_of(d);
    float v = 0.0f;
    for (int k0 = 0; k0 < parts; k0 += UB) {
      if (d > tid || k0) ask(x, d, k0);
#pragma unroll
      for (int k = 0; k < UB; ++k)  // a part without keys has not written its sums
        if (k0 + k < parts && weight[k0 + k] > 0.0f) v = __builtin_fmaf(x[k], weight[k0 + k], v);
    }
    out[d] = Elem<T>::make(a.g_off >= 0 ? v * kx_sigmoidf(gate) : v);
  }
}

// ---- bf16, several positions: one head, 128 consecutive positions of one sequence, two groups of 4 waves of 32 queries ----
// S^T = K Q^T and O^T = V^T P^T, so that a lane holds one query (lane % 32) in both products: the running maximum and
// denominator are one value per lane, and the weights go from the first product's result into the second product's
// operand without leaving the registers.  The result layout gives lane (q, h) the keys 8 (v / 4) + 4 h + v % 4 of 32; the rows of V that
// a transposing read (ds_read_b64_tr_b16) gathers for it are those.  Scores are in units of log 2, so that a weight is one exp2.
// What bounds it: a wave reads 20 KB of keys and values of 192 and 128 columns for 20 products of 32 cycles, and as many cycles of
// vector arithmetic make the weights of its 32 x 32 scores, so every SIMD has two waves, whose products and weights overlap: group g
// has half g of every tile's keys, its own maximum, denominator and sums, and the groups' sums meet at the end.  Tiles are
// copied to LDS two ahead, the second group asking for its share of a tile behind its scores, so that the address path is free
// when the first one begins.  Workgroups with the most keys come first.
// 64 heads of 192 and 128, 2048 positions: 382 us with one wave per SIMD and tiles through registers, 184 now; 952 positions behind 2048:
// 265 and 194; 16 heads of 128, 2048 positions, window 1024: 64 and 49.  The whole operator, 16 heads on 4 key heads, 2048 positions, over keys of 32 to 256 and
// values of 32 to 256 columns takes 0.51 to 0.89 of what it did (256 and 256, whose tiles leave room for two stages and spill 40 bytes a lane, 245 and 125
// us; 64 and 128 91 and 67; 192 and 32 84 and 74), and 72 other steps 0.49 to 1.00.
// A key that a query does not see has a weight of zero, and its value is multiplied all the same; zero times a value that is not
// finite would make the query's output follow a position behind it, or one that its window has left.  So a workgroup whose sums
// are not all finite makes them once more: in tiles that not every query sees as a whole, such values are replaced by zeros, and
// added at the end by the queries that see them.
constexpr int FQ = 128, FK = 64, FLASH_WAVES = 8;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t LdsByte;

template <int ND, int NV>  // 32-column blocks of a key and of a value
struct Flash {
  static constexpr int KP = ND * 4, VP = NV * 4;  // pieces of 16 bytes of a row
  static constexpr int KB = FK * KP * 16, TILE = KB + FK * VP * 16, STAGES = 3 * TILE <= 128 * 1024 ? 3 : 2;
  static constexpr int COPIES = TILE / 1024, CPW = (COPIES + FLASH_WAVES - 1) / FLASH_WAVES;  // of a tile, of a wave
  static constexpr int KEEP = NV > 1 ? NV / 2 : 1;  // blocks of the result that a group finishes; of one block group 0
  static constexpr int MERGE = FLASH_WAVES * KEEP * 4096, ENDS = MERGE + FLASH_WAVES * 64 * 8;
  static constexpr int ODD = STAGES * TILE > ENDS ? STAGES * TILE : ENDS, LDS = ODD + 16;
  // Where piece p of row r lies in the row: eight consecutive rows read the same piece of a key, four rows the same 64 bytes of
  // a value, each without meeting in a bank.
  static __device__ __forceinline__ int key_piece(int r, int p) { return p ^ (ND == 1 ? r >> 1 & 3 : r & 7); }
  static __device__ __forceinline__ int value_piece(int r, int p) { return p ^ (NV == 1 ? 0 : NV == 2 ? (r >> 1 & 1) * 4 : (r & 3) * 4); }
};

template <int ND, int NV>
__global__ void __launch_bounds__(FLASH_WAVES * 64, 2) win_flash_k(KxWindowArgs a) {
  using F = Flash<ND, NV>;
  extern __shared__ __attribute__((aligned(16))) uint8_t fl_lds[];
  LdsByte *const lds = (LdsByte *)fl_lds;
  int &odd_s = *(int *)(fl_lds + F::ODD);  // a sum that is not finite
  const KxWindowSpec &s = a.s;
  const KxWindowCache &c = a.c;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), me = wave & 3, half = wave >> 2, lq = lane & 31, hh = lane >> 5;
  const int h = blockIdx.x % s.heads, b = blockIdx.x / s.heads, g = h / (s.heads / s.kv_heads);
  const int i0 = (gridDim.y - 1 - blockIdx.y) * FQ, i = i0 + me * 32 + lq;  // this lane's position of the step
  const bool live = i < a.positions;
  const int p = a.pos + min(i, a.positions - 1), tok = min(i, a.positions - 1) * (a.tok_batch ? a.tok_batch : a.batch) + b;
  const int p_first = a.pos + i0, p_last = a.pos + min(i0 + FQ, a.positions) - 1;
  const int nb = seen_blocks(p, s.size, s.pool), lo = window_lo(p, s.size);
  const size_t head = (size_t)b * s.kv_heads + g;
  const uint16_t *kc = (const uint16_t *)c.k + head * c.cap * c.dp, *vc = (const uint16_t *)c.v + head * c.cap * c.vp;
  const uint16_t *pkc = (const uint16_t *)c.pk + head * c.blocks * c.dp, *pvc = (const uint16_t *)c.pv + head * c.blocks * c.vp;
  bf16x8 q[ND * 2];
  {
    const uint16_t *qr = (const uint16_t *)a.q + (size_t)tok * (a.q_ld ? a.q_ld : (size_t)s.heads * c.dp) + (size_t)h * c.dp;
#pragma unroll
    for (int kk = 0; kk < ND * 2; ++kk) q[kk] = kk * 16 < c.dp ? *(const bf16x8 *)(qr + kk * 16 + hh * 8) : bf16x8{};
  }
  f32x16 o[NV];
  float m, z;  // z: of this lane's half of the group's keys
  const float scale2 = s.scale * 1.44269504088896341f;

  // tiles: the blocks the last query sees, then the positions from the first query's window on
  const int tb = (seen_blocks(p_last, s.size, s.pool) + FK - 1) / FK;
  const int j0 = window_lo(p_first, s.size) & ~(FK - 1), tiles = tb + (p_last - j0) / FK + 1;
  // what all and what any of this wave's queries see
  const int q0 = __builtin_amdgcn_readfirstlane(a.pos + min(i0 + me * 32, a.positions - 1));
  const int q1 = __builtin_amdgcn_readfirstlane(a.pos + min(i0 + me * 32 + 31, a.positions - 1));
  const int nb0 = seen_blocks(q0, s.size, s.pool), nb1 = seen_blocks(q1, s.size, s.pool), lo0 = window_lo(q0, s.size), lo1 = window_lo(q1, s.size);
  auto first_key = [&](int t) { return t < tb ? t * FK : j0 + (t - tb) * FK; };
  auto seen_by_all = [&](int t) {
    return t < tb ? (t + 1) * FK <= seen_blocks(p_first, s.size, s.pool) : first_key(t) >= window_lo(p_last, s.size) && first_key(t) + FK - 1 <= p_first;
  };
  // This wave's copies of a tile, 1024 bytes of LDS each.  Where there are fewer the last one is made again, so that every wave waits
  // for the same number.  A row has no more than c.dp and c.vp columns: a piece past them is the last one, which meets zeros of the query or a
  // result that is not stored.
  int crow[F::CPW], ccol[F::CPW];
#pragma unroll
  for (int y = 0; y < F::CPW; ++y) {
    const int k = min(wave + FLASH_WAVES * y, F::COPIES - 1);
    const bool key = k < F::KB / 1024;
    const int x = (key ? k : k - F::KB / 1024) * 64 + lane, per = key ? F::KP : F::VP, r = x / per;
    crow[y] = r;
    ccol[y] = min((key ? F::key_piece(r, x % per) : F::value_piece(r, x % per)) * 8, (key ? c.dp : c.vp) - 8);
  }
  // Rows of a tile: a window tile starts at a multiple of FK and the ring's length is one, so it does not wrap inside; past the
  // last block there is nothing to read.  What is read beyond the keys a query sees meets zeros.
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  auto ask = [&](int t, int stage) {
    const bool pooled = t < tb;
    const int k0 = first_key(t), last = pooled ? c.blocks - 1 - k0 : FK - 1;
    const uint16_t *kr = pooled ? pkc + (size_t)k0 * c.dp : kc + (size_t)(k0 % c.cap) * c.dp;
    const uint16_t *vr = pooled ? pvc + (size_t)k0 * c.vp : vc + (size_t)(k0 % c.cap) * c.vp;
#pragma unroll
    for (int y = 0; y < F::CPW; ++y) {
      const int k = min(wave + FLASH_WAVES * y, F::COPIES - 1);
      const bool key = k < F::KB / 1024;
      kx_copy16_to_lds((key ? kr : vr) + (uint32_t)(min(crow[y], last) * (key ? c.dp : c.vp) + ccol[y]), __builtin_amdgcn_readfirstlane(lds0 + stage * F::TILE + k * 1024));
    }
  };
  // this lane's operands: pieces of key `half * 32 + lq`, and rows half * 32 + 4 hh + (lane % 16) / 4 of 16 columns of the values
  int kp[4], vp[NV];
#pragma unroll
  for (int y = 0; y < 4; ++y) kp[y] = (half * 32 + lq) * (F::KP * 16) + F::key_piece(lq, (2 * y + hh) & (F::KP - 1 < 7 ? 3 : 7)) * 16;
  const int vrow = 4 * hh + (lane >> 2 & 3);
#pragma unroll
  for (int j = 0; j < NV; ++j)
    vp[j] = F::KB + (half * 32 + vrow) * (F::VP * 16) + F::value_piece(vrow, j * 4) * 16 + (lane >> 4 & 1) * 32 + (lane & 3) * 8;
  auto attend = [&](auto replace) {
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[j][v] = 0.0f;
    const bool sink = s.sink && half == 0;
    m = sink ? (a.sinks ? a.sinks[h] * 1.44269504088896341f : 0.0f) : NEG_INF;
    z = sink && hh == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int t = 0; t < F::STAGES - 1; ++t)
      if (t < tiles) ask(t, t);
    int stage = 0;
    for (int t = 0; t < tiles; ++t) {
      const bool pooled = t < tb;
      const int k0 = first_key(t);
      if (F::STAGES > 2 && t + 1 < tiles) kx_wait_copies<F::CPW>();
      else kx_wait_copies<0>();
      kx_lds_barrier();  // the tile is in LDS for every wave, and the tile before has been multiplied
      const LdsByte *const at = lds + stage * F::TILE;
      const int next = stage == 0 ? F::STAGES - 1 : stage - 1;  // of the tile before
      stage = stage == F::STAGES - 1 ? 0 : stage + 1;
      if constexpr (decltype(replace)::value) {
        if (t + F::STAGES - 1 < tiles) ask(t + F::STAGES - 1, next);
        if (!seen_by_all(t)) {
          typedef __attribute__((address_space(3))) u32x4 LdsPiece;
          for (int x = tid; x < FK * F::VP; x += FLASH_WAVES * 64) {
            LdsPiece *w = (LdsPiece *)(at + F::KB) + x;
            u32x4 y = *w;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] &= ~(((((y[e] & 0x7f807f80u) + 0x00800080u) & 0x80008000u) >> 15) * 0xffffu);  // an exponent of all ones carries into the sign's place
            *w = y;
          }
          kx_lds_barrier();
        }
      } else {
        if (half == 0 && t + F::STAGES - 1 < tiles) ask(t + F::STAGES - 1, next);
      }
      const int kh = k0 + half * 32;  // this group's first key
      const bool none = pooled ? kh >= nb1 : kh > q1 || kh + 31 < lo0;
      const bool all = pooled ? kh + 32 <= nb0 : kh >= lo1 && kh + 31 <= q0;
      f32x16 sc;
      if (!none) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < ND * 2; ++kk) {
          const bf16x8 kf = *(const __attribute__((address_space(3))) bf16x8 *)(at + kp[kk & 3] + (kk >> 2) * 128);
          sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, q[kk], sc, 0, 0, 0);
        }
      }
      if constexpr (!decltype(replace)::value) {
        __builtin_amdgcn_sched_barrier(0);
        if (half == 1 && t + F::STAGES - 1 < tiles) ask(t + F::STAGES - 1, next);
      }
      if (none) continue;
      const int from = (pooled ? 0 : lo) - kh - 4 * hh, to = (pooled ? nb - 1 : p) - kh - 4 * hh;  // the keys this lane's query sees, from its first one on
#pragma unroll
      for (int v = 0; v < 16; ++v) sc[v] *= scale2;
      if (!all) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int e = 8 * (v >> 2) + (v & 3);
          sc[v] = ((e < from) | (e > to)) ? NEG_INF : sc[v];
        }
      }
      float tm = NEG_INF;
#pragma unroll
      for (int v = 0; v < 16; ++v) tm = fmaxf(tm, sc[v]);
      {
        const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, tm), __builtin_bit_cast(uint32_t, tm), false, false);
        tm = fmaxf(__builtin_bit_cast(float, (uint32_t)both[0]), __builtin_bit_cast(float, (uint32_t)both[1]));
      }
      if (__any(tm > m)) {
        const float m1 = fmaxf(m, tm), al = m == NEG_INF ? 0.0f : __builtin_amdgcn_exp2f(m - m1);
        m = m1;
        z *= al;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[j][v] *= al;
      }
      const float mm = m == NEG_INF ? 0.0f : m;  // nothing seen so far
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        sc[v] = __builtin_amdgcn_exp2f(sc[v] - mm);
        z += sc[v];
      }
#pragma unroll
      for (int ss = 0; ss < 2; ++ss) {
        uint32_t pw[4];
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          const f32x2 two = {sc[ss * 8 + 2 * y], sc[ss * 8 + 2 * y + 1]};
          pw[y] = __builtin_bit_cast(uint32_t, __builtin_convertvector(two, bf16x2));
        }
        const bf16x8 pf = __builtin_bit_cast(bf16x8, make_uint4(pw[0], pw[1], pw[2], pw[3]));
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          s16x4 v4[2];
#pragma unroll
          for (int u = 0; u < 2; ++u)
            v4[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(at + vp[j] + (ss * 16 + u * 8) * (F::VP * 16)));
          const bf16x8 vf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v4[0], v4[1], 0, 1, 2, 3, 4, 5, 6, 7));
          o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[j], 0, 0, 0);
        }
      }
    }
  };
  if (tid == 0) odd_s = 0;
  attend(std::false_type{});
  float odd[4] = {};  // zero, unless a sum is not finite
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) odd[v & 3] = __builtin_fmaf(o[j][v], 0.0f, odd[v & 3]);
  if ((odd[0] + odd[1]) + (odd[2] + odd[3]) != 0.0f) odd_s = 1;
  __syncthreads();
  if (__builtin_expect(odd_s, 0)) {
    attend(std::true_type{});
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll 1
      for (int t = 0; t < tiles; ++t) {
        if (seen_by_all(t)) continue;
        const bool pooled = t < tb;
        const int k0 = first_key(t), e1 = min(half * 32 + 31, (pooled ? nb - 1 : p) - k0);
        const uint16_t *vr = pooled ? pvc + (size_t)k0 * c.vp : vc + (size_t)(k0 % c.cap) * c.vp;
#pragma unroll 1
        for (int e = max(half * 32, (pooled ? 0 : lo) - k0); e <= e1; ++e)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const float x = kx_bf16_f32(vr[(size_t)e * c.vp + min(j * 32 + 8 * (v >> 2) + 4 * hh + (v & 3), c.vp - 1)]);
            o[j][v] = __builtin_isfinite(x) ? o[j][v] : o[j][v] + x;
          }
      }
    __syncthreads();  // the tiles are not read any more
  }
  // the groups' sums meet: each gives what the other finishes
  z += __shfl_xor(z, 32);
  const int other = (half ^ 1) * 4 + me;
  f32x4 *const sums = (f32x4 *)fl_lds;
  float *const ends = (float *)(fl_lds + F::MERGE);
#pragma unroll
  for (int j = 0; j < F::KEEP; ++j)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const f32x16 x = NV == 1 ? o[0] : half ? o[j] : o[NV - F::KEEP + j];
      sums[((wave * F::KEEP + j) * 4 + y) * 64 + lane] = f32x4{x[4 * y], x[4 * y + 1], x[4 * y + 2], x[4 * y + 3]};
    }
  ends[(wave * 64 + lane) * 2] = m;
  ends[(wave * 64 + lane) * 2 + 1] = z;
  __syncthreads();
  if (!live || (NV == 1 && half)) return;
  const float m2 = ends[(other * 64 + lane) * 2], top = fmaxf(m, m2);
  const float w1 = m == NEG_INF ? 0.0f : __builtin_amdgcn_exp2f(m - top), w2 = m2 == NEG_INF ? 0.0f : __builtin_amdgcn_exp2f(m2 - top);
  const float inv = 1.0f / __builtin_fmaf(ends[(other * 64 + lane) * 2 + 1], w2, z * w1);
  uint16_t *out = (uint16_t *)a.out + (size_t)tok * a.out_ld + h * s.vdim;
  const float *gate = a.g_off >= 0 ? a.proj + (size_t)tok * a.proj_ld + a.g_off + h * s.vdim : nullptr;
  const bool wide = ((s.vdim | a.out_ld) & 3) == 0 && ((uintptr_t)a.out & 7) == 0 &&
                    (!gate || (((a.proj_ld | a.g_off) & 3) == 0 && ((uintptr_t)a.proj & 15) == 0));  // four columns at a time
  f32x4 gt[F::KEEP][4];
#pragma unroll
  for (int j = 0; j < F::KEEP; ++j)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int d = (half * F::KEEP + j) * 32 + 8 * y + 4 * hh;
      if (!gate) continue;
      if (wide) gt[j][y] = *(const f32x4 *)(gate + min(d, s.vdim - 4));
      else
#pragma unroll
        for (int v = 0; v < 4; ++v) gt[j][y][v] = gate[min(d + v, s.vdim - 1)];
    }
#pragma unroll
  for (int j = 0; j < F::KEEP; ++j)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int d = (half * F::KEEP + j) * 32 + 8 * y + 4 * hh;
      const f32x16 x = NV > 1 && half ? o[NV - F::KEEP + j] : o[j];
      const f32x4 x2 = sums[((other * F::KEEP + j) * 4 + y) * 64 + lane];
      uint16_t r[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = kx_bf16_rne(__builtin_fmaf(x2[v], w2, x[4 * y + v] * w1) * inv * (gate ? kxr::sigmoid_for<uint16_t>(gt[j][y][v]) : 1.0f));
      if (wide && d < s.vdim) {
        *(u32x2 *)(out + d) = u32x2{r[0] | (uint32_t)r[1] << 16, r[2] | (uint32_t)r[3] << 16};
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (d + v < s.vdim) out[d + v] = r[v];
      }
    }
}

// ---- f32, several positions: one head, 32 consecutive positions of one sequence ----
// As above with 32-bit products (v_mfma_f32_32x32x2_f32) and without LDS: wave w of four has every fourth tile of 32 keys to itself, from
// memory into the operands' registers.  Lane (r, h) holds columns 8 k + 4 h .. +3 of key r and of query r, so that the first product
// meets two of them at a time, in four chains; its result in register v is the weight of key 8 (v / 4) + 4 h + v % 4, which the second
// product takes as it is, with NV columns of that key's value from NV r on.  The keys of the next tile are asked for when the scores are
// made, its values behind the second product.  Bound by the products, 8192 cycles of a SIMD for 32 keys of 128 and 128 columns.
// The waves' sums meet at the end.  In tiles that not every query sees as a whole a value that is not finite is replaced by
// zero in the product, and added by the queries that see it.
// 777 positions, 8 heads of 128: 52 us, 141 in parts of 256 keys on the vector ALU.  The error is no larger: chains are short, and a
// tile's sums are added to those before it (1.02e-7 to 2.05e-7 for 33 to 2048 positions, 0.96 to 1.00 of the parts').
using kxwin::GQ;
template <int N> struct Floats { typedef float Type __attribute__((ext_vector_type(N))); };

template <int ND, int NV>
__global__ void __launch_bounds__(256, 1) win_flash_f32_k(KxWindowArgs a) {
  typedef typename Floats<NV>::Type Value;
  constexpr int KP = ND * 4, ENDS = 4 * 4 * NV * 1024, QUERIES = ENDS + 4 * 64 * 8;
  extern __shared__ __attribute__((aligned(16))) uint8_t fl_lds[];
  const KxWindowSpec &s = a.s;
  const KxWindowCache &c = a.c;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lq = lane & 31, hh = lane >> 5;
  const int h = blockIdx.x % s.heads, b = blockIdx.x / s.heads, g = h / (s.heads / s.kv_heads);
  const int i0 = (gridDim.y - 1 - blockIdx.y) * GQ, i = i0 + lq;
  const int p = a.pos + min(i, a.positions - 1), tok = min(i, a.positions - 1) * a.batch + b;
  const int p_first = a.pos + i0, p_last = a.pos + min(i0 + GQ, a.positions) - 1;
  const int nb = seen_blocks(p, s.size, s.pool), lo = window_lo(p, s.size);
  const size_t head = (size_t)b * s.kv_heads + g;
  const float *kc = (const float *)c.k + head * c.cap * c.dp, *vc = (const float *)c.v + head * c.cap * c.vp;
  const float *pkc = (const float *)c.pk + head * c.blocks * c.dp, *pvc = (const float *)c.pv + head * c.blocks * c.vp;
  f32x4 k[KP];
  f32x4 *const q = (f32x4 *)(fl_lds + QUERIES) + lane;  // [piece][lane], the same for all waves
  {
    const float *qr = (const float *)a.q + ((size_t)tok * s.heads + h) * c.dp;
    for (int x = wave; x < KP; x += 4) q[x * 64] = x * 8 < c.dp ? *(const f32x4 *)(qr + x * 8 + hh * 4) : f32x4{};
  }
  __syncthreads();
  // tiles: the blocks the last query sees, then the positions from the first query's window on; the ring's length is a multiple of 32
  const int tb = (seen_blocks(p_last, s.size, s.pool) + 31) / 32;
  const int j0 = window_lo(p_first, s.size) & ~31, tiles = tb + (p_last - j0) / 32 + 1;
  auto first_key = [&](int t) { return t < tb ? t * 32 : j0 + (t - tb) * 32; };
  // past the last block there is nothing to read, and past a row's columns its last ones are read again, which meet zeros of the query or a
  // result that is not stored
  auto ask_keys = [&](int t) {
    const int k0 = first_key(t), last = t < tb ? c.blocks - 1 - k0 : 31;
    const float *kr = t < tb ? pkc + (size_t)k0 * c.dp : kc + (size_t)(k0 % c.cap) * c.dp;
    const uint32_t at = min(lq, last) * c.dp + hh * 4;
#pragma unroll
    for (int x = 0; x < KP; ++x) k[x] = *(const f32x4 *)(kr + min(x * 8, c.dp - 8) + at);
  };
  Value val[16];
  auto ask_values = [&](int t) {
    const int k0 = first_key(t), last = t < tb ? c.blocks - 1 - k0 : 31, d = min(lq * NV, c.vp - NV);
    const float *vr = t < tb ? pvc + (size_t)k0 * c.vp : vc + (size_t)(k0 % c.cap) * c.vp;
    if (last >= 31) {
      const uint32_t at = 4 * hh * c.vp + d;
#pragma unroll
      for (int v = 0; v < 16; ++v) val[v] = *(const Value *)(vr + (8 * (v >> 2) + (v & 3)) * c.vp + at);
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) val[v] = *(const Value *)(vr + (uint32_t)(min(8 * (v >> 2) + 4 * hh + (v & 3), last) * c.vp + d));
    }
  };
  f32x16 o[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[j][v] = 0.0f;
  const bool sink = s.sink && wave == 0;
  float m = sink ? (a.sinks ? a.sinks[h] : 0.0f) : NEG_INF, z = sink && hh == 0 ? 1.0f : 0.0f;  // z: of this lane's half of the keys
  if (wave < tiles) {
    ask_keys(wave);
    ask_values(wave);
  }
  for (int t = wave; t < tiles; t += 4) {
    asm volatile("" ::: "memory");  // the query's pieces are read again for each tile: there are no registers to keep them in
    const bool pooled = t < tb, more = t + 4 < tiles;
    const int k0 = first_key(t);
    f32x16 part[2][4], sc;  // short chains: four products each, of which four are added, and those in their order
    auto gather = [&](const f32x16 (&four)[4]) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sc[v] += (four[0][v] + four[1][v]) + (four[2][v] + four[3][v]);
      asm volatile("" : "+v"(sc));  // here: the sums of all pieces at once have no registers
    };
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
#pragma unroll
    for (int x = 0; x < KP; x += 4) {
      f32x16(&four)[4] = part[x >> 2 & 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) four[e] = f32x16{};
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const f32x4 qx = q[(x + y) * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) four[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[x + y][e], qx[e], four[e], 0, 0, 0);
      }
      if (x > 0) gather(part[(x >> 2 & 1) ^ 1]);  // under the products of this one
      __builtin_amdgcn_sched_barrier(0);
    }
    gather(part[(KP / 4 - 1) & 1]);
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] *= s.scale;
    if (more) ask_keys(t + 4);
    const int from = (pooled ? 0 : lo) - k0, to = (pooled ? nb - 1 : p) - k0;  // the keys of the tile that this lane's query sees
    const bool all = pooled ? k0 + 32 <= seen_blocks(p_first, s.size, s.pool) : k0 >= window_lo(p_last, s.size) && k0 + 31 <= p_first;
    bool odd = false;
    if (!all) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int e = 8 * (v >> 2) + 4 * hh + (v & 3);
        sc[v] = ((e < from) | (e > to)) ? NEG_INF : sc[v];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const bool fine = __builtin_isfinite(val[v][j]);
          odd |= !fine;
          val[v][j] = fine ? val[v][j] : 0.0f;
        }
      }
    }
    float top[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) top[y] = fmaxf(fmaxf(sc[y], sc[4 + y]), fmaxf(sc[8 + y], sc[12 + y]));
    float tm = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
    tm = fmaxf(tm, __shfl_xor(tm, 32));
    if (__any(tm > m)) {
      const float m1 = fmaxf(m, tm), al = m == NEG_INF ? 0.0f : kx_expf(m - m1);
      m = m1;
      z *= al;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[j][v] *= al;
    }
    const float mm = m == NEG_INF ? 0.0f : m;  // nothing seen so far
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = kx_expf(sc[v] - mm);
#pragma unroll
    for (int y = 0; y < 4; ++y) top[y] = (sc[y] + sc[4 + y]) + (sc[8 + y] + sc[12 + y]);
    z += (top[0] + top[1]) + (top[2] + top[3]);
    constexpr int JW = NV > 1 ? 2 : 1;
    f32x16 own[2][JW];  // the tile's, two blocks of columns at a time
    auto keep = [&](int j) {
#pragma unroll
      for (int y = 0; y < JW; ++y)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[j + y][v] += own[j / JW & 1][y][v];
#pragma unroll
      for (int y = 0; y < JW; ++y) asm volatile("" : "+v"(o[j + y]));
    };
#pragma unroll
    for (int j = 0; j < NV; j += JW) {
      f32x16(&now)[JW] = own[j / JW & 1];
#pragma unroll
      for (int y = 0; y < JW; ++y) now[y] = f32x16{};
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int y = 0; y < JW; ++y) now[y] = __builtin_amdgcn_mfma_f32_32x32x2f32(val[v][j + y], sc[v], now[y], 0, 0, 0);
      if (j > 0) keep(j - JW);
      __builtin_amdgcn_sched_barrier(0);
    }
    keep(NV - JW);
    if (__builtin_expect(__any(odd), 0)) {
      const float *vr = pooled ? pvc + (size_t)k0 * c.vp : vc + (size_t)(k0 % c.cap) * c.vp;
#pragma unroll 1
      for (int e = max(0, from); e <= min(31, to); ++e) {
        int d0 = 4 * hh;
        asm volatile("" : "+v"(d0));  // the places are worked out here, not kept for the whole kernel
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const Value x = *(const Value *)(vr + (uint32_t)(e * c.vp + min((8 * (v >> 2) + d0 + (v & 3)) * NV, c.vp - NV)));
#pragma unroll
          for (int j = 0; j < NV; ++j) o[j][v] = __builtin_isfinite(x[j]) ? o[j][v] : o[j][v] + x[j];
        }
      }
    }
    if (more) ask_values(t + 4);
  }
  // the waves' sums meet: [wave][v / 4][column][lane]
  z += __shfl_xor(z, 32);
  f32x4 *const sums = (f32x4 *)fl_lds;
  float *const ends = (float *)(fl_lds + ENDS);
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int y = 0; y < 4; ++y) sums[((wave * 4 + y) * NV + j) * 64 + lane] = f32x4{o[j][4 * y], o[j][4 * y + 1], o[j][4 * y + 2], o[j][4 * y + 3]};
  ends[(wave * 64 + lane) * 2] = m;
  ends[(wave * 64 + lane) * 2 + 1] = z;
  __syncthreads();
  if (i >= a.positions) return;
  float mw[4], weight[4], most = NEG_INF, total = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) most = fmaxf(most, mw[w] = ends[(w * 64 + lane) * 2]);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    weight[w] = mw[w] == NEG_INF ? 0.0f : kx_expf(mw[w] - most);
    total = __builtin_fmaf(ends[(w * 64 + lane) * 2 + 1], weight[w], total);
  }
  const float inv = 1.0f / total;
  const int d0 = (8 * wave + 4 * hh) * NV;  // this lane's 4 NV columns
  float y[4 * NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    f32x4 sum = {};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const f32x4 x = sums[((w * 4 + wave) * NV + j) * 64 + lane];
#pragma unroll
      for (int v = 0; v < 4; ++v) sum[v] = weight[w] > 0.0f ? __builtin_fmaf(x[v], weight[w], sum[v]) : sum[v];  // a wave without keys has none
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) y[v * NV + j] = sum[v] * inv;
  }
  float *out = (float *)a.out + (size_t)tok * a.out_ld + h * s.vdim;
  const float *gate = a.g_off >= 0 ? a.proj + (size_t)tok * a.proj_ld + a.g_off + h * s.vdim : nullptr;
#pragma unroll
  for (int x = 0; x < 4 * NV; ++x)
    if (d0 + x < s.vdim) out[d0 + x] = y[x] * (gate ? kx_sigmoidf(gate[d0 + x]) : 1.0f);
}

// keys per workgroup of win_partial_k: few parts, but enough workgroups
int part_keys(const KxWindowSpec &s, int total, int tokens) {
  const int R = s.heads / s.kv_heads;
  int ch = R <= 16 ? 256 : R <= 32 ? 128 : 64;  // R * ch scores in LDS
  while (ch > 64 && (long)kx_cdiv(total, ch) * s.kv_heads * tokens < 256) ch >>= 1;
  return ch;
}
// most keys a token of a sequence of `context` positions sees
int most_keys(const KxWindowSpec &s, int context) { return std::min(s.size, context) + seen_blocks(context - 1, s.size, s.pool); }
size_t floats_per_part(const KxWindowSpec &s) { return (size_t)s.heads * (kx_pad(s.vdim, 32) + 2); }

template <int ND>
int flash_nv(const KxWindowArgs &a, int nv, hipStream_t st) {
  const dim3 grid(a.s.heads * a.batch, kx_cdiv(a.positions, FQ));
#define KX_FLASH(NV)                                                                                                          \
  {                                                                                                                           \
    constexpr int lds = Flash<ND, NV>::LDS;                                                                                   \
    static std::atomic<bool> attr{false};                                                                                     \
    if (!attr) {                                                                                                              \
      KX_HIP(hipFuncSetAttribute((const void *)win_flash_k<ND, NV>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));        \
      attr = true;                                                                                                            \
    }                                                                                                                         \
    hipLaunchKernelGGL((win_flash_k<ND, NV>), grid, dim3(FLASH_WAVES * 64), lds, st, a);                                      \
  }
  if (nv == 1) KX_FLASH(1) else if (nv == 2) KX_FLASH(2) else if (nv <= 4) KX_FLASH(4) else KX_FLASH(8)
#undef KX_FLASH
  KX_LAUNCH_CHECK();
  return KX_OK;
}

template <int ND>
int flash_f32_nv(const KxWindowArgs &a, int nv, hipStream_t st) {
  const dim3 grid(a.s.heads * a.batch, kx_cdiv(a.positions, GQ));
#define KX_FLASH(NV)                                                                                                          \
  {                                                                                                                           \
    constexpr int lds = 4 * 4 * NV * 1024 + 4 * 64 * 8 + ND * 4 * 1024;                                                       \
    static std::atomic<bool> attr{false};                                                                                     \
    if (!attr) {                                                                                                              \
      KX_HIP(hipFuncSetAttribute((const void *)win_flash_f32_k<ND, NV>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));    \
      attr = true;                                                                                                            \
    }                                                                                                                         \
    hipLaunchKernelGGL((win_flash_f32_k<ND, NV>), grid, dim3(256), lds, st, a);                                               \
  }
  if (nv == 1) KX_FLASH(1) else if (nv == 2) KX_FLASH(2) else KX_FLASH(4)
#undef KX_FLASH
  KX_LAUNCH_CHECK();
  return KX_OK;
}
// Parts of a step's keys: keys of each, how many, and the tokens of a launch.
struct Parts {
  int keys, n;
  size_t per_token, at_once;  // floats; tokens, 0 where the scratch does not hold one's
};
Parts parts_of(const KxWindowArgs &a) {
  const int tokens = a.batch * a.positions, total = most_keys(a.s, a.pos + a.positions), ch = part_keys(a.s, total, tokens), n = kx_cdiv(total, ch);
  const size_t per_token = n * floats_per_part(a.s);
  return {ch, n, per_token, std::min<size_t>({(size_t)tokens, a.part_floats / per_token, (size_t)65535})};
}
bool flash_f32(const KxWindowArgs &a) {
  const KxWindowSpec &s = a.s;
  if (a.c.dp > 256 || a.c.vp > 128 || a.tok_batch || a.q_ld) return false;
  const Parts p = parts_of(a);
  const int most = most_keys(s, a.pos + a.positions);
  return kxwin::matrix_cores_f32({s.heads, s.kv_heads, a.c.dp + a.c.vp, a.batch, a.positions}, most, 0.5 * (most + most_keys(s, a.pos + 1)), {p.keys, p.n, (long)p.at_once},
                                 std::max(1, kx_device_cus()));
}

int check(const KxWindowArgs &a) {
  const KxWindowSpec &s = a.s;
  KX_REQUIRE(s.heads > 0 && s.kv_heads > 0 && s.heads % s.kv_heads == 0 && s.dim > 0 && s.vdim > 0 && s.size > 0 && s.pool >= 0,
             "window attention: heads=%d kv_heads=%d dim=%d vdim=%d size=%d pool=%d", s.heads, s.kv_heads, s.dim, s.vdim, s.size, s.pool);
  KX_REQUIRE(a.c.vp <= 2048, "window attention: values of %d columns", s.vdim);
  KX_REQUIRE(a.batch > 0 && a.positions > 0 && a.pos >= 0, "window attention: %d x %d tokens at position %d", a.batch, a.positions, a.pos);
  return KX_OK;
}

// parts and merge
template <class T>
int attend_parts(const KxWindowArgs &a, bool fused, hipStream_t st) {
  const KxWindowSpec &s = a.s;
  const Parts p = parts_of(a);
  const int tokens = a.batch * a.positions, R = s.heads / s.kv_heads, ch = p.keys, parts = p.n, at_once = (int)p.at_once;
  KX_REQUIRE(at_once > 0, "window attention: %zu floats of partials, room for %zu", p.per_token, a.part_floats);
  const size_t lds = ((size_t)R * a.c.dp + (size_t)R * ch + (size_t)(PART_THREADS / (a.c.vp / 8)) * RB * a.c.vp) * 4;
  KX_REQUIRE(lds <= 160 * 1024 - 256, "window attention: %d query heads of %d per key head do not fit a workgroup", R, s.dim);
  static std::atomic<bool> attr{false};
  if (!attr) {
    KX_HIP(hipFuncSetAttribute((const void *)win_partial_k<T, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256));
    KX_HIP(hipFuncSetAttribute((const void *)win_partial_k<T, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256));
    attr = true;
  }
  for (int t0 = 0; t0 < tokens; t0 += at_once) {
    const int n = std::min(at_once, tokens - t0);
    float *po = a.part, *pm = po + (size_t)n * parts * s.heads * a.c.vp, *pz = pm + (size_t)n * parts * s.heads;
    const dim3 grid(parts, s.kv_heads, n);
    if (fused) hipLaunchKernelGGL((win_partial_k<T, true>), grid, dim3(PART_THREADS), lds, st, a, t0, ch, po, pm, pz);
    else hipLaunchKernelGGL((win_partial_k<T, false>), grid, dim3(PART_THREADS), lds, st, a, t0, ch, po, pm, pz);
    KX_LAUNCH_CHECK();
    hipLaunchKernelGGL((win_merge_k<T>), dim3(s.heads, n), dim3(MERGE_THREADS), (size_t)parts * 4, st, a, t0, parts, po, pm, pz);
    KX_LAUNCH_CHECK();
  }
  return KX_OK;
}

// queries and cache rows in place
template <class T>
int attend(const KxWindowArgs &a, hipStream_t st) {
  if (sizeof(T) == 2 && a.c.dp <= 256 && a.c.vp <= 256) {
    const int nd = a.c.dp / 32, nv = a.c.vp / 32;
    return nd == 1 ? flash_nv<1>(a, nv, st) : nd == 2 ? flash_nv<2>(a, nv, st) : nd <= 4 ? flash_nv<4>(a, nv, st)
         : nd <= 6 ? flash_nv<6>(a, nv, st) : flash_nv<8>(a, nv, st);
  }
  if (sizeof(T) == 4 && flash_f32(a)) {
    const int nd = a.c.dp / 32, nv = a.c.vp / 32;
    return nd == 1 ? flash_f32_nv<1>(a, nv, st) : nd == 2 ? flash_f32_nv<2>(a, nv, st) : nd <= 4 ? flash_f32_nv<4>(a, nv, st)
         : nd <= 6 ? flash_f32_nv<6>(a, nv, st) : flash_f32_nv<8>(a, nv, st);
  }
  KX_REQUIRE(!a.tok_batch && !a.q_ld, "window attention: a part of a step with keys of %d and values of %d", a.s.dim, a.s.vdim);
  return attend_parts<T>(a, false, st);
}

template <class T>
int attention(const KxWindowArgs &a, hipStream_t st) {
  const KxWindowSpec &s = a.s;
  int rc = check(a);
  if (rc) return rc;
  if (a.positions == 1) return attend_parts<T>(a, true, st);
  hipLaunchKernelGGL((win_prep_k<T>), dim3(a.batch * a.positions), dim3(256), 0, st, a);
  KX_LAUNCH_CHECK();
  if (s.pool > 0) {  // blocks whose last position is in this step
    const int b0 = a.pos / s.pool, b1 = std::min((a.pos + a.positions) / s.pool, a.c.blocks);
    if (b1 > b0) {
      hipLaunchKernelGGL((win_pool_k<T>), dim3(b1 - b0, s.kv_heads, a.batch), dim3(256), 0, st, a, b0);
      KX_LAUNCH_CHECK();
    }
  }
  return attend<T>(a, st);
}

}  // namespace

void kx_window_shape(const KxWindowSpec &s, int max_context, int max_positions, KxWindowCache *c, size_t elems[4]) {
  // a step writes its positions before any of them attends, and a block that completes in it may have begun before it
  const int64_t back = std::max(std::min(s.size, max_context), std::min(s.pool, max_context));
  c->cap = (int)std::min<int64_t>(kx_pad(max_context, FK), (back - 1 + max_positions + FK - 1) / FK * FK);
  c->blocks = s.pool > 0 ? max_context / s.pool : 0;
  c->dp = kx_pad(s.dim, 32);
  c->vp = kx_pad(s.vdim, 32);
  elems[0] = (size_t)s.kv_heads * c->cap * c->dp;
  elems[1] = (size_t)s.kv_heads * c->cap * c->vp;
  elems[2] = (size_t)s.kv_heads * c->blocks * c->dp;
  elems[3] = (size_t)s.kv_heads * c->blocks * c->vp;
}

size_t kx_window_part_floats(const KxWindowSpec &s, int max_context, int tokens) {
  // part_keys never goes below 64
  return (size_t)kx_cdiv(most_keys(s, max_context), 64) * floats_per_part(s) * tokens;
}

int kx_window_launch(bool f32, const KxWindowArgs &a, hipStream_t st) { return f32 ? attention<float>(a, st) : attention<uint16_t>(a, st); }

int kx_window_attend(bool f32, const KxWindowArgs &a, hipStream_t st) {
  const int rc = check(a);
  return rc ? rc : f32 ? attend<float>(a, st) : attend<uint16_t>(a, st);
}
