// kx_delta.hip -- see kx_delta.h.  Nothing here is less than 32-bit.  No counterpart in the reference, which has no recurrent layer.
//
// One token per sequence: delta_step_k.  A workgroup owns 32 columns of one head's state; it convolves and norms the
// head's q and k itself, reads its columns once, and writes them once.  All it needs from memory is asked
// for first, and the columns stay in registers (figures in kx_conv.h).
//
// Several positions: the convolutions (kx_conv.hip), then blocks of 16 tokens counted from the step's first position.  With S the
// state before a block, D(i, j) the product of the decays of its tokens i + 1 .. j and G(j) that of tokens 1 .. j,
//   u_j = beta_j (v_j - G(j) S^T k_j - sum_{i < j} D(i, j) (k_i . k_j) u_i)
//   o_j = G(j) S^T q_j + sum_{i <= j} D(i, j) (k_i . q_j) u_i
//   S  <- G(16) S + sum_i D(i, 16) k_i u_i^T,
// which is the recurrence written out for sixteen tokens: only products of decays occur, never a quotient.  The first line is a
// triangular system with the same matrix for every column, I + L, L(j, i) = beta_j D(i, j) (k_i . k_j); delta_block_k inverts it
// once per block and head -- T = (I + L)^-1 diag(beta); its entries are those of products of contractions, beta being at
// most 1 and the keys of unit length, and so do not grow -- and delta_scan_k is left with
//   U = T (V - G K S),  O = G Q S + A U,  S <- G(16) S + (E K)^T U,
// products of 32-bit matrix instructions on the state, which it keeps in registers.  Lengths, decays and T are computed in 64 bits and
// rounded once, which pays for the sums over more tokens: the error is below that of the recurrence in 32 bits, token by token.
#include <algorithm>
#include <atomic>
#include <type_traits>
#include "kx_common.h"
#include "kx_conv.h"
#include "kx_lds_copy.h"
#include "kx_rows.h"
#include "kx_delta.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int SC = 32;  // columns per workgroup of delta_step_k

__device__ __forceinline__ float decay_of(float proj, float a_log, float dt_bias) { return kx_expf(-kx_expf(a_log) * kxr::softplus(proj + dt_bias)); }

__host__ __device__ __forceinline__ KxConvArgs conv_of(const KxDeltaArgs &a) {
  const int nq = a.s.kv_heads * a.s.dim;
  KxConvArgs c;
  c.proj = a.proj; c.proj_ld = a.proj_ld;
  c.segs = 3;
  c.end[0] = nq; c.end[1] = 2 * nq; c.end[2] = c.channels = kx_delta_channels(a.s);
  c.off[0] = a.q_off; c.off[1] = a.k_off; c.off[2] = a.v_off;
  c.taps = a.s.taps; c.w = a.conv;
  c.hist = a.hist; c.hist_out = a.hist_out; c.batch = a.batch; c.positions = a.positions;
  return c;
}

template <int RPT>  // rows of the state per thread
__global__ void __launch_bounds__(256) delta_step_k(KxDeltaArgs a, KxConvArgs cv) {
  __shared__ float q[8 * RPT], k[8 * RPT], v[SC], red[2][4];
  __shared__ float part[2][8][SC];
  const KxDeltaSpec &s = a.s;
  const int D = s.dim, V = s.vdim, tid = threadIdx.x, slices = (V + SC - 1) / SC;
  const int h = blockIdx.x / slices, c0 = (blockIdx.x - h * slices) * SC, b = blockIdx.y;
  const int ratio = s.heads / s.kv_heads, kvh = h / ratio, nq = s.kv_heads * D;
  const int c = tid & (SC - 1), rg = tid / SC, col = min(c0 + c, V - 1);
  float *st = a.state + ((size_t)b * s.heads + h) * D * V;
  // all that comes from memory is asked for first: what the convolutions need, the numbers of the step, the state
  auto channel = [&](int x) { return x < D ? kvh * D + x : nq + kvh * D + x - D; };
  constexpr int CH = (2 * 8 * RPT + 255) / 256;  // channels of q and k per thread
  const bool few = cv.taps <= kxc::FEW, first = c0 == 0 && h % ratio == 0;
  kxc::Channel ch[CH], vch;
  if (few) {
#pragma unroll
    for (int y = 0; y < CH; ++y) ch[y] = kxc::ask(cv, b, channel(min(tid + y * 256, 2 * D - 1)));
    vch = kxc::ask(cv, b, 2 * nq + h * V + min(c0 + (tid & (SC - 1)), V - 1));
  }
  const float *pr = a.proj + (size_t)b * a.proj_ld;
  const float pb = pr[a.b_off + h], pa = pr[a.a_off + h], a_log = a.a_log[h], dt_bias = a.dt_bias[h];
  float S[RPT];
#pragma unroll
  for (int r = 0; r < RPT; ++r) S[r] = st[(size_t)min(rg + 8 * r, D - 1) * V + col];
  float qq = 0.0f, kk = 0.0f;
  auto put = [&](int x, float y) {
    (x >= D ? k : q)[x >= D ? x - D : x] = y;
    if (x >= D) kk = __builtin_fmaf(y, y, kk);
    else qq = __builtin_fmaf(y, y, qq);
  };
  // the convolutions, and their inputs for the next token: this workgroup's value channels, and q and k once per head of theirs
  if (few) {
#pragma unroll
    for (int y = 0; y < CH; ++y) {
      const int x = tid + y * 256;
      if (x >= 2 * D) continue;
      put(x, kxc::silu_of(cv, ch[y]));
      if (first) kxc::shift(cv, b, channel(x), ch[y]);
    }
    if (tid < SC) v[tid] = c0 + tid < V ? kxc::silu_of(cv, vch) : 0.0f;
    if (tid < SC && c0 + tid < V) kxc::shift(cv, b, 2 * nq + h * V + c0 + tid, vch);
  } else {
    for (int x = tid; x < 2 * D; x += 256) {
      put(x, kxc::conv_silu(cv, b, 0, channel(x)));
      if (first) kxc::shift(cv, b, channel(x));
    }
    if (tid < SC) v[tid] = c0 + tid < V ? kxc::conv_silu(cv, b, 0, 2 * nq + h * V + c0 + tid) : 0.0f;
    if (tid < SC && c0 + tid < V) kxc::shift(cv, b, 2 * nq + h * V + c0 + tid);
  }
  qq = kxr::wave_sum(qq);
  kk = kxr::wave_sum(kk);
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = qq;
    red[1][tid >> 6] = kk;
  }
  __syncthreads();
  qq = kk = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    qq += red[0][w];
    kk += red[1][w];
  }
  const float qsc = kx_rsqrtf(qq + s.unit_eps) * kx_rsqrtf((float)D), ksc = kx_rsqrtf(kk + s.unit_eps);
  const float beta = kx_sigmoidf(pb), g = decay_of(pa, a_log, dt_bias);
  float sk = 0.0f;
#pragma unroll
  for (int r = 0; r < RPT; ++r)
    if (rg + 8 * r < D) sk = __builtin_fmaf(S[r], k[rg + 8 * r], sk);
  part[0][rg][c] = sk;
  __syncthreads();
  sk = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) sk += part[0][j][c];
  const float u = beta * (v[c] - g * (sk * ksc)) * ksc;
  float o = 0.0f;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int row = rg + 8 * r;
    if (row >= D) continue;
    const float n = __builtin_fmaf(k[row], u, g * S[r]);
    o = __builtin_fmaf(n, q[row], o);
    if (c0 + c < V) st[(size_t)row * V + c0 + c] = n;
  }
  part[1][rg][c] = o;
  __syncthreads();
  if (rg == 0 && c0 + c < V) {
    o = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) o += part[1][j][c];
    a.o[(size_t)b * s.heads * V + h * V + c0 + c] = o * qsc;
  }
}

constexpr int NB = KX_DELTA_BLOCK, NCF = KX_DELTA_COEF * NB;  // numbers of a block and head:
enum { CF_T = 0, CF_A = NB * NB, CF_GAMMA = 2 * NB * NB, CF_END = CF_GAMMA + NB };  // T, A [token][token], G(j), D(j, 16)
static_assert(CF_END + NB == NCF, "room for a block's numbers");

struct Work {
  float *coef;  // [batch][heads][blocks][NCF]
  float *qk;    // [batch][kv_heads][blocks][k, q, k^T][row / 16][lane][4]: unit k, unit q times dim^-1/2, zeros behind them, as delta_scan_k takes them
  float *raw;   // [tokens][channels]: q, k, v behind convolution and silu
  int blocks;
};
__host__ __device__ __forceinline__ Work work_of(const KxDeltaArgs &a) {
  Work w;
  w.blocks = kx_delta_blocks(a.positions);
  w.coef = a.work;
  w.qk = w.coef + (size_t)a.batch * a.s.heads * w.blocks * NCF;
  w.raw = w.qk + (size_t)a.batch * a.s.kv_heads * w.blocks * 3 * NB * kx_delta_row(a.s);
  return w;
}

// 1 / sqrt of a sum over 16 lanes, in every one of them
__device__ __forceinline__ double row_rsqrt(double v, float eps) {
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m);
  return 1.0 / sqrt(v + eps);
}

// One workgroup per (block, key head): unit norms, the products of the block's keys and queries (thread (j, i) those of tokens
// j and i), then the numbers of each head that shares the key.
__host__ __device__ constexpr int block_stride(int row) { return row + 4; }  // 16 rows at one column fall into different banks
constexpr size_t block_lds(int row) { return (size_t)2 * NB * block_stride(row) * 4; }
__global__ void __launch_bounds__(256) delta_block_k(KxDeltaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float bl_lds[];
  __shared__ float g_s[NB][NB], beta_s[NB][NB];  // [head of the key's][token]
  __shared__ double L[NB][NB + 1];
  const KxDeltaSpec &s = a.s;
  const int D = s.dim, DP = kx_delta_row(s), STR = block_stride(DP), tid = threadIdx.x, sl = tid & 15, j = tid >> 4;
  const int blk = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z, n = a.positions, nq = s.kv_heads * D, C = kx_delta_channels(s), ratio = s.heads / s.kv_heads;
  const Work w = work_of(a);
  float *qs = bl_lds, *ks = qs + NB * STR;
  // tokens of this block; a wave without any makes zeros, which meet step sizes of zero
  const int cnt = min(NB, n - blk * NB);
  const bool any = __builtin_amdgcn_readfirstlane(j) < cnt;
  // decays and step sizes of NB heads at a time, thread (j, sl) those of head r0 + j and token sl, asked for ahead of the rows; a position
  // past the end leaves the state as it is
  float pb = 0.0f, pa = 0.0f, pl = 0.0f, pt = 0.0f;
  auto ask = [&](int r0) {
    const int h = kvh * ratio + min(r0 + j, ratio - 1);
    const float *pr = a.proj + (size_t)(min(blk * NB + sl, n - 1) * a.batch + b) * a.proj_ld;
    pb = pr[a.b_off + h];
    pa = pr[a.a_off + h];
    pl = a.a_log[h];
    pt = a.dt_bias[h];
  };
  auto keep = [&]() {
    g_s[j][sl] = sl < cnt ? decay_of(pa, pl, pt) : 1.0f;
    beta_s[j][sl] = sl < cnt ? kx_sigmoidf(pb) : 0.0f;
  };
  ask(0);
  if (!any) {
    for (int d = sl; d < DP; d += 16) qs[j * STR + d] = ks[j * STR + d] = 0.0f;
  } else {
    const float *row = w.raw + (size_t)(min(blk * NB + j, n - 1) * a.batch + b) * C + kvh * D;
    double qq = 0.0, kk = 0.0;  // the lengths in 64 bits: their error is one of every number of the row
    for (int d0 = sl; d0 < DP; d0 += 64) {
      float q[4], k[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int d = min(d0 + 16 * x, D - 1);
        q[x] = row[d];
        k[x] = row[nq + d];
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const bool in = d0 + 16 * x < D;
        q[x] = in ? q[x] : 0.0f;
        k[x] = in ? k[x] : 0.0f;
        qs[j * STR + d0 + 16 * x] = q[x];
        ks[j * STR + d0 + 16 * x] = k[x];
        qq = __builtin_fma((double)q[x], (double)q[x], qq);
        kk = __builtin_fma((double)k[x], (double)k[x], kk);
      }
    }
    const double qsc = row_rsqrt(qq, s.unit_eps) / sqrt((double)D), ksc = row_rsqrt(kk, s.unit_eps);
    for (int d = sl; d < DP; d += 16) {
      ks[j * STR + d] = (float)(ks[j * STR + d] * ksc);
      qs[j * STR + d] = (float)(qs[j * STR + d] * qsc);
    }
  }
  keep();
  __syncthreads();
  f32x4 *out = (f32x4 *)(w.qk + (((size_t)b * s.kv_heads + kvh) * w.blocks + blk) * 3 * NB * DP);
  for (int x = tid; x < 4 * DP; x += 256) {
    const int c = x & 15, d = (x >> 6) * 16, t = (x >> 4 & 3) * 4;
    out[x] = *(const f32x4 *)(ks + c * STR + d + t);
    out[4 * DP + x] = *(const f32x4 *)(qs + c * STR + d + t);
    f32x4 kt;
#pragma unroll
    for (int e = 0; e < 4; ++e) kt[e] = ks[(t + e) * STR + d + c];
    out[8 * DP + x] = kt;
  }
  const int i = sl;
  f32x4 kk4[4] = {}, kq4[4] = {};  // sixteen partial sums each: short chains, also of roundings
  for (int d0 = 0; d0 < (any ? DP : 0); d0 += 16)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int d = d0 + 4 * x;
      const f32x4 ki = *(const f32x4 *)(ks + i * STR + d), kj = *(const f32x4 *)(ks + j * STR + d), qj = *(const f32x4 *)(qs + j * STR + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kk4[x][e] = __builtin_fmaf(ki[e], kj[e], kk4[x][e]);
        kq4[x][e] = __builtin_fmaf(ki[e], qj[e], kq4[x][e]);
      }
    }
  auto total = [](const f32x4 (&p)[4]) {
    const f32x4 t = (p[0] + p[1]) + (p[2] + p[3]);
    return (t[0] + t[1]) + (t[2] + t[3]);
  };
  const float kk = total(kk4), kq = total(kq4);  // k_i . k_j, k_i . q_j
  for (int r = 0; r < ratio; ++r) {
    const int h = kvh * ratio + r;
    float *cf = w.coef + (((size_t)b * s.heads + h) * w.blocks + blk) * NCF;
    __syncthreads();  // the head before has been worked on
    if (r && r % NB == 0) {
      ask(r);
      keep();
      __syncthreads();
    }
    const float *const g = g_s[r % NB], *const beta = beta_s[r % NB];
    double d = 1.0;  // D(i, j): rounded once, not with each decay; a state that decays by it has fewer roundings than token by token
    for (int m = i + 1; m <= min(j, cnt - 1); ++m) d *= g[m];
    L[j][i] = i < j ? beta[j] * d * kk : 0.0;
    cf[CF_A + j * NB + i] = i <= j ? (float)(d * kq) : 0.0f;
    if (i == 0) cf[CF_GAMMA + j] = (float)(d * g[0]);
    if (j == NB - 1) cf[CF_END + i] = (float)d;
    __syncthreads();
    if (tid < NB) {  // column tid of the inverse; rows past the end are zero
      auto invert = [&](auto few) {
        constexpr int ROWS = decltype(few)::value ? 4 : NB;
        double t[ROWS];
#pragma unroll
        for (int y = 0; y < NB; ++y) {
          float c = 0.0f;
          if (y < ROWS) {
            double v = y == tid ? 1.0 : 0.0;
#pragma unroll
            for (int m = 0; m < y; ++m) v = __builtin_fma(-L[y][m], t[m], v);
            t[y] = v;
            c = (float)(v * beta[tid]);
          }
          cf[CF_T + y * NB + tid] = y < tid ? 0.0f : c;  // nothing of a token in the rows before it, whatever its numbers are
        }
      };
      if (cnt <= 4) invert(std::true_type{});
      else invert(std::false_type{});
    }
  }
}

// A block's lower triangular matrix times a row per token, in 32-bit matrix instructions.  Those multiply the zeros above the
// diagonal too, so a row that is not finite would reach the tokens before it; then the products are made token by token
// from the rows up to it.
__device__ __forceinline__ f32x4 lower(f32x4 m, f32x4 x) {
  auto product = [&](f32x4 y) {
    f32x4 p = __builtin_amdgcn_mfma_f32_16x16x4f32(m[0], y[0], f32x4{}, 0, 0, 0), q = __builtin_amdgcn_mfma_f32_16x16x4f32(m[2], y[2], f32x4{}, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x4f32(m[1], y[1], p, 0, 0, 0);
    return p + __builtin_amdgcn_mfma_f32_16x16x4f32(m[3], y[3], q, 0, 0, 0);
  };
  const bool odd = !(__builtin_isfinite(x[0]) && __builtin_isfinite(x[1]) && __builtin_isfinite(x[2]) && __builtin_isfinite(x[3]));
  if (__builtin_expect(__ballot(odd) == 0, 1)) return product(x);
  const int g = (threadIdx.x & 63) >> 4;
  f32x4 out = {};
#pragma unroll 1
  for (int j = 0; j < NB; ++j) {
    f32x4 y;
#pragma unroll
    for (int v = 0; v < 4; ++v) y[v] = 4 * g + v <= j ? x[v] : 0.0f;
    y = product(y);
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = 4 * g + v == j ? y[v] : out[v];
  }
  return out;
}

// A workgroup owns 16 columns of a head's state, four waves a quarter of the rows each: row-block rb of wave w is rows 16 (w RB +
// rb) .. + 15 as v_mfma_f32_16x16x4_f32 leaves its result -- lane (c, g) holds rows 4 g + v of column c --, which is also how
// that instruction takes its second operand if the columns of a row-block meet in the order 4 g + v.
// Bound by the chain of a block: 4 RB products for K S, their sums over the waves through LDS and a barrier, 4 products with
// T, 4 RB with the keys' transpose.  Q S fills the time the exchange takes; a fifth wave makes the read-outs, a block
// behind the others, which do not wait for it.  The numbers of the next SETS blocks are on their way meanwhile.
// The whole operator, us: 2048 tokens of 16 heads of 128 x 128 175 with two sets, 190 with three, 198 with one (the registers of three
// leave a CU one workgroup instead of two); on the vector ALU, four tokens per dependent step, 370.  With 32 sequences of 512
// tokens, where workgroups hide each other's waits, 894 with one set (three workgroups per CU), 1015 with two, 1085 with three;
// rows of 64, 192 and 256 columns keep two (867, 943 and 1469 of 32 sequences against 981, 1105 and 1568).  A step of few tokens
// is the state's way through the chip and little else: 32 sequences of 2 tokens 64 with one set, 94 with two (four tokens per
// dependent step 64), and 38 for 32 heads of 64 x 64 -- 50 if the block after the only one is asked for -- where four tokens per
// dependent step took 33.  Steps of 17 tokens, a block of them and one token, are what blocks of 16 pay least for: 32 sequences, 64 heads
// of 128 x 128 338 (302), 32 of 64 x 64 73 (66), at 32 tokens 368 (407) and 76 (85).
template <int RB, int SETS, bool MORE>  // MORE: the step may have more than SETS blocks
__global__ void __launch_bounds__(320, 2) delta_scan_k(KxDeltaArgs a) {
  __shared__ f32x4 sk_s[2][4][64], sq_s[2][4][64], u_s[2][64];
  const KxDeltaSpec &s = a.s;
  const int D = s.dim, V = s.vdim, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.z, kvh = h / (s.heads / s.kv_heads), n = a.positions, C = kx_delta_channels(s);
  const int col = blockIdx.y * 16 + c;
  const Work w = work_of(a);
  constexpr int DP = RB * 64;
  const f32x4 *coef = (const f32x4 *)(w.coef + ((size_t)b * s.heads + h) * w.blocks * NCF);
  if (wave == 4) {
    auto numbers = [&](int blk, int at) { return coef[(size_t)min(blk, w.blocks - 1) * (NCF / 4) + at]; };
    f32x4 A = numbers(0, CF_A / 4 + c * 4 + g), gamma = numbers(0, CF_GAMMA / 4 + g);
    kx_lds_barrier();
    for (int blk = 0; blk < w.blocks; ++blk) {
      kx_lds_barrier();  // the sums and the rows u of block blk are there
      f32x4 nextA = A, nextG = gamma;
      if constexpr (MORE) {
        nextA = numbers(blk + 1, CF_A / 4 + c * 4 + g);
        nextG = numbers(blk + 1, CF_GAMMA / 4 + g);
      }
      const f32x4(*q)[64] = sq_s[blk & 1];
      const f32x4 qs = (q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane]), au = lower(A, u_s[blk & 1][lane]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int t = blk * NB + 4 * g + v;
        if (t < n && col < V) a.o[((size_t)(t * a.batch + b) * s.heads + h) * V + col] = __builtin_fmaf(gamma[v], qs[v], au[v]);
      }
      A = nextA;
      gamma = nextG;
    }
    return;
  }
  const int row0 = wave * RB * 16, last = (n - 1) / NB;
  const f32x4 *qk = (const f32x4 *)(w.qk + ((size_t)b * s.kv_heads + kvh) * w.blocks * 3 * NB * DP) + wave * RB * 64 + lane;
  const float *raw = w.raw + (size_t)b * C + (size_t)2 * s.kv_heads * D + h * V + min(col, V - 1);
  float *st = a.state + ((size_t)b * s.heads + h) * D * V;
  size_t row_at[4], last_at[4];  // of a token's values in their block; in the last one its last token stands for those past the end
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    row_at[v] = (size_t)(4 * g + v) * a.batch * C;
    last_at[v] = (size_t)min(4 * g + v, n - 1 - last * NB) * a.batch * C;
  }
  struct Set {
    f32x4 k[RB], q[RB], kt[RB], t, gamma, end, v;
  };
  auto load = [&](Set &x, int blk) {
    blk = min(blk, w.blocks - 1);  // past the end: not used
    const f32x4 *kp = qk + (size_t)blk * 12 * DP, *cf = coef + (size_t)blk * (NCF / 4);
    const float *rows = raw + (size_t)blk * NB * a.batch * C;
#pragma unroll
    for (int v = 0; v < 4; ++v) x.v[v] = rows[blk < last ? row_at[v] : last_at[v]];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      x.k[r] = kp[r * 64];
      x.q[r] = kp[4 * DP + r * 64];
      x.kt[r] = kp[8 * DP + r * 64];
    }
    x.t = cf[(CF_T + c * NB) / 4 + g];
    x.gamma = cf[CF_GAMMA / 4 + g];
    x.end = cf[CF_END / 4 + g];
  };
  f32x4 S[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = row0 + r * 16 + 4 * g + v;
      const float x = st[(size_t)min(row, D - 1) * V + min(col, V - 1)];
      S[r][v] = row < D && col < V ? x : 0.0f;
    }
  // the wave's part of a product with the state; sums of four, then those of sums: no more roundings in a row than a sum over lanes has
  auto times_state = [&](const f32x4 (&m)[RB]) {
    f32x4 p[RB][4];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) p[r][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r][v], S[r][v], f32x4{}, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < RB; ++r) p[r][0] = (p[r][0] + p[r][1]) + (p[r][2] + p[r][3]);
    if constexpr (RB == 1) return p[0][0];
    if constexpr (RB == 2) return p[0][0] + p[1][0];
    if constexpr (RB == 3) return (p[0][0] + p[1][0]) + p[2][0];
    if constexpr (RB == 4) return (p[0][0] + p[1][0]) + (p[2][0] + p[3][0]);
  };
  auto step = [&](Set &x, int blk) {
    sk_s[blk & 1][wave][lane] = times_state(x.k);
    kx_lds_barrier();  // the waves' sums; and everybody is done with the block before the last
    const f32x4 sk = (sk_s[blk & 1][0][lane] + sk_s[blk & 1][1][lane]) + (sk_s[blk & 1][2][lane] + sk_s[blk & 1][3][lane]);
    sq_s[blk & 1][wave][lane] = times_state(x.q);
    f32x4 e;
#pragma unroll
    for (int v = 0; v < 4; ++v) e[v] = __builtin_fmaf(-x.gamma[v], sk[v], x.v[v]);
    const f32x4 u = lower(x.t, e);
    if (wave == 0) u_s[blk & 1][lane] = u;
    const float all = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, (float)x.gamma[3]), 48));  // G(16)
#pragma unroll
    for (int v = 0; v < 4; ++v) e[v] = u[v] * x.end[v];
    f32x4 p[RB];  // the block's sums first: the state is rounded once a block
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int r = 0; r < RB; ++r) p[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[r][v], e[v], v ? p[r] : f32x4{}, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) S[r][v] = __builtin_fmaf(all, S[r][v], p[r][v]);
    if constexpr (MORE) load(x, blk + SETS);
  };
  Set x[SETS];  // the loads in flight stay in the registers that they arrive in
#pragma unroll
  for (int y = 0; y < SETS; ++y) load(x[y], y);
  int blk = 0;
  for (; blk + SETS <= w.blocks; blk += SETS) {
#pragma unroll
    for (int y = 0; y < SETS; ++y) step(x[y], blk + y);
  }
  if (MORE && SETS == 2 && blk < w.blocks) step(x[0], blk);
  kx_lds_barrier();
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = row0 + r * 16 + 4 * g + v;
      if (row < D && col < V) st[(size_t)row * V + col] = S[r][v];
    }
}

template <int RB>
void scan(const KxDeltaArgs &a, dim3 grid, hipStream_t st) {
  const int blocks = work_of(a).blocks;
  auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(320), 0, st, a); };
  if (blocks == 1) return run(delta_scan_k<RB, 1, false>);
  // one set where rows of 128 make more workgroups than the chip has CUs (figures at delta_scan_k)
  if constexpr (RB == 2)
    if ((long)grid.x * grid.y * grid.z > kx_device_cus()) return run(delta_scan_k<RB, 1, true>);
  run(delta_scan_k<RB, 2, true>);
}

}  // namespace

int kx_delta_launch(const KxDeltaArgs &a, hipStream_t st) {
  const KxDeltaSpec &s = a.s;
  KX_REQUIRE(s.heads > 0 && s.kv_heads > 0 && s.heads % s.kv_heads == 0 && s.dim > 0 && s.vdim > 0 && s.taps > 0,
             "delta rule: heads=%d kv_heads=%d dim=%d vdim=%d taps=%d", s.heads, s.kv_heads, s.dim, s.vdim, s.taps);
  KX_REQUIRE(s.dim <= 256, "delta rule: keys of %d columns, at most 256", s.dim);
  KX_REQUIRE(a.batch > 0 && a.positions > 0 && (s.taps == 1 || (a.hist && a.hist_out && a.hist != a.hist_out)), "delta rule: %d x %d tokens", a.batch, a.positions);
  if (a.positions == 1) {
    const dim3 grid(s.heads * kx_cdiv(s.vdim, SC), a.batch);
    if (s.dim <= 64) hipLaunchKernelGGL(delta_step_k<8>, grid, dim3(256), 0, st, a, conv_of(a));
    else if (s.dim <= 128) hipLaunchKernelGGL(delta_step_k<16>, grid, dim3(256), 0, st, a, conv_of(a));
    else hipLaunchKernelGGL(delta_step_k<32>, grid, dim3(256), 0, st, a, conv_of(a));
    KX_LAUNCH_CHECK();
    return KX_OK;
  }
  KX_REQUIRE(a.work && (uintptr_t)a.work % 16 == 0, "delta rule: no scratch, or none for pieces of 16 bytes");
  const int rc = kx_conv_launch(conv_of(a), work_of(a).raw, st);
  if (rc) return rc;
  const int row = kx_delta_row(s);
  hipLaunchKernelGGL(delta_block_k, dim3(work_of(a).blocks, s.kv_heads, a.batch), dim3(256), block_lds(row), st, a);
  KX_LAUNCH_CHECK();
  const dim3 grid(s.heads, kx_cdiv(s.vdim, 16), a.batch);
  if (row == 64) scan<1>(a, grid, st);
  else if (row == 128) scan<2>(a, grid, st);
  else if (row == 192) scan<3>(a, grid, st);
  else scan<4>(a, grid, st);
  KX_LAUNCH_CHECK();
  return KX_OK;
}
