// kx_rows.h -- activation rows of the hybrid decoder, built by one workgroup: what a matrix product reads as its
// input.  The same code fills a row in LDS (the prologue of a decode GEMV, kx_linear.hip) and in memory (row_k, for
// steps of many tokens).  No counterpart in the reference, whose decoder has one residual stream.
//
//   NORM   h = w * groupnorm(sum_s in[s] x_s): the input of a sublayer with several residual streams
//   GATED  per head: a recurrence's read-out over its root mean square, times a weight, with silu(gate) behind the norm or in
//          front of it
//   SHIFT  several mixes of a normed row with the one of the position before it, and the row itself
//   TANH   tanh of a 32-bit row
//   PLAIN  a row that is in memory already
// Rows are padded to the matrix's leading dimension; pad columns are zero (or, in memory, finite: the matrix's pad
// columns are zero).
#pragma once
#include "kx_linear.h"
#include "kx_math.h"
#include "kx_wave.h"

namespace kxr {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <class T> struct Elem;
template <> struct Elem<uint16_t> {
  static __device__ __forceinline__ float load(const uint16_t *p) { return kx_bf16_f32(*p); }
  static __device__ __forceinline__ uint16_t make(float v) { return kx_bf16_rne(v); }
  // eight elements of a weight stream, as they come
  struct Raw { u32x4 a; };
  static __device__ __forceinline__ Raw stream(const uint16_t *p) { return Raw{__builtin_nontemporal_load((const u32x4 *)p)}; }
  static __device__ __forceinline__ Raw cached(const uint16_t *p) { return Raw{*(const u32x4 *)p}; }
  static __device__ __forceinline__ void unpack(float (&f)[8], const Raw &r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = kx_bits_f32(r.a[i] << 16);
      f[2 * i + 1] = kx_bits_f32(r.a[i] & 0xffff0000u);
    }
  }
};
template <> struct Elem<float> {
  static __device__ __forceinline__ float load(const float *p) { return *p; }
  static __device__ __forceinline__ float make(float v) { return v; }
  struct Raw { u32x4 a, b; };
  static __device__ __forceinline__ Raw stream(const float *p) {
    return Raw{__builtin_nontemporal_load((const u32x4 *)p), __builtin_nontemporal_load((const u32x4 *)(p + 4))};
  }
  static __device__ __forceinline__ Raw cached(const float *p) { return Raw{((const u32x4 *)p)[0], ((const u32x4 *)p)[1]}; }
  static __device__ __forceinline__ void unpack(float (&f)[8], const Raw &r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[i] = kx_bits_f32(r.a[i]);
      f[4 + i] = kx_bits_f32(r.b[i]);
    }
  }
};

// sigmoid for a value that is rounded to T next: without branches and with the approximate reciprocal for bf16
template <class T>
__device__ __forceinline__ float sigmoid_for(float x) {
  if constexpr (sizeof(T) == 4) return kx_sigmoidf(x);
  else return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * x));
}

// log(1 + exp(x))
__device__ __forceinline__ float softplus(float x) { return fmaxf(x, 0.0f) + log1pf(kx_expf(-fabsf(x))); }

// sum over the lanes of a wave, in every lane
__device__ __forceinline__ float wave_sum(float v) {
  float t = v;
  kxw::swap_halves32(v, t);
  v += t;
  t = v;
  kxw::swap_rows16(v, t);
  v += t;
  v += kxw::dpp_f<kxw::DPP_ROW_MIRROR>(v);
  v += kxw::dpp_f<kxw::DPP_ROW_HALF_MIRROR>(v);
  v += kxw::dpp_f<kxw::DPP_QUAD_XOR2>(v);
  v += kxw::dpp_f<kxw::DPP_QUAD_XOR1>(v);
  return v;
}
// sum over a workgroup, in every thread; red: one float per wave
__device__ __forceinline__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  const int nw = blockDim.x >> 6;
  __syncthreads();  // red may still be read from the last call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = red[0];
  for (int w = 1; w < nw; ++w) s += red[w];
  return s;
}

// sums of squares of `groups` equal parts of u[0 .. cols) -> part[g * spg] = 1 / root mean square; spg slices per group, whose
// sums are in part[] and behind a barrier
__device__ __forceinline__ void group_scales(float *part, int groups, int spg, int gs, float eps) {
  for (int g = threadIdx.x; g < groups; g += blockDim.x) {
    float s = part[g * spg];
    for (int j = 1; j < spg; ++j) s += part[g * spg + j];
    part[g * spg] = kx_rsqrtf(s / (float)gs + eps);
  }
  __syncthreads();
}

// Row `tok` into dst[0 .. ld), variants vstride apart.  u: LDS scratch of kx_row_scratch(a) floats.  Whole workgroup; ends
// with a barrier.  keep: this workgroup writes what the row's kind carries over to the next step.  need: the variants
// to build, a bit each.
// KIND: the row's kind where it is known when the kernel is compiled.
// A row is a few KB and the time to build one is the time of its loads one after the other: every loop asks for what UB of its
// turns read before the first of them stores anything (a store through `dst` would keep the compiler from doing so), and what
// comes behind a sum is asked for in front of it.
constexpr int UB = 4;
template <class T, int KIND = -1>
__device__ __forceinline__ void build_row(const KxRowArgs &a, int tok, T *dst, int ld, float *u, size_t vstride = 0, bool keep = false,
                                          uint32_t need = ~0u) {
  const int tid = threadIdx.x, n = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = n >> 6, kind = KIND >= 0 ? KIND : a.kind;
  if (a.rows_map) tok = a.rows_map[tok];
  const int xld = a.streams_ld ? a.streams_ld : a.n_streams * a.cols;
  if (kind == KX_ROW_NORM) {
    float *part = u + a.cols;
    const float *x = a.streams + (size_t)tok * xld;
    const int gs = a.cols / a.groups, spg = max(1, nw / a.groups), units = a.groups * spg, per = (gs + spg - 1) / spg;
    float wf[UB];
#pragma unroll
    for (int k = 0; k < UB; ++k) wf[k] = a.w[min(tid + k * n, a.cols - 1)];
    for (int k = wave; k < units; k += nw) {  // a wave takes a slice of one group
      const int g = k / spg, s = k - g * spg, hi = min(gs, (s + 1) * per);
      float v = 0.0f;
      for (int j0 = s * per + lane; j0 < hi; j0 += 64 * UB) {
        float y[UB] = {};
        for (int t = 0; t < a.n_streams; ++t) {
          const float in = a.in ? a.in[t] : 1.0f;
#pragma unroll
          for (int i = 0; i < UB; ++i) y[i] = __builtin_fmaf(in, x[(size_t)t * a.cols + g * gs + min(j0 + 64 * i, hi - 1)], y[i]);
        }
#pragma unroll
        for (int i = 0; i < UB; ++i)
          if (j0 + 64 * i < hi) {
            u[g * gs + j0 + 64 * i] = y[i];
            v = __builtin_fmaf(y[i], y[i], v);
          }
      }
      v = wave_sum(v);
      if (lane == 0) part[k] = v;
    }
    __syncthreads();
    group_scales(part, a.groups, spg, gs, a.eps);
    for (int c0 = tid; c0 < ld; c0 += n * UB) {
      if (c0 != tid)
#pragma unroll
        for (int k = 0; k < UB; ++k) wf[k] = a.w[min(c0 + k * n, a.cols - 1)];
#pragma unroll
      for (int k = 0; k < UB; ++k) {
        const int c = c0 + k * n;
        if (c < ld) dst[c] = Elem<T>::make(c < a.cols ? u[c] * part[(c / gs) * spg] * wf[k] : 0.0f);
      }
    }
  } else if (kind == KX_ROW_SHIFT) {
    const bool first = tok < a.batch;
    const float *x = a.streams + (size_t)tok * xld, *x1 = first ? a.prev + (size_t)tok * a.cols : x - (size_t)a.batch * xld;
    float xv[UB], yv[UB], wv[UB];  // of the present UB columns
    auto ask = [&](int c0) {
#pragma unroll
      for (int k = 0; k < UB; ++k) {
        const int c = min(c0 + k * n, a.cols - 1);
        xv[k] = x[c];
        yv[k] = x1[c];
        wv[k] = a.w[c];
      }
    };
    float v = 0.0f, v1 = 0.0f;
    for (int c0 = tid; c0 < a.cols; c0 += n * UB) {
      ask(c0);
#pragma unroll
      for (int k = 0; k < UB; ++k)
        if (c0 + k * n < a.cols) {
          v = __builtin_fmaf(xv[k], xv[k], v);
          v1 = __builtin_fmaf(yv[k], yv[k], v1);
        }
    }
    const float sc = kx_rsqrtf(block_sum(v, u) / (float)a.cols + a.eps), sc1 = kx_rsqrtf(block_sum(v1, u) / (float)a.cols + a.eps);
    const bool last = keep && tok + a.batch >= a.tokens;
    for (int c0 = tid; c0 < ld; c0 += n * UB) {
      if (a.cols > n * UB) ask(c0);  // otherwise they are still there
      float h[UB], d[UB];
#pragma unroll
      for (int k = 0; k < UB; ++k) {
        const int c = c0 + k * n;
        h[k] = c < a.cols ? xv[k] * sc * wv[k] : 0.0f;
        d[k] = c < a.cols ? (first ? yv[k] : yv[k] * sc1 * wv[k]) - h[k] : 0.0f;
        if (last && c < a.cols) a.prev_out[(size_t)(tok + a.batch - a.tokens) * a.cols + c] = h[k];
      }
      for (int m = 0; m < a.n_mix; ++m)
        if (need >> m & 1) {
          float mu[UB];
#pragma unroll
          for (int k = 0; k < UB; ++k) mu[k] = a.mu[(size_t)m * a.cols + min(c0 + k * n, a.cols - 1)];
#pragma unroll
          for (int k = 0; k < UB; ++k)
            if (c0 + k * n < ld) dst[m * vstride + c0 + k * n] = Elem<T>::make(c0 + k * n < a.cols ? __builtin_fmaf(d[k], mu[k], h[k]) : 0.0f);
        }
#pragma unroll
      for (int k = 0; k < UB; ++k)
        if (c0 + k * n < ld) dst[a.n_mix * vstride + c0 + k * n] = Elem<T>::make(h[k]);
    }
  } else if (kind == KX_ROW_GATED) {
    const int cols = a.heads * a.vdim, hl = a.tail ? a.head_ld : ld;
    const float *o = a.o + (size_t)tok * cols, *gate = a.gate + (size_t)tok * a.gate_ld;
    auto gated = [&](float y, float g) { return a.gate_first ? y * g * sigmoid_for<T>(g) : y; };
    auto out = [&](int c, float y, float g, float w) {
      y *= w;
      dst[c] = Elem<T>::make(a.gate_first ? y : y * g * sigmoid_for<T>(g));
    };
    auto weight = [&](int c, int d) { return a.w[a.w_per_column ? c : d]; };
    if (a.heads < 8) {  // a few long parts: several waves each
      float *part = u + cols;
      const int spg = max(1, nw / a.heads), units = a.heads * spg, per = (a.vdim + spg - 1) / spg;
      for (int k = wave; k < units; k += nw) {
        const int h = k / spg, s = k - h * spg, hi = min(a.vdim, (s + 1) * per);
        float v = 0.0f;
        for (int d0 = s * per + lane; d0 < hi; d0 += 64 * UB) {
          float ov[UB], gv[UB];
#pragma unroll
          for (int i = 0; i < UB; ++i) {
            const int c = h * a.vdim + min(d0 + 64 * i, hi - 1);
            ov[i] = o[c];
            gv[i] = a.gate_first ? gate[c] : 0.0f;
          }
#pragma unroll
          for (int i = 0; i < UB; ++i)
            if (d0 + 64 * i < hi) {
              const float y = gated(ov[i], gv[i]);
              u[h * a.vdim + d0 + 64 * i] = y;
              v = __builtin_fmaf(y, y, v);
            }
        }
        v = wave_sum(v);
        if (lane == 0) part[k] = v;
      }
      __syncthreads();
      group_scales(part, a.heads, spg, a.vdim, a.eps);
      for (int c0 = tid; c0 < cols; c0 += n * UB) {
        float wv[UB], gv[UB];
#pragma unroll
        for (int i = 0; i < UB; ++i) {
          const int c = min(c0 + i * n, cols - 1);
          wv[i] = weight(c, c % a.vdim);
          gv[i] = a.gate_first ? 0.0f : gate[c];
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
          const int c = c0 + i * n;
          if (c < cols) out(c, u[c] * part[(c / a.vdim) * spg], gv[i], wv[i]);
        }
      }
    } else if (a.vdim <= 128) {  // a wave takes UB heads at a time, two columns of each per lane
      const int two = a.vdim > 64;
      for (int h0 = wave; h0 < a.heads; h0 += nw * UB) {
        float ov[UB][2], gv[UB][2], wv[UB][2];
#pragma unroll
        for (int i = 0; i < UB; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if (j && !two) continue;
            const int d = min(lane + 64 * j, a.vdim - 1), c = min(h0 + i * nw, a.heads - 1) * a.vdim + d;
            ov[i][j] = o[c];
            gv[i][j] = gate[c];
            wv[i][j] = weight(c, d);
          }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
          const int h = h0 + i * nw;
          if (h >= a.heads) break;
          float v = 0.0f, y[2];
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (lane + 64 * j < a.vdim) {
              y[j] = gated(ov[i][j], gv[i][j]);
              v = __builtin_fmaf(y[j], y[j], v);
            }
          const float sc = kx_rsqrtf(wave_sum(v) / (float)a.vdim + a.eps);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (lane + 64 * j < a.vdim) out(h * a.vdim + lane + 64 * j, y[j] * sc, gv[i][j], wv[i][j]);
        }
      }
    } else {
      for (int h = wave; h < a.heads; h += nw) {
        float v = 0.0f;
        for (int d = lane; d < a.vdim; d += 64) {
          const int c = h * a.vdim + d;
          const float y = gated(o[c], gate[c]);
          v = __builtin_fmaf(y, y, v);
        }
        const float sc = kx_rsqrtf(wave_sum(v) / (float)a.vdim + a.eps);
        for (int d = lane; d < a.vdim; d += 64) {
          const int c = h * a.vdim + d;
          out(c, gated(o[c], gate[c]) * sc, gate[c], weight(c, d));
        }
      }
    }
    for (int c = cols + tid; c < hl; c += n) dst[c] = Elem<T>::make(0.0f);
    if (a.tail) {
      const T *x = (const T *)a.tail + (size_t)tok * a.tail_ld;
#pragma unroll 1
      for (int c0 = tid * 8; c0 < ld - hl; c0 += n * 8 * UB) {
        typename Elem<T>::Raw r[UB];
#pragma unroll
        for (int k = 0; k < UB; ++k) r[k] = Elem<T>::cached(x + min(c0 + k * n * 8, ld - hl - 8));
#pragma unroll
        for (int k = 0; k < UB; ++k)
          if (c0 + k * n * 8 < ld - hl) *(typename Elem<T>::Raw *)(dst + hl + c0 + k * n * 8) = r[k];
      }
    }
  } else if (kind == KX_ROW_TANH) {
    const float *x = a.streams + (size_t)tok * xld;
    for (int c = tid; c < ld; c += n) dst[c] = Elem<T>::make(c < a.cols ? tanhf(x[c]) : 0.0f);
  } else {
    // turn by turn: a row takes one or two, and asking for UB, most of them past the end, cost 0.2 us a token (1024 x 4096, 4 tokens,
    // bf16 8.7 -> 9.3 us, f32 9.6 -> 11.1; 8.6 and 10.1 now)
    const T *x = (const T *)a.x + (size_t)tok * a.x_ld;
    for (int c = tid * 8; c < ld; c += n * 8) *(typename Elem<T>::Raw *)(dst + c) = Elem<T>::cached(x + c);
  }
  __syncthreads();
}

}  // namespace kxr
