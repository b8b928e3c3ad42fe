// kx_experts.hip -- see kx_experts.h.
//
// The counterpart of the router and of expert_accum_k (src/kimi_exec.cu:372-391, :835-877) for a decoder whose experts are
// bf16 or f32 matrices of any size: the host never sees the expert ids.
#include <algorithm>
#include "kx_common.h"
#include "kx_experts.h"
#include "kx_read_once.h"

namespace {

__global__ void __launch_bounds__(256) route_k(KxExpertArgs e, int tokens) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t < tokens) kxe::route_wave(e.logits + (size_t)t * e.logits_ld, e.bias, e.experts, e.top, e.ids + (size_t)t * e.top, e.weights + (size_t)t * e.top);
}

// One workgroup: counts per expert, their running sums, tiles, and a slot for every pair.  ROUTE: of up to BUCKET_WAVES tokens, which it routes itself, a
// wave each.  It is one chain of waits, so a thread asks for PAIRS_AHEAD pairs at once and a wave makes its own running sums.  2046 tokens, 8 experts
// each: 17.4 us with a pair at a time and sums over LDS, 12.0 now; 8 tokens: 6.5 + 4.2 and a launch between them, 11.8 in one; 10.6 and, with
// their pairs kept in LDS instead of read back from memory, 9.8.
constexpr int BUCKET_WAVES = KX_MAX_EXPERTS / 64, PAIRS_AHEAD = 16;
template <bool ROUTE>
__global__ void __launch_bounds__(KX_MAX_EXPERTS) bucket_k(KxExpertArgs e, KxExpertSlots s, int tokens) {
  __shared__ int count[KX_MAX_EXPERTS], total[2][BUCKET_WAVES];
  __shared__ int own_id[ROUTE ? BUCKET_WAVES * KX_MAX_TOP : 1];  // of the pairs it routes itself
  __shared__ float own_weight[ROUTE ? BUCKET_WAVES * KX_MAX_TOP : 1];
  static_assert(BUCKET_WAVES * KX_MAX_TOP <= KX_MAX_EXPERTS, "a thread has one pair of those");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), pairs = tokens * e.top;
  count[tid] = 0;
  if (ROUTE && wave < tokens) kxe::route_wave(e.logits + (size_t)wave * e.logits_ld, e.bias, e.experts, e.top, own_id + wave * e.top, own_weight + wave * e.top);
  __syncthreads();
  int id[PAIRS_AHEAD];
  float weight[PAIRS_AHEAD];
  auto ask = [&](int p0) {  // pairs p0 + tid, and so on
    if constexpr (ROUTE) {
      id[0] = own_id[min(tid, pairs - 1)];
      weight[0] = own_weight[min(tid, pairs - 1)];
      if (tid < pairs) {
        e.ids[tid] = id[0];
        e.weights[tid] = weight[0];
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < PAIRS_AHEAD; ++k)
      if (p0 + k * KX_MAX_EXPERTS < pairs) {
        const int p = min(p0 + k * KX_MAX_EXPERTS + tid, pairs - 1);
        id[k] = s.ids[p];
        weight[k] = s.weights[p];
      }
  };
  constexpr int AT_ONCE = PAIRS_AHEAD * KX_MAX_EXPERTS;
  for (int p0 = 0; p0 < pairs; p0 += AT_ONCE) {
    ask(p0);
#pragma unroll
    for (int k = 0; k < PAIRS_AHEAD; ++k)
      if (p0 + k * KX_MAX_EXPERTS + tid < pairs) atomicAdd(&count[id[k]], 1);
  }
  __syncthreads();
  const int n = count[tid], tiles = (n + e.tile_slots - 1) / e.tile_slots;
  int at = n, tile_at = tiles;  // inclusive sums
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(at, d), y = __shfl_up(tile_at, d);
    if (lane >= d) {
      at += x;
      tile_at += y;
    }
  }
  if (lane == 63) {
    total[0][wave] = at;
    total[1][wave] = tile_at;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < BUCKET_WAVES - 1; ++w)
    if (w < wave) {
      at += total[0][w];
      tile_at += total[1][w];
    }
  const int slot0 = at - n, tile0 = tile_at - tiles;
  if (tid == KX_MAX_EXPERTS - 1) *s.n_tiles = tile_at;
  for (int i = 0; i < tiles; ++i) s.tiles[tile0 + i] = make_int4(tid, slot0 + i * e.tile_slots, min(e.tile_slots, n - i * e.tile_slots), tiles);
  count[tid] = slot0;
  __syncthreads();
  for (int p0 = 0; p0 < pairs; p0 += AT_ONCE) {
    if (pairs > AT_ONCE) ask(p0);  // otherwise they are still there
#pragma unroll
    for (int k = 0; k < PAIRS_AHEAD; ++k) {
      const int p = p0 + k * KX_MAX_EXPERTS + tid;
      if (p >= pairs) continue;
      const int slot = atomicAdd(&count[id[k]], 1);
      s.gather[slot] = p / e.top;
      s.slot_weight[slot] = weight[k];
      s.slot_of[p] = slot;
    }
  }
}

// x of token blockIdx.x += its experts' rows, in their order; a thread has W columns.  Prompts are bound by memory (2046 tokens of 2048 columns and 8 experts
// 35 us, 4.8 TB/s), few tokens by one wait after the other, so everything is asked for before the first sum: 8 tokens 8.4 us before, 5.0 now.
constexpr int ROWS_AHEAD = 8;
template <int W>
__global__ void __launch_bounds__(256) combine_k(KxExpertSlots s, const float *__restrict__ y, float *__restrict__ x, int top, int width) {
  typedef float V __attribute__((ext_vector_type(W)));
  const int *slot = s.slot_of + (size_t)blockIdx.x * top;
  const int c = (blockIdx.y * 256 + threadIdx.x) * W;
  if (c >= width) return;
  V *to = (V *)(x + (size_t)blockIdx.x * width + c);
  const V old = *to;
  V v = {}, r[ROWS_AHEAD];
  for (int j0 = 0; j0 < top; j0 += ROWS_AHEAD) {
#pragma unroll
    for (int j = 0; j < ROWS_AHEAD; ++j)
      if (j0 + j < top) r[j] = *(const V *)(y + (size_t)slot[j0 + j] * width + c);
#pragma unroll
    for (int j = 0; j < ROWS_AHEAD; ++j)
      if (j0 + j < top) v = j0 + j ? v + r[j] : r[j];
  }
  *to = old + v;
}

}  // namespace

int kx_expert_route_launch(bool f32, KxExpertArgs &e, const KxExpertSlots &s, int tokens, const KxMat &in, const KxMat &out, hipStream_t st) {
  KX_REQUIRE(e.experts > 0 && e.experts <= KX_MAX_EXPERTS && e.top > 0 && e.top <= e.experts && e.top <= KX_MAX_TOP && tokens > 0 && e.logits && e.bias,
             "experts: %d of %d for %d tokens", e.top, e.experts, tokens);
  e.ids = s.ids; e.weights = s.weights;
  e.tile_slots = kx_expert_tile(f32, tokens, e.top, e.experts, in, out, std::max(1, kx_device_cus()));
  e.max_tiles = kx_expert_tiles(tokens, e.top, e.experts, e.tile_slots);
  e.tiles = s.tiles; e.n_tiles = s.n_tiles; e.slot_weight = s.slot_weight;
  if (tokens <= BUCKET_WAVES) {
    hipLaunchKernelGGL(bucket_k<true>, dim3(1), dim3(KX_MAX_EXPERTS), 0, st, e, s, tokens);
    KX_LAUNCH_CHECK();
    return KX_OK;
  }
  hipLaunchKernelGGL(route_k, dim3(kx_cdiv(tokens, 4)), dim3(256), 0, st, e, tokens);
  KX_LAUNCH_CHECK();
  hipLaunchKernelGGL(bucket_k<false>, dim3(1), dim3(KX_MAX_EXPERTS), 0, st, e, s, tokens);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

int kx_expert_combine_launch(const KxExpertSlots &s, const float *y, float *x, int tokens, int top, int width, hipStream_t st) {
  if (width % 4 == 0 && ((uintptr_t)x | (uintptr_t)y) % 16 == 0) hipLaunchKernelGGL(combine_k<4>, dim3(tokens, kx_cdiv(width, 1024)), dim3(256), 0, st, s, y, x, top, width);
  else hipLaunchKernelGGL(combine_k<1>, dim3(tokens, kx_cdiv(width, 256)), dim3(256), 0, st, s, y, x, top, width);
  KX_LAUNCH_CHECK();
  return KX_OK;
}

int kx_expert_ff_launch(bool f32, const KxExpertFf &f, int tokens, hipStream_t st) {
  KxLinArgs gu = f.gu;
  gu.model_mb = std::max(f.gu.model_mb, kxonce::megabytes((size_t)f.e.experts * (f.gu_stride + f.down_stride) * (f32 ? 4 : 2)));  // these at the least
  gu.epi = KX_LIN_GLU;
  gu.mid = f.mid;
  gu.mid_ld = f.down.ld;
  KxExpertArgs e = f.e, eo = f.e;
  e.ids = eo.ids = f.s.ids;
  e.weights = eo.weights = f.s.weights;
  e.stride = f.gu_stride;
  eo.stride = f.down_stride; eo.w = f.down.w; eo.ld = f.down.ld; eo.mid = f.mid; eo.mid_ld = f.down.ld;
  if (kx_expert_small(f32, gu, f.out, eo, tokens)) {
    KX_DO(kx_expert_in_launch(f32, gu, e, st));
    return kx_expert_out_launch(f32, f.out, eo, st);
  }
  const void *h = f.h;
  if (!h) {
    KX_DO(kx_rows_launch(f32, gu.row, tokens, f.h_buf, gu.m.ld, st));
    h = f.h_buf;
  }
  KX_DO(kx_expert_route_launch(f32, e, f.s, tokens, gu.m, f.down, st));
  e.gather = f.s.gather;
  KX_DO(kx_expert_gemm_launch(f32, gu, e, h, gu.m.ld, st));
  KX_DO(kx_linear_launch(f32, f.out, f.row_buf, st));
  KxLinArgs down;
  down.m = f.down;
  down.tokens = tokens;
  down.model_mb = gu.model_mb;
  down.row.cols = f.down.cols;
  down.out = f.y;
  down.out_ld = f.down.rows;
  e.gather = nullptr;
  e.stride = f.down_stride;
  KX_DO(kx_expert_gemm_launch(f32, down, e, f.mid, f.down.ld, st));
  return kx_expert_combine_launch(f.s, f.y, f.out.streams, tokens, e.top, f.down.rows, st);
}
