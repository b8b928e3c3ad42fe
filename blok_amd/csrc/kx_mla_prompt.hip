// kx_mla_prompt.hip -- attention of a prefill step of several positions per sequence: keys and values of the whole context
// expanded from the latent cache per head, causal attention on the matrix cores (kx_window.hip) over them.
//
// The counterpart of tiled_attention (src/kimi_exec.cu:692-716) on the expanded keys and values that the reference keeps (:197,
// split_kv_k :364-370).  The decode form on the latent rows (kx_mla.hip) costs 2 x 1088 products per query, key and head and
// reads every cached row once per position of the step; expanded they are 2 x 320, and 128 positions of a step share each
// tile of keys.  What it costs is one product of the context with W_UK and W_UV per step, 2 x 512 x (128 + 128) per cached
// row and head, so that a short step behind a long context is better off with the decode form (kx_mla_prompt_fits).
// 64 heads, 2048 + 952 positions of one sequence: 3.25 ms a layer in the decode form (with absorb, merge and W_UV), 0.94 ms here.
#include <algorithm>
#include "kx_attn_parts.h"
#include "kx_common.h"
#include "kx_dense.h"
#include "kx_linear.h"
#include "kx_mla.h"
#include "kx_window.h"

namespace {

// token blockIdx.x: its cache row (kv_a norm, RoPE of the shared key, :817-824) and RoPE of its queries, in place
__global__ void __launch_bounds__(256) prompt_prep_k(KxMlaPromptArgs a) {
  __shared__ float ws[4];
  const int t = blockIdx.x, i = t / a.seqs, b = t - i * a.seqs, half = a.rope >> 1;
  const uint16_t *rr = a.rope_row + (size_t)i * a.rope;
  kxa::kv_finish_block(a.kva + (size_t)t * a.kva_stride, a.w_kv_ln, rr, a.cache + b * a.seq_stride + (size_t)(a.pos + i) * (a.kv_rank + a.rope), a.kv_rank, a.rope,
                       a.eps, ws);
  uint16_t *q = a.q + (size_t)t * a.heads * (a.nope + a.rope) + a.nope;
  // a wave has whole heads (half is a power of two up to 64): their pairs are read before any of them is written
  for (int x = threadIdx.x; x < a.heads * half; x += 256) {
    const int h = x / half, p = x - h * half;
    uint16_t *qh = q + (size_t)h * (a.nope + a.rope);
    const uint32_t two = *(const uint32_t *)(qh + 2 * p);
    float lo, hi;
    kxa::rope_pair(kx_bits_f32(two << 16), kx_bits_f32(two & 0xffff0000u), kx_bf16_f32(rr[p]), kx_bf16_f32(rr[half + p]), lo, hi);
    qh[p] = kx_bf16_rne(lo);
    qh[half + p] = kx_bf16_rne(hi);
  }
}

// the shared part of the keys (RoPE'd, 16-byte pieces) behind each head's own; zeros behind the last value, which meet weights of
// zero: what lies there may not be finite, and the attention would make its sums twice
__global__ void __launch_bounds__(256) share_key_k(const uint16_t *__restrict__ cache, size_t seq_stride, int row, int kv_rank, int pieces, uint16_t *__restrict__ k, int n,
                                                   int heads, int cap, int ld, int at, uint16_t *__restrict__ v, int dv) {
  const size_t total = (size_t)n * heads * pieces;
  const int b = blockIdx.y;
  for (size_t x = (size_t)blockIdx.x * 256 + threadIdx.x; x < total; x += (size_t)gridDim.x * 256) {
    const int p = (int)(x % pieces);
    const size_t y = x / pieces;
    const int t = (int)(y % n), h = (int)(y / n);
    *(uint4 *)(k + ((size_t)(b * heads + h) * cap + t) * ld + at + p * 8) = *(const uint4 *)(cache + b * seq_stride + (size_t)t * row + kv_rank + p * 8);
  }
  const int tail = (cap - n) * (dv / 8);
  for (int x = blockIdx.x * 256 + threadIdx.x; x < tail * heads; x += gridDim.x * 256)
    *(uint4 *)(v + ((size_t)(b * heads + x / tail) * cap + n) * dv + (size_t)(x % tail) * 8) = uint4{0, 0, 0, 0};
}

// How the heads and sequences of a launch take turns with the room for their keys and values.
struct Turns {
  int heads, seqs;  // of a turn
};
Turns turns_of(const kx_config *c, int seqs, int context, size_t expand_bytes) {
  const size_t head = (size_t)kx_pad(context, 64) * (c->qk_nope + c->qk_rope + c->v_head) * 2;  // bytes
  const int most = (int)std::min<size_t>(expand_bytes / head, (size_t)c->heads * seqs);
  if (most == 0) return {0, 0};
  const int heads = kx_cdiv(c->heads, kx_cdiv(c->heads, std::min(most, c->heads)));
  return {heads, heads == c->heads ? most / heads : 1};
}

}  // namespace

// The shorter of two estimates, in us per layer, measured with 8 to 128 heads, 1 to 16 sequences and contexts of up to 60000 positions.  The
// decode form does its work per position, cached row and head (with 64 heads, on the matrix cores, per position and row) and
// some per position; expanded, a cached row costs its share of the product per head and sequence, and of the way of a workgroup
// through all keys, alone on its CU, as often as there are more of them than CUs.  Figures, decode form / this one: 64 heads, 96
// positions behind 1000 377 / 303, behind 4000 418 / 542, behind 16000 609 / 1499; 256 positions 433 / 314, 584 / 584, 1109 / 1521; 512
// positions behind 16000 2080 / 1572, behind 60000, in two turns, 6117 / 7417; 8 heads, 33 positions behind 16000 540 / 829, of 4 sequences
// behind 8000 916 / 675.  With no context the decode form is behind from 96 positions on (16 where heads is not 64) at the latest.
bool kx_mla_prompt_fits(const kx_config *c, int seqs, int positions, int pos, size_t expand_bytes) {
  const int half = c->qk_rope / 2;
  if ((c->qk_nope + c->qk_rope) % 32 || c->v_head % 32 || c->qk_nope % 32 || c->qk_nope + c->qk_rope > 256 || c->v_head > 256 || half > 64 || (half & (half - 1)) || c->kv_rank % 128) return false;
  const bool matrix_cores = c->heads == 64;
  if (positions < (matrix_cores ? 96 : 16)) return false;
  if (expand_bytes < (size_t)kx_pad(c->max_context, 64) * (c->qk_nope + c->qk_rope + c->v_head) * 2) return false;
  const Turns t = turns_of(c, seqs, pos + positions, expand_bytes);
  const int cus = std::max(1, kx_device_cus());
  const double trips = (double)kx_cdiv(c->heads, t.heads) * kx_cdiv(seqs, t.seqs) * kx_cdiv(t.heads * t.seqs * kx_cdiv(positions, 128), cus);
  const double expanded = (pos + positions) * (0.041 * trips + 0.00063 * c->heads * seqs);
  const double decode = (double)seqs * positions * ((matrix_cores ? 0.00017 : 0.00009 * c->heads) * (pos + positions / 2) + (matrix_cores ? 0.8 : 0.4));
  return expanded < decode;
}

int kx_mla_prompt_launch(const kx_config *c, const KxMlaPromptArgs &a, const KxDenseArgs &split, hipStream_t st) {
  const int n = a.pos + a.positions, cap = kx_pad(n, 64), dk = a.nope + a.rope, dv = c->v_head;
  hipLaunchKernelGGL(prompt_prep_k, dim3(a.positions * a.seqs), dim3(256), 0, st, a);
  KX_LAUNCH_CHECK();
  const Turns turn = turns_of(c, a.seqs, n, a.expand_bytes);
  KX_REQUIRE(turn.heads > 0, "kx_mla: no room for the keys of %d positions", n);
  const int hg = turn.heads, bg = turn.seqs;
  float rs, ms;
  kx_softmax_scale(c, &rs, &ms);
  for (int b0 = 0; b0 < a.seqs; b0 += bg)
    for (int h0 = 0; h0 < a.heads; h0 += hg) {
      const int nb = std::min(bg, a.seqs - b0), nh = std::min(hg, a.heads - h0);
      uint16_t *k = (uint16_t *)a.expand, *v = k + (size_t)nb * nh * cap * dk;
      const uint16_t *rows = a.cache + b0 * a.seq_stride;
      KxDenseArgs d = split;
      d.w0 = a.kvb + (size_t)h0 * (a.nope + dv) * a.kv_rank; d.w1 = nullptr;
      d.x = rows; d.x_stride = a.kv_rank + a.rope;
      d.out = k; d.out_v = v; d.mode = KX_GG_KV; d.out_stride = 0;
      d.tokens = nb * n; d.rows = nh * (a.nope + dv); d.cols = a.kv_rank;
      d.seq = n; d.seq_jump = (int)(a.seq_stride / (a.kv_rank + a.rope)); d.heads = nh; d.k_dim = a.nope; d.v_dim = dv; d.cap = cap; d.k_ld = dk; d.v_ld = dv;
      int rc = kx_dense_gemm_launch(d, st);
      if (rc) return rc;
      const size_t pieces = (size_t)n * nh * (a.rope / 8);
      hipLaunchKernelGGL(share_key_k, dim3((unsigned)std::min<size_t>((pieces + 255) / 256, 4096), nb), dim3(256), 0, st, rows, a.seq_stride, a.kv_rank + a.rope, a.kv_rank,
                         a.rope / 8, k, n, nh, cap, dk, a.nope, v, dv);
      KX_LAUNCH_CHECK();
      KxWindowArgs w;
      w.s.heads = w.s.kv_heads = nh; w.s.dim = dk; w.s.vdim = dv; w.s.scale = rs * ms * ms;
      w.c.k = k; w.c.v = v; w.c.cap = cap; w.c.dp = dk; w.c.vp = dv;
      w.batch = nb; w.positions = a.positions; w.pos = a.pos;
      w.tok_batch = a.seqs; w.q_ld = (size_t)a.heads * dk;
      w.q = a.q + (size_t)b0 * w.q_ld + (size_t)h0 * dk;
      w.out_ld = a.heads * dv;
      w.out = a.out + (size_t)b0 * w.out_ld + (size_t)h0 * dv;
      if ((rc = kx_window_attend(false, w, st))) return rc;
    }
  return KX_OK;
}
