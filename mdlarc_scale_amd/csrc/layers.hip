// Whole layer stacks from one host call: the launches of every layer of a prompt or of a decode
// step, in the order the per-kernel entries are called one by one.  A layer is five to seven
// launches of 5 to 25 us at one to sixteen rows, and a call from Python cost as much: its argument
// checks, pointers and the foreign call took some 7 us.  Here a launch costs what the runtime
// takes.  With the one range check below in place of four reductions read back one by one, a
// decode call of 4 layers and 16 rows went from 500 to 290 us (213 of kernels) and a forward pass of
// 523 tokens from 483 to 393 (347).  Every check of the entries stays, and each entry still
// chooses its own kernel.
#include <climits>

#include "common.h"

using namespace mdl;

namespace mdl {

namespace {

// The part after the attention: out projection and residual, ln2, SwiGLU MLP and residual.
int mlp(const mdl_stack& s, const mdl_layer& l, bool prompt, void* st) {
  const int d = s.n_heads * kHeadDim, m = s.rows;
  int rc;
  if (prompt && s.f32) {
    rc = mdl_prefill_gemm_split_residual_f32w(s.attn, l.out, l.out_lo, s.x, nullptr, m, d, d, st);
    if (rc == MDL_OK)
      rc = mdl_prefill_gemm_norm_swiglu_f32w(s.x, l.ln2, s.eps, l.gu, l.gu_lo, l.b_gate, l.b_up,
                                             s.h, m, s.d_ff, d, st);
    if (rc == MDL_OK)
      rc = mdl_prefill_gemm_split_residual_f32w(s.h, l.down, l.down_lo, s.x, l.b_down, m, d,
                                                s.d_ff, st);
  } else if (prompt) {
    rc = mdl_prefill_gemm_split_residual(s.attn, 0, MDL_LAYOUT_TILES, 2, l.out, s.x, nullptr, m, d,
                                         d, st);
    if (rc == MDL_OK)
      rc = mdl_prefill_gemm_norm_swiglu(s.x, l.ln2, s.eps, s.gate_up_parts, l.gu, l.b_gate, l.b_up,
                                        s.h, s.down_parts, m, s.d_ff, d, st);
    if (rc == MDL_OK)
      rc = mdl_prefill_gemm_split_residual(s.h, 0, MDL_LAYOUT_TILES, s.down_parts, l.down, s.x,
                                           l.b_down, m, d, s.d_ff, st);
  } else {
    rc = mdl_gemm_split_residual(s.attn, l.out, l.out_lo, s.x, nullptr, m, d, d, 0, st);
    if (rc == MDL_OK)
      rc = mdl_gemm_norm_swiglu(s.x, l.ln2, s.eps, l.gu, l.gu_lo, l.b_gate, l.b_up, s.h, m, s.d_ff,
                                d, 0, st);
    if (rc == MDL_OK)
      rc = mdl_gemm_split_residual(s.h, l.down, l.down_lo, s.x, l.b_down, m, d, s.d_ff, 0, st);
  }
  return rc;
}

int prompt_layer(const mdl_stack& s, const mdl_layer& l, void* st) {
  const int ld = 3 * s.n_heads * kHeadDim;
  int rc;
  if (s.f32) {
    rc = mdl_prefill_gemm_norm_qkv_f32w(
        s.x, l.ln1, s.eps, l.qkv, l.qkv_lo, s.rows, s.n_heads, s.qkv, ld, s.rstd, s.pos, s.rope_tab,
        s.max_x, s.max_y, s.max_z, s.px, s.py, s.pz, s.q_scale, static_cast<float*>(s.q),
        static_cast<float*>(l.k_cache), static_cast<float*>(l.v_cache), l.slots, s.batch, s.seq,
        s.token_row, s.token_slot, st);
    if (rc == MDL_OK)
      rc = mdl_attn_prefill_f32(static_cast<const float*>(s.q),
                                static_cast<const float*>(l.k_cache),
                                static_cast<const float*>(l.v_cache), s.batch, s.seq, s.n_heads,
                                kHeadDim, l.slots, s.mask, s.kv_start, s.q_offset, s.causal, s.attn,
                                MDL_LAYOUT_TILES, st);
  } else {
    uint16_t* q = static_cast<uint16_t*>(s.q);
    uint16_t* k = static_cast<uint16_t*>(l.k_cache);
    uint16_t* v = static_cast<uint16_t*>(l.v_cache);
    rc = mdl_prefill_gemm_norm_qkv(s.x, l.ln1, s.eps, l.qkv, s.rows, s.n_heads, s.rstd, s.qkv, ld,
                                   s.lead, s.kv_start, s.pos, s.rope_tab, s.max_x, s.max_y,
                                   s.max_z, s.px, s.py, s.pz, s.q_scale, q, k, v, l.slots, s.batch,
                                   s.seq, s.token_row, s.token_slot, st);
    if (rc == MDL_OK)
      rc = s.q_offset
               ? mdl_attn_prefill_packed(q, k, v, s.batch, s.seq, s.n_heads, kHeadDim, l.slots,
                                         s.mask, s.row_holes, s.kv_start, s.q_offset, s.causal,
                                         s.attn, MDL_LAYOUT_TILES, st)
               : mdl_attn_prefill(q, k, v, s.batch, s.seq, s.n_heads, kHeadDim, l.slots, s.mask,
                                  s.row_holes, s.kv_start, s.causal, s.attn, MDL_LAYOUT_TILES, st);
    if (rc == MDL_OK && s.causal)
      rc = mdl_attn_prefill_lead(s.qkv, ld, s.rstd, s.pos, s.rope_tab, s.max_x, s.max_y, s.max_z,
                                 s.px, s.py, s.pz, s.lead_scale, s.batch, s.seq, s.n_heads,
                                 kHeadDim, s.mask, s.kv_start, s.q_offset, s.attn,
                                 MDL_LAYOUT_TILES, st);
  }
  return rc == MDL_OK ? mlp(s, l, true, st) : rc;
}

int decode_layer(const mdl_stack& s, const mdl_layer& l, void* st) {
  int rc;
  if (s.f32) {
    float* q = static_cast<float*>(s.q);
    float* k = static_cast<float*>(l.k_cache);
    float* v = static_cast<float*>(l.v_cache);
    rc = mdl_gemm_norm_qkv_f32w(s.x, l.ln1, s.eps, l.qkv, l.qkv_lo, s.rows, s.n_heads, nullptr,
                                s.pos, s.rope_tab, s.max_x, s.max_y, s.max_z, s.px, s.py, s.pz,
                                s.q_scale, q, k, v, l.slots, 0, s.slot_dev, 0, st);
    if (rc == MDL_OK)
      rc = mdl_attn_decode_f32(q, k, v, s.batch, s.n_heads, kHeadDim, l.slots, s.mask, s.seq,
                               s.kv_start, 0, s.slot_dev, s.ws, s.ws_bytes, s.split_len, s.attn,
                               MDL_LAYOUT_TILES, st);
  } else {
    uint16_t* q = static_cast<uint16_t*>(s.q);
    uint16_t* k = static_cast<uint16_t*>(l.k_cache);
    uint16_t* v = static_cast<uint16_t*>(l.v_cache);
    rc = mdl_gemm_norm_qkv(s.x, l.ln1, s.eps, l.qkv, s.rows, s.n_heads, nullptr, s.pos, s.rope_tab,
                           s.max_x, s.max_y, s.max_z, s.px, s.py, s.pz, s.q_scale, q, k, v,
                           l.slots, 0, s.slot_dev, 0, st);
    if (rc == MDL_OK)
      rc = mdl_attn_decode(q, k, v, s.batch, s.n_heads, kHeadDim, l.slots, s.mask, s.seq,
                           s.row_holes, s.kv_start, s.row_order, 0, s.slot_dev, s.ws, s.ws_bytes,
                           s.split_len, s.attn, MDL_LAYOUT_TILES, st);
  }
  return rc == MDL_OK ? mlp(s, l, false, st) : rc;
}

// What the entries of a layer cannot see: they take the slots as an int, an absent low part as a
// bf16 weight and, at decode, the projections' rows, the attention's batch and the slot each by itself.
int check_stack(const mdl_stack* s, bool decode) {
  if (!s || (!s->layers && s->n_layers > 0)) return MDL_ERR_NULL;
  if (s->n_layers < 0 || s->n_heads <= 0 || s->n_heads > (1 << 16)) return MDL_ERR_SHAPE;
  if (decode && s->rows != s->batch) return MDL_ERR_SHAPE;
  if (decode && !s->slot_dev) return MDL_ERR_NULL;
  for (int i = 0; i < s->n_layers; ++i) {
    const mdl_layer& l = s->layers[i];
    if (l.slots < 1 || l.slots > INT_MAX) return MDL_ERR_SHAPE;
    if (s->f32 && (!l.qkv_lo || !l.out_lo || !l.gu_lo || !l.down_lo)) return MDL_ERR_NULL;
  }
  return MDL_OK;
}

// min and max of two int64 lists (a call's token and example ids), one pair per block
__global__ __launch_bounds__(1024) void id_range_kernel(const int64_t* __restrict__ a, int64_t na,
                                                        const int64_t* __restrict__ b, int64_t nb,
                                                        int64_t* __restrict__ out) {
  __shared__ int64_t red[4][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int list = 0; list < 2; ++list) {
    const int64_t* v = list ? b : a;
    const int64_t n = list ? nb : na;
    int64_t lo = INT64_MAX, hi = INT64_MIN;
    for (int64_t i = blockIdx.x * 1024ll + threadIdx.x; i < n; i += 1024ll * gridDim.x) {
      const int64_t x = v[i];
      lo = x < lo ? x : lo;
      hi = x > hi ? x : hi;
    }
    for (int o = 32; o > 0; o >>= 1) {
      const int64_t l2 = __shfl_xor(lo, o, kWave), h2 = __shfl_xor(hi, o, kWave);
      lo = l2 < lo ? l2 : lo;
      hi = h2 > hi ? h2 : hi;
    }
    if (lane == 0) {
      red[2 * list][wave] = lo;
      red[2 * list + 1][wave] = hi;
    }
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    const int64_t* r = red[threadIdx.x];
    int64_t best = r[0];
    for (int w = 1; w < 16; ++w)
      best = (threadIdx.x & 1) ? (r[w] > best ? r[w] : best) : (r[w] < best ? r[w] : best);
    out[threadIdx.x * gridDim.x + blockIdx.x] = best;
  }
}

}  // namespace

}  // namespace mdl

extern "C" int mdl_prompt_layers(const mdl_stack* stack, void* stream) {
  int rc = check_stack(stack, false);
  for (int i = 0; rc == MDL_OK && i < stack->n_layers; ++i)
    rc = prompt_layer(*stack, stack->layers[i], stream);
  return rc;
}

extern "C" int mdl_decode_layers(const mdl_stack* stack, void* stream) {
  int rc = check_stack(stack, true);
  for (int i = 0; rc == MDL_OK && i < stack->n_layers; ++i)
    rc = decode_layer(*stack, stack->layers[i], stream);
  return rc;
}

extern "C" int mdl_id_range(const int64_t* ids, int64_t n_ids, const int64_t* example_ids,
                            int64_t n_examples, int blocks, int64_t* out, void* stream) {
  if (!out || (n_ids > 0 && !ids) || (n_examples > 0 && !example_ids)) return MDL_ERR_NULL;
  if (n_ids < 0 || n_examples < 0 || blocks < 1 || blocks > 1024) return MDL_ERR_SHAPE;
  hipLaunchKernelGGL(id_range_kernel, dim3(blocks), dim3(1024), 0,
                     static_cast<hipStream_t>(stream), ids, n_ids, example_ids, n_examples, out);
  return launch_status();
}
