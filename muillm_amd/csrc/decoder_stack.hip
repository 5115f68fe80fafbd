// One call for the decoder layers of a decode step.
//
// The reference walks its layers from C++ only under tensor parallelism
// (csrc/modules/parallel_decoder_stack.cpp; per-layer order in
// csrc/modules/parallel_decoder_module.cpp:22-62: fused-norm QKV, attention with RoPE and
// cache write, o_proj + residual, fused-norm gate/up + SiLU, down + residual); on one GPU it
// goes through its Python modules (muillm/modules/decoder/decoder.py:130-165). Here the same
// order is enqueued by one C call, which removes the per-launch host work of an interpreter
// loop (about 160 launches per token) when the step is not replayed from a HIP graph. Each
// projection takes 16-bit weights or int8 codes, the latter with per-channel scales or in the
// reference's group-wise (scale, min) format (muillm/modules/quantized/int8linear.py:279-293,
// int8gateupdownmlp.py, muillm/quantization/rtnquantizer.py:49-88).
#include "skinny.cuh"

using namespace mui;

namespace {

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct StackWorkspace {
  char* h_a;      // [batch, hidden]   o_proj output (residual stream after attention)
  char* h_b;      // [batch, hidden]   layer output
  char* qkv;      // [batch, (Hq + 2 Hkv) * D]
  char* attn;     // [batch, Hq * D]
  char* mid;      // [batch, intermediate]
  char* scratch;  // flash-decoding partials
  size_t total;
};

StackWorkspace carve(const mui_decoder_stack_t* m, int batch, int n_splits, char* base) {
  StackWorkspace w;
  const size_t e = 2;  // 16-bit activations
  const size_t hid = align256((size_t)batch * m->hidden * e);
  const size_t qkv = align256((size_t)batch * (m->n_q_heads + 2 * m->n_kv_heads) * m->head_dim * e);
  const size_t att = align256((size_t)batch * m->n_q_heads * m->head_dim * e);
  const size_t mid = align256((size_t)batch * m->intermediate * e);
  const size_t scr = align256(mui_flash_decode_scratch_bytes(batch, m->n_q_heads, m->head_dim, n_splits));
  size_t off = 0;
  w.h_a = base + off; off += hid;
  w.h_b = base + off; off += hid;
  w.qkv = base + off; off += qkv;
  w.attn = base + off; off += att;
  w.mid = base + off; off += mid;
  w.scratch = base + off; off += scr;
  w.total = off;
  return w;
}

}  // namespace

extern "C" size_t mui_decoder_stack_workspace_bytes(const mui_decoder_stack_t* m, int batch, int n_splits) {
  if (!m || batch < 1 || n_splits < 1) return 0;
  return carve(m, batch, n_splits, nullptr).total;
}

extern "C" int mui_decoder_stack_step(mui_stream_t stream, const mui_decoder_stack_t* m, int batch,
                                      const void* hidden_in, void* hidden_out,
                                      const int64_t* position_ids, long position_batch_stride,
                                      const int64_t* cache_position, int seq_len, const void* mask,
                                      long mask_batch_stride, int n_splits, void* workspace) {
  MUI_CHECK_ARG(m && m->layers && m->n_layers > 0 && hidden_in && hidden_out && workspace);
  MUI_CHECK_ARG(batch >= 1 && batch <= MUI_MAX_TOKENS && n_splits >= 1);
  MUI_CHECK_ARG(position_ids && cache_position);
  MUI_CHECK_ARG(((uintptr_t)workspace & 255u) == 0);
  const StackWorkspace w = carve(m, batch, n_splits, (char*)workspace);
  const int qd = m->n_q_heads * m->head_dim, kvd = m->n_kv_heads * m->head_dim;
  const int qkv_n = qd + 2 * kvd;
  const char* h = (const char*)hidden_in;  // residual stream entering the layer
  for (int l = 0; l < m->n_layers; ++l) {
    const mui_decoder_layer_t& L = m->layers[l];
    char* out = (l + 1 == m->n_layers) ? (char*)hidden_out : w.h_b;
    const int gs = L.int8_group_size_shift;  // 0: per-channel scales; else the reference's group format
    if (gs < 0) return MUI_ERR_INVALID_ARG;
    int st = !L.qkv_scales
                 ? mui_linear(stream, m->dtype, L.qkv_weight, L.qkv_pitch, h, L.input_norm, m->norm_eps, nullptr,
                              nullptr, nullptr, w.qkv, qkv_n, m->hidden, batch)
             : gs ? mui_int8_group_linear(stream, m->dtype, L.qkv_weight, L.qkv_pitch, L.qkv_scales, gs, h,
                                          L.input_norm, m->norm_eps, nullptr, nullptr, w.qkv, qkv_n, m->hidden,
                                          batch)
                  : mui_int8_linear(stream, m->dtype, L.qkv_weight, L.qkv_pitch, L.qkv_scales, h, L.input_norm,
                                    m->norm_eps, nullptr, nullptr, w.qkv, qkv_n, m->hidden, batch);
    if (st != MUI_OK) return st;
    const char* q = w.qkv;
    // the attention launch is told what follows it: at short context its idle workgroups fetch the
    // o_proj matrix on chip while the few busy ones wait on latency
    const int o_bits = L.o_scales ? 8 : 16;
    const long o_pitch_bytes = L.o_pitch * (o_bits / 8);
    const int o_slab = batch == 1 ? mui_linear_row_group_bytes(o_bits, qd, o_pitch_bytes) : 0;
    const size_t o_bytes = o_slab > 0 ? (size_t)m->hidden * (size_t)o_pitch_bytes : 0;
    st = mui_attn_decode_fused_warm(stream, m->dtype, q, qkv_n, q + (size_t)qd * 2, qkv_n,
                                    q + (size_t)(qd + kvd) * 2, qkv_n, m->cos_table, m->sin_table, (int)m->rope_row_stride, (int)m->rope_rows,
                                    position_ids, position_batch_stride, cache_position, seq_len, L.k_cache,
                                    L.v_cache, m->cache_batch_stride, m->cache_head_stride, m->cache_token_stride,
                                    mask, mask_batch_stride, nullptr, w.scratch, n_splits, w.attn, batch,
                                    m->n_q_heads, m->n_kv_heads, m->head_dim, m->max_cache_len,
                                    o_bytes ? L.o_weight : nullptr, o_bytes, o_slab);
    if (st != MUI_OK) return st;
    st = !L.o_scales ? mui_linear(stream, m->dtype, L.o_weight, L.o_pitch, w.attn, nullptr, 0.f, nullptr, nullptr, h,
                                  w.h_a, m->hidden, qd, batch)
         : gs ? mui_int8_group_linear(stream, m->dtype, L.o_weight, L.o_pitch, L.o_scales, gs, w.attn, nullptr, 0.f,
                                      nullptr, h, w.h_a, m->hidden, qd, batch)
              : mui_int8_linear(stream, m->dtype, L.o_weight, L.o_pitch, L.o_scales, w.attn, nullptr, 0.f, nullptr, h,
                                w.h_a, m->hidden, qd, batch);
    if (st != MUI_OK) return st;
    if ((L.gate_scales == nullptr) != (L.up_scales == nullptr)) return MUI_ERR_INVALID_ARG;
    st = !L.gate_scales
             ? mui_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch, w.h_a, L.post_norm,
                               m->norm_eps, w.mid, m->intermediate, m->hidden, batch)
         : gs ? mui_int8_group_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch,
                                           L.gate_scales, L.up_scales, L.gateup_scale_stride, gs, w.h_a,
                                           L.post_norm, m->norm_eps, w.mid, m->intermediate, m->hidden, batch)
              : mui_int8_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch, L.gate_scales,
                                     L.up_scales, L.gateup_scale_stride, w.h_a, L.post_norm, m->norm_eps, w.mid,
                                     m->intermediate, m->hidden, batch);
    if (st != MUI_OK) return st;
    st = !L.down_scales ? mui_linear(stream, m->dtype, L.down_weight, L.down_pitch, w.mid, nullptr, 0.f, nullptr,
                                     nullptr, w.h_a, out, m->hidden, m->intermediate, batch)
         : gs ? mui_int8_group_linear(stream, m->dtype, L.down_weight, L.down_pitch, L.down_scales, gs, w.mid,
                                      nullptr, 0.f, nullptr, w.h_a, out, m->hidden, m->intermediate, batch)
              : mui_int8_linear(stream, m->dtype, L.down_weight, L.down_pitch, L.down_scales, w.mid, nullptr, 0.f,
                                nullptr, w.h_a, out, m->hidden, m->intermediate, batch);
    if (st != MUI_OK) return st;
    h = out;
  }
  return MUI_OK;
}

// ---------------------------------------------------------------------------------------
// Any number of rows: prompts, and steps of more batch rows than the decode kernels take
// ---------------------------------------------------------------------------------------
namespace {

struct PromptWorkspace {
  char *h_a, *h_b;  // [rows, hidden]  residual stream
  char* normed;     // [rows, hidden]  the next linear's input
  char *qkv, *q_rot, *attn, *scratch;  // up to the output projection
  char* spread;  // [batch * tokens, .] qkv with the padding, where the rows leave it out
  char* mid;                           // [rows, intermediate], in the same place
  size_t total;
};

// real: rows that are no padding (batch * tokens: all of them)
PromptWorkspace carve_rows(const mui_decoder_stack_t* m, int batch, int tokens, int n_splits, char* base, int real) {
  PromptWorkspace w;
  const size_t all = (size_t)batch * tokens, rows = real, e = 2;
  const size_t hid = align256(rows * m->hidden * e), att = align256(all * m->n_q_heads * m->head_dim * e);
  const size_t qkv = align256(rows * (m->n_q_heads + 2 * m->n_kv_heads) * m->head_dim * e), mid = align256(rows * m->intermediate * e);
  const size_t scr = tokens == 1 ? align256(mui_flash_decode_scratch_bytes(batch, m->n_q_heads, m->head_dim, n_splits)) : 0;
  w.h_a = base;
  w.h_b = w.h_a + hid;
  w.normed = w.h_b + hid;
  w.qkv = w.normed + hid;
  w.spread = w.qkv + qkv;
  w.q_rot = w.spread + (rows < all ? align256(all * (m->n_q_heads + 2 * m->n_kv_heads) * m->head_dim * e) : 0);
  w.attn = w.q_rot + (tokens == 1 ? 0 : att);
  w.scratch = w.attn + att;
  w.mid = w.qkv;  // (the output projection has read the rest when the gate and up products start)
  const size_t before = (size_t)(w.scratch - w.qkv) + scr;
  w.total = 3 * hid + (before > mid ? before : mid);
  return w;
}

}  // namespace

extern "C" size_t mui_decoder_stack_prompt_bytes(const mui_decoder_stack_t* m, int batch, int tokens, int n_splits) {
  if (!m || batch < 1 || tokens < 1 || n_splits < 1) return 0;
  return carve_rows(m, batch, tokens, n_splits, nullptr, batch * tokens).total;
}

// rows, slots (both or neither): the rows that are no padding -- hidden_in and hidden_out have `real` rows, number r of them token rows[r] of [batch, tokens] --,
// and every token's number among them, or -1
static int prompt_layers(mui_stream_t stream, const mui_decoder_stack_t* m, int batch, int tokens, int real, const int64_t* real_rows, const int64_t* slots,
                         const void* hidden_in, void* hidden_out, const int64_t* position_ids, long position_batch_stride, const int64_t* cache_position,
                         int seq_len, const void* mask, long mask_batch_stride, int n_splits, void* workspace, void* linear_workspace,
                         size_t linear_workspace_bytes) {
  MUI_CHECK_ARG(m && m->layers && m->n_layers > 0 && hidden_in && hidden_out && workspace);
  MUI_CHECK_ARG(batch >= 1 && tokens >= 1 && n_splits >= 1 && position_ids && cache_position);
  MUI_CHECK_ARG(((uintptr_t)workspace & 255u) == 0 && (long)batch * tokens <= (1L << 30));
  MUI_CHECK_ARG(tokens == 1 || seq_len >= tokens);
  MUI_CHECK_ARG(seq_len <= m->max_cache_len);  // (the prompt's attention takes no capacity: it reads seq_len rows of every head)
  const int rows = real;
  const PromptWorkspace w = carve_rows(m, batch, tokens, n_splits, (char*)workspace, real);
  const int hid = m->hidden, qd = m->n_q_heads * m->head_dim, kvd = m->n_kv_heads * m->head_dim, qkv_n = qd + 2 * kvd;
  const bool fused = rows <= MUI_MAX_TOKENS;  // the decode kernels take the norm in front of a linear; beyond, it is a launch of its own or rides behind the linear in front
  for (int l = 0; l < m->n_layers; ++l) {
    const mui_decoder_layer_t& L = m->layers[l];
    if (L.int8_group_size_shift < 0 || (L.gate_scales == nullptr) != (L.up_scales == nullptr)) return MUI_ERR_INVALID_ARG;
  }
  // y = W x (+ residual); next: the gain of the norm behind it, into w.normed
  auto linear = [&](const void* weight, long pitch, const void* scales, int shift, const void* x, const void* gain, const void* residual, void* y, int n,
                    int k, const void* next) -> int {
    int st;
    if (scales) {
      if (next && residual) {
        SkinnyParams q = {};
        q.w0 = weight; q.pitch = pitch; q.s0 = (const uint16_t*)scales; q.group_shift = shift;
        q.x = (const uint16_t*)x; q.residual = (const uint16_t*)residual; q.y = (uint16_t*)y; q.n = n; q.k = k; q.tokens = rows;
        q.workspace = linear_workspace; q.workspace_bytes = linear_workspace_bytes;
        st = gain ? MUI_ERR_UNSUPPORTED : launch_codes_norm((hipStream_t)stream, m->dtype, shift ? WF_U8_GROUP : WF_I8_CHANNEL, q, next, m->norm_eps, w.normed);
        if (st != MUI_ERR_UNSUPPORTED) return st;
      }
      st = shift ? mui_int8_group_linear_ws(stream, m->dtype, weight, pitch, scales, shift, x, gain, m->norm_eps, nullptr, residual, y, n, k, rows, linear_workspace,
                                            linear_workspace_bytes)
                 : mui_int8_linear_ws(stream, m->dtype, weight, pitch, scales, x, gain, m->norm_eps, nullptr, residual, y, n, k, rows, linear_workspace,
                                      linear_workspace_bytes);
    } else if (next) {
      return mui_linear_norm(stream, m->dtype, weight, pitch, x, nullptr, residual, next, m->norm_eps, y, w.normed, n, k, rows, linear_workspace,
                             linear_workspace_bytes);
    } else {
      st = mui_linear_ws(stream, m->dtype, weight, pitch, x, gain, m->norm_eps, nullptr, nullptr, residual, y, n, k, rows, linear_workspace,
                         linear_workspace_bytes);
    }
    if (st != MUI_OK || !next) return st;
    return mui_rmsnorm(stream, m->dtype, next, y, m->norm_eps, w.normed, rows, n);
  };
  const char* h = (const char*)hidden_in;  // residual stream entering the layer
  if (!fused) {
    const int st = mui_rmsnorm(stream, m->dtype, m->layers[0].input_norm, h, m->norm_eps, w.normed, rows, hid);
    if (st != MUI_OK) return st;
  }
  for (int l = 0; l < m->n_layers; ++l) {
    const mui_decoder_layer_t& L = m->layers[l];
    const bool last = l + 1 == m->n_layers;
    const int gs = L.int8_group_size_shift;
    char* out = last ? (char*)hidden_out : w.h_b;
    int st = linear(L.qkv_weight, L.qkv_pitch, L.qkv_scales, gs, fused ? h : w.normed, fused ? L.input_norm : nullptr, nullptr, w.qkv, qkv_n, hid, nullptr);
    if (st != MUI_OK) return st;
    if (slots) {
      st = mui_take_rows(stream, w.qkv, real, (size_t)qkv_n * 2, slots, w.spread, (long)batch * tokens);
      if (st != MUI_OK) return st;
    }
    const char *q = slots ? w.spread : w.qkv, *k = q + (size_t)qd * 2, *v = k + (size_t)kvd * 2;
    if (tokens == 1) {
      st = mui_attn_decode_fused_warm(stream, m->dtype, q, qkv_n, k, qkv_n, v, qkv_n, m->cos_table, m->sin_table, (int)m->rope_row_stride,
                                      (int)m->rope_rows, position_ids, position_batch_stride, cache_position, seq_len, L.k_cache, L.v_cache,
                                      m->cache_batch_stride, m->cache_head_stride, m->cache_token_stride, mask, mask_batch_stride, nullptr,
                                      w.scratch, n_splits, w.attn, batch, m->n_q_heads, m->n_kv_heads, m->head_dim, m->max_cache_len, nullptr, 0, 0);
    } else {
      const long tb = (long)tokens * qkv_n;
      st = mui_rope_kv_write(stream, m->dtype, q, tb, qkv_n, m->head_dim, k, tb, qkv_n, m->head_dim, v, tb, qkv_n, m->head_dim, m->cos_table,
                             m->sin_table, (int)m->rope_row_stride, (int)m->rope_rows, position_ids, position_batch_stride, cache_position, w.q_rot,
                             L.k_cache, L.v_cache, m->cache_batch_stride, m->cache_head_stride, m->cache_token_stride, batch, tokens, m->n_q_heads,
                             m->n_kv_heads, m->head_dim, m->max_cache_len);
      if (st != MUI_OK) return st;
      st = mask ? mui_prefill_attention_masked(stream, m->dtype, w.q_rot, L.k_cache, L.v_cache, m->cache_batch_stride, m->cache_head_stride,
                                               m->cache_token_stride, seq_len, seq_len - tokens, mask, mask_batch_stride, w.attn, batch, m->n_q_heads,
                                               m->n_kv_heads, tokens, m->head_dim)
                : mui_prefill_attention(stream, m->dtype, w.q_rot, L.k_cache, L.v_cache, m->cache_batch_stride, m->cache_head_stride,
                                        m->cache_token_stride, seq_len, seq_len - tokens, w.attn, batch, m->n_q_heads, m->n_kv_heads, tokens, m->head_dim);
    }
    if (st != MUI_OK) return st;
    const char* attended = w.attn;
    if (slots) {  // (the queries have been read)
      st = mui_take_rows(stream, w.attn, (long)batch * tokens, (size_t)qd * 2, real_rows, w.q_rot, real);
      if (st != MUI_OK) return st;
      attended = w.q_rot;
    }
    st = linear(L.o_weight, L.o_pitch, L.o_scales, gs, attended, nullptr, h, w.h_a, hid, qd, fused ? nullptr : L.post_norm);
    if (st != MUI_OK) return st;
    const void *mx = fused ? w.h_a : w.normed, *gain = fused ? L.post_norm : nullptr;
    st = !L.gate_scales ? mui_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch, mx, gain, m->norm_eps, w.mid, m->intermediate, hid, rows)
         : gs ? mui_int8_group_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch, L.gate_scales, L.up_scales,
                                           L.gateup_scale_stride, gs, mx, gain, m->norm_eps, w.mid, m->intermediate, hid, rows)
              : mui_int8_gateup_silu(stream, m->dtype, L.gate_weight, L.up_weight, L.gateup_pitch, L.gate_scales, L.up_scales, L.gateup_scale_stride, mx,
                                     gain, m->norm_eps, w.mid, m->intermediate, hid, rows);
    if (st != MUI_OK) return st;
    st = linear(L.down_weight, L.down_pitch, L.down_scales, gs, w.mid, nullptr, w.h_a, out, hid, m->intermediate,
                fused || last ? nullptr : m->layers[l + 1].input_norm);
    if (st != MUI_OK) return st;
    h = out;
  }
  return MUI_OK;
}

extern "C" int mui_decoder_stack_prompt(mui_stream_t stream, const mui_decoder_stack_t* m, int batch, int tokens, const void* hidden_in,
                                        void* hidden_out, const int64_t* position_ids, long position_batch_stride,
                                        const int64_t* cache_position, int seq_len, const void* mask, long mask_batch_stride, int n_splits,
                                        void* workspace, void* linear_workspace, size_t linear_workspace_bytes) {
  return prompt_layers(stream, m, batch, tokens, (int)((long)batch * tokens), nullptr, nullptr, hidden_in, hidden_out, position_ids,
                       position_batch_stride, cache_position, seq_len, mask, mask_batch_stride, n_splits, workspace, linear_workspace,
                       linear_workspace_bytes);
}

extern "C" size_t mui_decoder_stack_prompt_rows_bytes(const mui_decoder_stack_t* m, int batch, int tokens, int real_rows) {
  if (!m || batch < 1 || tokens < 1 || real_rows < 1 || real_rows > (long)batch * tokens) return 0;
  return carve_rows(m, batch, tokens, 1, nullptr, real_rows).total;
}

extern "C" int mui_decoder_stack_prompt_rows(mui_stream_t stream, const mui_decoder_stack_t* m, int batch, int tokens, int real_rows, const int64_t* rows,
                                             const int64_t* slots, const void* hidden_in, void* hidden_out, const int64_t* position_ids,
                                             long position_batch_stride, const int64_t* cache_position, int seq_len, const void* mask,
                                             long mask_batch_stride, void* workspace, void* linear_workspace, size_t linear_workspace_bytes) {
  MUI_CHECK_ARG(rows && slots && batch >= 1 && tokens > 1 && real_rows >= 1 && real_rows < (long)batch * tokens);
  return prompt_layers(stream, m, batch, tokens, real_rows, rows, slots, hidden_in, hidden_out, position_ids, position_batch_stride, cache_position, seq_len,
                       mask, mask_batch_stride, 1, workspace, linear_workspace, linear_workspace_bytes);
}
