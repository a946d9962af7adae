// The layer calls of one step, with the arguments that every layer shares in one host struct.
//
// No device code: each entry point forwards to the kernels' own (which check every argument), so a
// caller that makes 24 calls a step passes 4 to 8 pointers a call instead of converting 20 to 32
// arguments, most of them the same each time.
#include "mip_common.h"

using namespace mip;

extern "C" int mip_decode_step_append(const mip_decode_step* s, const void* k_new, const void* v_new, void* out,
                                      const void* q, void* k_cache, void* v_cache, void* stream) {
  if (!s) return MIP_EINVAL;
  return mip_paged_decode_append(k_new, v_new, s->k_stride_tok, s->k_stride_head, s->v_stride_tok, s->v_stride_head,
                                 s->slot_mapping, out, s->out_stride_b, s->out_stride_h, q, s->q_stride_b, s->q_stride_h,
                                 k_cache, v_cache, s->num_cache_blocks, s->block_tables, s->bt_stride, s->context_lens,
                                 s->batch, s->num_heads, s->num_kv_heads, s->head_dim, s->block_size,
                                 s->max_blocks_per_seq, s->scale, s->workspace, s->workspace_bytes, s->plan,
                                 s->plan_bytes, s->dtype, stream);
}

extern "C" int mip_decode_step_attend(const mip_decode_step* s, void* out, const void* q, const void* k_cache,
                                      const void* v_cache, void* stream) {
  if (!s) return MIP_EINVAL;
  return mip_paged_decode(out, s->out_stride_b, s->out_stride_h, q, s->q_stride_b, s->q_stride_h, k_cache, v_cache,
                          s->num_cache_blocks, s->block_tables, s->bt_stride, s->context_lens, s->batch, s->num_heads,
                          s->num_kv_heads, s->head_dim, s->block_size, s->max_blocks_per_seq, s->scale, s->workspace,
                          s->workspace_bytes, s->plan, s->plan_bytes, s->dtype, stream);
}

extern "C" int mip_rope_step_append(const mip_rope_step* s, void* q, void* k, const void* v, const void* cos,
                                    const void* sin, void* k_cache, void* v_cache, void* stream) {
  if (!s) return MIP_EINVAL;
  return mip_rope_kv_append(q, s->q_stride_tok, s->q_stride_head, k, s->k_stride_tok, s->k_stride_head, v,
                            s->v_stride_tok, s->v_stride_head, cos, sin, s->cs_stride_tok, k_cache, v_cache,
                            s->num_cache_blocks, s->slot_mapping, s->n_tokens, s->num_heads, s->num_kv_heads,
                            s->head_dim, s->block_size, s->dtype, stream);
}

extern "C" int mip_prefill_step_append(const mip_prefill_step* s, const void* k_new, const void* v_new, void* k_cache,
                                       void* v_cache, void* stream) {
  if (!s) return MIP_EINVAL;
  return mip_kv_append(k_new, v_new, s->k_stride_tok, s->k_stride_head, s->v_stride_tok, s->v_stride_head, k_cache,
                       v_cache, s->num_cache_blocks, s->slot_mapping, s->n_tokens, s->num_kv_heads, s->head_dim,
                       s->block_size, s->dtype, stream);
}

extern "C" int mip_prefill_step_attend(const mip_prefill_step* s, void* out, const void* q, const void* k_cache,
                                       const void* v_cache, void* stream) {
  if (!s) return MIP_EINVAL;
  return mip_paged_prefill(out, s->out_stride_tok, s->out_stride_head, q, s->q_stride_tok, s->q_stride_head, k_cache,
                           v_cache, s->num_cache_blocks, s->block_tables, s->bt_stride, s->cu_q, s->ctx_start,
                           s->num_seqs, s->max_q_len, s->num_heads, s->num_kv_heads, s->head_dim, s->block_size,
                           s->max_blocks_per_seq, s->scale, s->dtype, stream);
}
