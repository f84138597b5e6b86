/* Whole steps of the attention layer on libmuxattn.so: entry points that do in
 * one call what rotary, cache write and attention of muxserve_attn.h do in turn.
 * Conventions (pointers, streams, return codes) are those of that header. */
#ifndef MUXSERVE_ATTN_STEP_H
#define MUXSERVE_ATTN_STEP_H

#include "muxserve_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* A whole prompt step of the attention layer (models/llama.py:159-161): rotary
 * embedding of q and k in place, causal attention, and the cache write of the
 * rotated k and of v.  Two launches: k is rotated by itself, the attention
 * kernel rotates q and scatters the K and V tiles that it reads anyway; one launch
 * for short prompts with as many kv heads as query heads (csrc/prompt_step.h).  `attn`
 * and `write` describe the same q, k and v (equal pointers, strides and head
 * counts); attn->prompt_lens_host is required, adds up to write->num_tokens and
 * agrees with cu_seqlens, so that every token belongs to a prompt; the head
 * rotates as a whole (rotary_dim 128).  Same results as mux_rotary_neox,
 * mux_reshape_and_cache and mux_prefill_causal in turn. */
int32_t mux_rope_prefill_and_cache(const MuxPrefillItem *attn, const MuxCacheWriteItem *write, void *k_pool,
                                   void *v_pool, int64_t num_pool_blocks, int32_t head_size, int32_t block_size,
                                   int32_t dtype, void *stream);

/* mux_build_step_inputs and the widening of n_wide int32 (the step's token ids
 * and positions) to int64, in one launch.  narrow, wide: DEVICE; n_wide may be 0. */
int32_t mux_build_step(int32_t *mirror, int32_t max_rows, int32_t max_blocks_per_seq, int32_t num_layers,
                       int32_t num_heads, int32_t block_size, const int32_t *desc, int32_t num_seqs,
                       const int32_t *block_info, int64_t n_block_info, int32_t max_new_blocks, int32_t num_tokens,
                       int64_t *slot_mapping, int32_t *block_tables, int32_t max_blocks_out, const int32_t *narrow,
                       int64_t *wide, int64_t n_wide, void *stream);

#ifdef __cplusplus
}
#endif

#endif
