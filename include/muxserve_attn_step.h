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
 * kernel rotates q and scatters the K and V tiles that it reads anyway.  `attn`
 * and `write` describe the same q, k and v (equal pointers, strides and head
 * counts); attn->prompt_lens_host is required, adds up to write->num_tokens and
 * agrees with cu_seqlens, so that every token belongs to a prompt; the head
 * rotates as a whole (rotary_dim 128).  Same results as mux_rotary_neox,
 * mux_reshape_and_cache and mux_prefill_causal in turn. */
int32_t mux_rope_prefill_and_cache(const MuxPrefillItem *attn, const MuxCacheWriteItem *write, void *k_pool,
                                   void *v_pool, int64_t num_pool_blocks, int32_t head_size, int32_t block_size,
                                   int32_t dtype, void *stream);

#ifdef __cplusplus
}
#endif

#endif
