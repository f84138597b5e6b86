// The decode step of one short sequence as one launch (paged_decode.hip), for the
// operator that takes it where it can.
#pragma once
#include "muxserve_attn.h"

namespace mux {

// Rotation of q and k in place, cache write and attention of what `d` and `w` describe
// (the same q).  *taken: 0 where this is not such a step; nothing has been launched then.
int32_t single_row_step(const MuxDecodeItem &d, const MuxCacheWriteItem &w, void *k_pool, void *v_pool,
                        int64_t num_pool_blocks, int32_t block_size, int32_t dtype, void *stream, int32_t *taken);

}  // namespace mux
