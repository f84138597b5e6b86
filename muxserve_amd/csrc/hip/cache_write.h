// Pieces shared by the KV-cache write kernels and the prompt attention kernel
// that writes the cache itself.
#pragma once

#include "mux_common.h"
#include "muxserve_attn_step.h"

namespace mux {

struct RopeArgs {
  uint16_t *q;                 // rotated in place; may be null
  int64_t q_stride;
  int32_t ratio;               // query heads per kv head
  const int64_t *positions;    // [num_tokens]
  const float *cos_sin;        // [max_position, 128] = [cos | sin]
  int32_t max_position;
};

// out = own * cos + (is_y ? +1 : -1) * partner * sin, elementwise on 8 packed values.
template <typename T>
__device__ __forceinline__ uint4 rotate_chunk(const uint4 own, const uint4 partner, const float (&cs)[8],
                                              const float (&sn)[8], bool is_y) {
  const uint32_t a[4] = {own.x, own.y, own.z, own.w};
  const uint32_t b[4] = {partner.x, partner.y, partner.z, partner.w};
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float a0, a1, b0, b1;
    if constexpr (__is_same(T, F16)) {
      const half2_t ah = as_half2(a[e]), bh = as_half2(b[e]);
      a0 = static_cast<float>(ah.x); a1 = static_cast<float>(ah.y);
      b0 = static_cast<float>(bh.x); b1 = static_cast<float>(bh.y);
    } else {
      a0 = bf16_lo(a[e]); a1 = bf16_hi(a[e]);
      b0 = bf16_lo(b[e]); b1 = bf16_hi(b[e]);
    }
    // x' = x c - y s for the low half of a head, y' = y c + x s for the high half.
    const float r0 = is_y ? a0 * cs[2 * e] + b0 * sn[2 * e] : a0 * cs[2 * e] - b0 * sn[2 * e];
    const float r1 = is_y ? a1 * cs[2 * e + 1] + b1 * sn[2 * e + 1] : a1 * cs[2 * e + 1] - b1 * sn[2 * e + 1];
    o[e] = to_storage2<T>(r0, r1);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// Stores that fill whole 128-byte lines by themselves go out non-temporal
// (nothing to merge with, and the pool is not read back soon): K rows of a run
// of 8 consecutive slots, V rows when the workgroup holds every run of the row.
typedef uint32_t cw_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store16(void *p, const uint4 x, bool streaming) {
  const cw_u32x4 v = {x.x, x.y, x.z, x.w};
  if (streaming) {
    // Written as an instruction: as two C++ stores that differ only in the hint,
    // the optimiser folds the branches into one store and drops it.  The
    // compiler does not know that the instruction is still reading its data
    // registers when the next one issues, so the wait states between a 16-byte
    // store and a write of its data registers are spelled out (one was not
    // enough once the next store's operands were already in registers).
    asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 4" ::"v"(p), "v"(v) : "memory");
  } else {
    *static_cast<cw_u32x4 *>(p) = v;
  }
}

// What every entry point that writes the pool refuses.
inline int32_t check_cache_write(const void *k, const void *v, int64_t kv_row_stride, const void *k_pool,
                                 const void *v_pool, int64_t num_pool_blocks, const int64_t *slot_mapping, int32_t layer,
                                 int32_t num_layers, int32_t num_tokens, int32_t num_kv_heads, int32_t head_size,
                                 int32_t block_size, int32_t dtype) {
  // (pointers are only required when there is something to do)
  if (num_tokens > 0 && (!k || !v || !k_pool || !v_pool || !slot_mapping)) return MUXA_EINVAL;
  if (num_tokens < 0 || num_kv_heads <= 0 || num_pool_blocks <= 0) return MUXA_EINVAL;
  if (layer < 0 || layer >= num_layers) return MUXA_EINVAL;
  if (head_size != kHeadSize) return MUXA_EUNSUPPORTED;
  if (block_size != 8 && block_size != 16 && block_size != 32) return MUXA_EUNSUPPORTED;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  if (kv_row_stride < static_cast<int64_t>(num_kv_heads) * kHeadSize || kv_row_stride % 8 != 0)
    return MUXA_EINVAL;
  const uintptr_t align = reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                          reinterpret_cast<uintptr_t>(k_pool) | reinterpret_cast<uintptr_t>(v_pool);
  if (align & 15u) return MUXA_EINVAL;
  if (num_tokens > 16 * 65535) return MUXA_EUNSUPPORTED;      // one grid row per 16 tokens
  if (num_pool_blocks > (int64_t{1} << 56)) return MUXA_EINVAL;   // slot arithmetic stays in 64 bits
  return MUXA_OK;
}

// Rotates k alone (rotary.hip), for a launch whose attention kernel rotates q.
hipError_t launch_rotary_k(const int64_t *positions, uint16_t *k, int64_t k_stride, const float *cos_sin,
                           int32_t max_position, int32_t num_tokens, int32_t num_kv_heads, int32_t dtype,
                           hipStream_t st);

}  // namespace mux
