// Device-side construction of a step's index tensors, gfx950.
//
// The reference builds slot_mapping [tokens, L, H] and the block table on the
// host every step and uploads them (csrc/batch_scheduler.cpp:131-169,
// muxserve/flexserver/llm_runtime.py:301-327).  Here the device keeps a mirror
// of every live request's block-id run in the reference's own order,
//     mirror[row][token block][layer][head]          (csrc/batch_scheduler.h:19,44-52)
// and a step uploads only the allocator's reply plus 8 ints per sequence
// (mux_sched_get_batch_compact).  One kernel of four kinds of workgroups, all
// plain coalesced integer copies; the kinds do not wait for each other, because
// ids that this step appends are read from the reply rather than from the mirror.
// (As three kernels and two conversions a decode step of 32 sequences spent 20 us
// of the GPU and five launches on them, now 11.3 and one.  The 17 steps of a batch
// of 32 requests are mostly host work: 2070 - 2110 -> 1860 - 1900 us in four runs of
// both in turn on one machine; two runs of one side have differed by 13 % on another.)
//   append   the reply's new ids are copied behind each request's run
//   slots    slot_mapping[t][l][h] = id * block_size + offset, read from the
//            mirror: prompt token k -> block k / bs, offset k % bs; decode token ->
//            last block, offset (ctx - 1) % bs    (csrc/batch_scheduler.h:42-67)
//   table    decode steps: mirror rows transposed through LDS into the layout the
//            attention kernel reads, [L][sequence][H][token block]
//   widen    token ids and positions, uploaded as int32, to the int64 that the
//            model takes
// Results are bit-identical to what mux_sched_get_batch writes.
#include <algorithm>

#include "mux_common.h"
#include "muxserve_attn_step.h"

namespace mux {

constexpr int kDescInts = 8;   // row, blocks, first new block, new blocks, offset in reply, length, first token, decoding

struct StepParams {
  int32_t *mirror;               // [max_rows][max_blocks_per_seq][per]
  const int32_t *desc;           // [num_seqs][kDescInts]
  const int32_t *block_info;     // the allocator's reply, [n_block_info]
  int64_t *slot_mapping;         // [num_tokens][per]
  int32_t *block_tables;         // [L][num_seqs][H][max_blocks_out]
  const int32_t *narrow;         // [n_wide]
  int64_t *wide;                 // [n_wide]
  int64_t n_block_info, n_wide;
  // Workgroups: append_chunks per sequence, then slot_rows per token, then
  // table_x * table_y per sequence, then those of widen.
  int64_t begin_slots, begin_table, begin_widen, end;
  int32_t append_chunks, slot_rows, table_x, table_y;
  int32_t num_seqs, per, H, max_rows, max_blocks_per_seq, block_size, max_blocks_out;
};

// A descriptor that does not fit the mirror or the reply is skipped, never followed.
__device__ __forceinline__ bool desc_ok(const StepParams &P, const int32_t *d) {
  const int64_t count = static_cast<int64_t>(d[3]) * P.per;
  return d[0] >= 0 && d[0] < P.max_rows && d[1] >= 0 && d[1] <= P.max_blocks_per_seq && d[2] >= 0 && d[3] >= 0 &&
         static_cast<int64_t>(d[2]) + d[3] <= d[1] && d[4] >= 1 && d[4] + count <= P.n_block_info && d[5] >= 0 && d[6] >= 0;
}

// Id j (layer and head) of a sequence's token block tb.
__device__ __forceinline__ const int32_t *block_ids(const StepParams &P, const int32_t *d, int tb) {
  const int fresh = tb - d[2];
  if (fresh >= 0 && fresh < d[3]) return P.block_info + d[4] + static_cast<int64_t>(fresh) * P.per;
  return P.mirror + (static_cast<int64_t>(d[0]) * P.max_blocks_per_seq + tb) * P.per;
}

__device__ __forceinline__ void step_append(const StepParams &P, int seq, int chunk) {
  const int32_t *d = P.desc + seq * kDescInts;
  if (!desc_ok(P, d)) return;
  const int64_t count = static_cast<int64_t>(d[3]) * P.per;
  const int64_t begin = static_cast<int64_t>(chunk) * 1024;
  const int64_t end = min(count, begin + 1024);
  int32_t *dst = P.mirror + (static_cast<int64_t>(d[0]) * P.max_blocks_per_seq + d[2]) * P.per;
  const int32_t *src = P.block_info + d[4];
  for (int64_t e = begin + threadIdx.x; e < end; e += 256) dst[e] = src[e];
}

__device__ __forceinline__ void step_slots(const StepParams &P, int t, int part) {
  const int lane = threadIdx.x & 63;
  // The batch entry that owns token t: the last one whose first token is <= t.
  int before = 0;
  for (int base = 0; base < P.num_seqs; base += 64) {
    const int i = base + lane;
    const int first = i < P.num_seqs ? P.desc[i * kDescInts + 6] : 0x7fffffff;
    before += __popcll(__builtin_amdgcn_ballot_w64(first <= t));
  }
  if (before == 0) return;
  const int32_t *d = P.desc + (before - 1) * kDescInts;
  if (!desc_ok(P, d)) return;
  int tb, off;
  if (d[7]) {                                 // decoding: the token just appended
    tb = d[1] - 1;
    off = (d[5] - 1) % P.block_size;
    if (t != d[6] || d[5] < 1) return;
  } else {
    const int k = t - d[6];
    if (k >= d[5]) return;
    tb = k / P.block_size;
    off = k % P.block_size;
  }
  if (tb < 0 || tb >= d[1]) return;
  const int32_t *ids = block_ids(P, d, tb);
  int64_t *out = P.slot_mapping + static_cast<int64_t>(t) * P.per;
  for (int j = part * 1024 + threadIdx.x; j < min(P.per, (part + 1) * 1024); j += 256)
    out[j] = static_cast<int64_t>(ids[j]) * P.block_size + off;
}

// One 64 x 64 tile of a sequence's [token block][layer, head] matrix, transposed.
__device__ __forceinline__ void step_table(const StepParams &P, int c, int bx, int by) {
  __shared__ int32_t tile[64][65];
  const int32_t *d = P.desc + c * kDescInts;
  const bool ok = desc_ok(P, d) && d[7];
  const int n_blocks = ok ? d[1] : 0;
  const int j0 = bx * 64, tb0 = by * 64;
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  if (n_blocks > tb0) {
#pragma unroll 4
    for (int r = y; r < 64; r += 4) {
      const int tb = tb0 + r, j = j0 + x;
      tile[r][x] = (tb < n_blocks && j < P.per) ? block_ids(P, d, tb)[j] : 0;
    }
  }
  __syncthreads();
#pragma unroll 4
  for (int r = y; r < 64; r += 4) {
    const int j = j0 + r, tb = tb0 + x;
    if (j < P.per && tb < P.max_blocks_out) {
      const int l = j / P.H, h = j - l * P.H;
      // Entries past the sequence's blocks are never read; zero keeps them defined.
      P.block_tables[((static_cast<int64_t>(l) * P.num_seqs + c) * P.H + h) * P.max_blocks_out + tb] =
          tb < n_blocks ? tile[x][r] : 0;
    }
  }
}

__global__ __launch_bounds__(256) void step_build_kernel(const StepParams P) {
  const int64_t w = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
  if (w >= P.end) return;
  if (w < P.begin_slots) {
    step_append(P, static_cast<int>(w / P.append_chunks), static_cast<int>(w % P.append_chunks));
  } else if (w < P.begin_table) {
    const int64_t u = w - P.begin_slots;
    step_slots(P, static_cast<int>(u / P.slot_rows), static_cast<int>(u % P.slot_rows));
  } else if (w < P.begin_widen) {
    const int64_t u = w - P.begin_table, xy = static_cast<int64_t>(P.table_x) * P.table_y;
    const int in = static_cast<int>(u % xy);
    step_table(P, static_cast<int>(u / xy), in % P.table_x, in / P.table_x);
  } else {
    const int64_t e = (w - P.begin_widen) * 256 + threadIdx.x;
    if (e < P.n_wide) P.wide[e] = P.narrow[e];
  }
}

}  // namespace mux

extern "C" int32_t mux_build_step_inputs(int32_t *mirror, int32_t max_rows, int32_t max_blocks_per_seq,
                                         int32_t num_layers, int32_t num_heads, int32_t block_size,
                                         const int32_t *desc, int32_t num_seqs, const int32_t *block_info,
                                         int64_t n_block_info, int32_t max_new_blocks, int32_t num_tokens,
                                         int64_t *slot_mapping, int32_t *block_tables, int32_t max_blocks_out,
                                         void *stream) {
  return mux_build_step(mirror, max_rows, max_blocks_per_seq, num_layers, num_heads, block_size, desc, num_seqs,
                        block_info, n_block_info, max_new_blocks, num_tokens, slot_mapping, block_tables,
                        max_blocks_out, nullptr, nullptr, 0, stream);
}

extern "C" int32_t mux_build_step(int32_t *mirror, int32_t max_rows, int32_t max_blocks_per_seq, int32_t num_layers,
                                  int32_t num_heads, int32_t block_size, const int32_t *desc, int32_t num_seqs,
                                  const int32_t *block_info, int64_t n_block_info, int32_t max_new_blocks,
                                  int32_t num_tokens, int64_t *slot_mapping, int32_t *block_tables,
                                  int32_t max_blocks_out, const int32_t *narrow, int64_t *wide, int64_t n_wide,
                                  void *stream) {
  using namespace mux;
  if (!mirror || max_rows <= 0 || max_blocks_per_seq <= 0 || num_layers <= 0 || num_heads <= 0 || block_size <= 0)
    return MUXA_EINVAL;
  if (num_seqs < 0 || num_tokens < 0 || n_block_info < 1 || max_new_blocks < 0 || max_blocks_out < 0) return MUXA_EINVAL;
  if (n_wide < 0 || (n_wide > 0 && (!narrow || !wide))) return MUXA_EINVAL;
  if (num_seqs == 0) num_tokens = max_new_blocks = max_blocks_out = 0;      // nothing but the conversion
  if (num_seqs > 0 && (!desc || !block_info || (num_tokens > 0 && !slot_mapping) || (max_blocks_out > 0 && !block_tables)))
    return MUXA_EINVAL;
  const int64_t per = static_cast<int64_t>(num_layers) * num_heads;
  // Sizes that no step has (the workgroup count below stays far from 64 bits).
  if (per > 65535 * 1024 || num_seqs > 65535 || max_blocks_out > 65535 * 64 ||
      static_cast<int64_t>(max_new_blocks) * per > (int64_t{1} << 40))
    return MUXA_EUNSUPPORTED;
  StepParams P;
  P.mirror = mirror;
  P.desc = desc;
  P.block_info = block_info;
  P.slot_mapping = slot_mapping;
  P.block_tables = block_tables;
  P.n_block_info = n_block_info;
  P.num_seqs = num_seqs;
  P.per = static_cast<int32_t>(per);
  P.H = num_heads;
  P.max_rows = max_rows;
  P.max_blocks_per_seq = max_blocks_per_seq;
  P.block_size = block_size;
  P.max_blocks_out = max_blocks_out;
  P.narrow = narrow;
  P.wide = wide;
  P.n_wide = n_wide;
  const int64_t chunks = (static_cast<int64_t>(max_new_blocks) * per + 1023) / 1024;
  if (chunks > 0x7fffffff) return MUXA_EUNSUPPORTED;
  P.append_chunks = static_cast<int32_t>(chunks);
  P.slot_rows = static_cast<int32_t>((per + 1023) / 1024);
  P.table_x = static_cast<int32_t>((per + 63) / 64);
  P.table_y = (max_blocks_out + 63) / 64;
  P.begin_slots = chunks * num_seqs;
  P.begin_table = P.begin_slots + static_cast<int64_t>(num_tokens) * P.slot_rows;
  P.begin_widen = P.begin_table + static_cast<int64_t>(P.table_x) * P.table_y * num_seqs;
  P.end = P.begin_widen + (n_wide + 255) / 256;
  if (P.end == 0) return MUXA_OK;
  // (a dimension of the grid holds fewer than 2^32 threads)
  const int64_t gx = std::min<int64_t>(P.end, 1 << 20), gy = (P.end + gx - 1) / gx;
  if (gy > 65535) return MUXA_EUNSUPPORTED;
  hipLaunchKernelGGL(step_build_kernel, dim3(static_cast<uint32_t>(gx), static_cast<uint32_t>(gy)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), P);
  MUX_HIP_TRY(hipGetLastError());
  return MUXA_OK;
}
