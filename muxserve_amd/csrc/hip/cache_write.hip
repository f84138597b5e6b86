// KV-cache write (reshape_and_cache) into the head-granular pool, gfx950.
//
// Pure byte movement.  A 256-thread workgroup takes about 16 consecutive
// tokens of one kv head.  Loading, thread (i, c) takes the 16-byte chunk c (dims
// 8c..8c+7) of token i of both K and V, so that a token's 256-byte head slice is
// read by 16 neighbouring threads; the tile goes to LDS, one row per token, and
// is stored from there by thread (c, i):
//   K pool [D/8][BS][8]: the chunk goes out as one 16-byte store; the token
//     lanes of a chunk row are adjacent, so tokens in consecutive slots of one
//     block fill a contiguous run.
//   V pool [D][BS]: 8 consecutive tokens of one dim are a 16-byte chunk of the
//     pool.  Where 8 consecutive tokens go to 8 consecutive slots that start at
//     a multiple of 8 (every prompt written through a block table does, up to
//     its last few tokens) one thread gathers a dim's 8 values from the LDS rows
//     and stores the whole chunk.  Tokens outside such runs (decode steps,
//     arbitrary slots, prompt tails) take the element path: a chunk's 8 dims
//     as 8 two-byte stores BS*2 bytes apart.
// Packed prompts start anywhere in the token stream, so runs are not aligned
// to multiples of 16 tokens.  The boundary between workgroups w-1 and w is
// therefore moved back from token 16w to the start of the run that contains
// token 16w - and, when that run is the second half of a pool block whose first
// half precedes it, on to the start of the block: inside a prompt every window
// is then exactly one pool block (whole K and V rows, streamed past the L2),
// whatever the prompt's position in the stream.  Both neighbours derive the
// boundary from the same slots, the windows still tile the token stream
// exactly, each holds 1..31 tokens, and no run straddles two workgroups.  The
// slots are read first and only the window's own tokens are loaded.
//
// Fused variant (ROPE): the same kernel first applies the NeoX rotary embedding
// to k (and to the query heads that share this kv head) for the tokens of its
// window, in place, and scatters the rotated k - one launch and one pass over k
// instead of a rotary kernel followed by the cache write.  A thread's chunk c
// pairs with chunk c^8 (dims +-64) of the same token: both are read, the
// workgroup meets, then the rotated chunk goes back in place and into the pool.
#include "cache_write.h"

namespace mux {

constexpr int kVtRow = kHeadSize + 8;    // LDS row of one token: 256 B + 16 B so that rows shift banks
constexpr int kBack = 16;                // tokens before the nominal 16 that a window may take over
constexpr int kSlotWin = 48;             // slots of tokens 16w-16 .. 16w+31 are examined
constexpr int kTileRows = 32;            // a window lies inside tokens 16w-16 .. 16w+15

// One workgroup's window: kv head h, tokens around T0 (a multiple of 16).
template <typename T, bool ROPE, bool EARLY_Q>
__device__ __forceinline__ void cache_write_window(
    uint16_t *k, const uint16_t *__restrict__ v, int64_t row_stride,
    uint4 *__restrict__ k_pool, uint16_t *__restrict__ v_pool, int64_t num_blocks,
    const int64_t *__restrict__ slots, int64_t slot_stride, int num_tokens, int block_size, const RopeArgs &R,
    const int h, const int T0) {
  constexpr int D = kHeadSize;
  __shared__ __attribute__((aligned(16))) uint16_t kt[kTileRows][kVtRow];
  __shared__ __attribute__((aligned(16))) uint16_t vt[kTileRows][kVtRow];
  __shared__ int64_t s_slot[kSlotWin + 8];
  const int lane = threadIdx.x & 63;
  const int i = threadIdx.x & 15;
  const int c = threadIdx.x >> 4;
  const int64_t pool_slots = num_blocks * block_size;
  // Block sizes are powers of two (8, 16, 32): slot -> (block, offset) by shift and mask.
  const int bs_shift = __builtin_ctz(static_cast<unsigned>(block_size));

  // Slots of tokens T0-16 .. T0+31 (bit j of the masks below is token T0-16+j);
  // -1 for tokens outside the batch, skipped tokens and slots outside the pool
  // (never written).
  if (threadIdx.x < kSlotWin + 8) {
    const int t = T0 - kBack + static_cast<int>(threadIdx.x);
    int64_t sl = -1;
    if (threadIdx.x < kSlotWin && t >= 0 && t < num_tokens) sl = slots[static_cast<int64_t>(t) * slot_stride + h];
    s_slot[threadIdx.x] = (sl >= 0 && sl < pool_slots) ? sl : -1;
  }
  __syncthreads();
  // Bit j of `starts`: token j begins a run (8 consecutive slots from a multiple of 8).
  // Bit j of `chained`: the next token goes to the slot behind token j's.
  bool is_start = false, is_valid = false, is_chained = false;
  if (lane < 40) {
    const int64_t s0 = s_slot[lane];
    is_valid = s0 >= 0;
    is_chained = is_valid && s_slot[lane + 1] == s0 + 1;
    is_start = is_chained && (s0 & 7) == 0;
#pragma unroll
    for (int e = 2; e < 8; ++e) is_start = is_start && s_slot[lane + e] == s0 + e;
  }
  const unsigned long long starts = __builtin_amdgcn_ballot_w64(is_start);
  // Tokens by themselves, as in a decode step (see the comment at rope_scatter_kernel): no
  // neighbour in the batch goes to the slot beside theirs.  Not the last token of a prompt
  // that has a block to itself: the token in front of it is in a run.
  const unsigned long long chained = __builtin_amdgcn_ballot_w64(is_chained), in_chain = chained | chained << 1;
  const unsigned long long lone = __builtin_amdgcn_ballot_w64(is_valid) & ~in_chain & ~(in_chain << 1);
  // The boundary next to nominal bit n: the start of the run that contains
  // token n, moved on to the start of that run's pool block when the run is the
  // block's second half and the first half sits right before it - so that
  // inside a prompt a window is exactly one pool block.  Both neighbours derive
  // the boundary from the same slots.
  auto boundary = [&](int n) {
    const unsigned long long cand = starts & (0xffull << (n - 7));      // runs starting at n-7 .. n
    if (cand == 0) return n;
    int sbit = __ffsll(cand) - 1;
    if (block_size == 16 && (s_slot[sbit] & 15) == 8 && ((starts >> (sbit - 8)) & 1ull) != 0 &&
        s_slot[sbit - 8] == s_slot[sbit] - 8)
      sbit -= 8;
    return sbit;
  };
  const int ja = boundary(kBack);
  const int jb = min(boundary(kBack + 16), num_tokens - T0 + kBack);
  const unsigned long long in_win = starts & (~0ull << ja) & ~(~0ull << jb);   // runs that start inside the window
  const unsigned long long lone_win = lone & (~0ull << ja) & ~(~0ull << jb);   // (prompts: none)
  // Does this window write whole pool rows and nothing else?  K rows of a run are
  // 128 bytes; a V row is block_size * 2 bytes: one run fills it at block size 8,
  // the two runs of a block at 16, never at 32.  Such a window streams its stores
  // past the L2 (uniform over the workgroup).
  const int n_runs = __popcll(in_win);
  const int first_bit = n_runs > 0 ? __ffsll(in_win) - 1 : 0;
  const bool rows_complete =
      n_runs > 0 && jb - ja == 8 * n_runs &&
      (block_size == 8 || (block_size == 16 && n_runs == 2 && ((in_win >> (first_bit + 8)) & 1ull) != 0 &&
                           (s_slot[first_bit] & 15) == 0 && s_slot[first_bit + 8] == s_slot[first_bit] + 8));

  // Loads: thread (token il, chunk cl) - the 16 threads of a token read its whole
  // 256-byte head slice, a wave four such slices, every line exactly once.
  // (Non-temporal loads make no difference whether k/v come from HBM or were
  // just written by the projection, and lose when the same buffers are read
  // again.)  Stores: thread
  // (chunk row c, token i) - the 16 threads of a chunk row write one whole
  // 256-byte K row of the block with a single store instruction (split over
  // two, the non-temporal stores would each leave partial lines).  In between
  // the tile sits in LDS, one row per token (rows are bit positions); V is
  // transposed on its way out.  A window has at most 31 tokens: two passes of
  // 16, the second one rare.
  const bool two_passes = jb - ja > 16;                    // uniform
  const int il = threadIdx.x >> 4, cl = threadIdx.x & 15;
  const int pc = (cl ^ 8) - cl;            // the partner chunk of the rotation, in chunks from this one
  // EARLY_Q, for one query head per kv head: the positions and the query rows are
  // requested with k and v, so that only the cos|sin row is a memory latency of
  // its own.
  uint4 kx2[2], vx2[2], kp2[2], qx2[EARLY_Q ? 2 : 1], qp2[EARLY_Q ? 2 : 1];
  int64_t pos2[EARLY_Q ? 2 : 1];
  const int n_q = ROPE && R.q != nullptr ? R.ratio : 0;
  const int64_t q_head0 = static_cast<int64_t>(h) * R.ratio * D + cl * 8;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    kx2[pass] = vx2[pass] = kp2[pass] = make_uint4(0, 0, 0, 0);
    if constexpr (EARLY_Q) {
      qx2[pass] = qp2[pass] = make_uint4(0, 0, 0, 0);
      pos2[pass] = 0;
    }
    if (pass == 1 && !two_passes) break;
    const int j = ja + 16 * pass + il;
    if (j < jb && (ROPE || s_slot[j] >= 0)) {
      const int64_t src = static_cast<int64_t>(T0 - kBack + j) * row_stride + h * D + cl * 8;
      kx2[pass] = *reinterpret_cast<const uint4 *>(k + src);
      vx2[pass] = *reinterpret_cast<const uint4 *>(v + src);
      if constexpr (EARLY_Q) pos2[pass] = R.positions[T0 - kBack + j];
      if constexpr (ROPE) kp2[pass] = *reinterpret_cast<const uint4 *>(k + src + pc * 8);
      if (EARLY_Q && n_q == 1) {
        const uint16_t *qp = R.q + static_cast<int64_t>(T0 - kBack + j) * R.q_stride + q_head0;
        qx2[pass] = *reinterpret_cast<const uint4 *>(qp);
        qp2[pass] = *reinterpret_cast<const uint4 *>(qp + pc * 8);
      }
    }
  }
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1 && !two_passes) break;
    const int j = ja + 16 * pass + il;
    const bool mine = j < jb;                              // token T0-16+j is in this window
    uint4 kx = kx2[pass];
    if constexpr (ROPE) {
      // Rotate k of every token of the window (also tokens without a slot), and
      // the query heads of this kv head, four at a time; all reads of a group
      // precede its writes (the workgroup meets in between), because a thread's
      // partner chunk is another thread's own.
      const int t = T0 - kBack + j;
      const int64_t src = static_cast<int64_t>(t) * row_stride + h * D + cl * 8;
      float cs[8], sn[8];
      if (mine) {
        int64_t pos;
        if constexpr (EARLY_Q) pos = pos2[pass];
        else pos = R.positions[t];
        pos = pos < 0 ? 0 : (pos >= R.max_position ? R.max_position - 1 : pos);
        const float *row = R.cos_sin + pos * D + (cl & 7) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          cs[e] = row[e];
          sn[e] = row[D / 2 + e];
        }
        kx = rotate_chunk<T>(kx, kp2[pass], cs, sn, cl >= 8);
      }
      uint16_t *q0 = R.q + static_cast<int64_t>(t) * R.q_stride + q_head0;
      for (int g0 = 0; g0 < max(n_q, 1); g0 += 4) {
        uint4 qx[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (mine && g0 + g < n_q) {
            const uint16_t *qp = q0 + (g0 + g) * D;
            if (EARLY_Q && n_q == 1)
              qx[g] = rotate_chunk<T>(qx2[pass], qp2[pass], cs, sn, cl >= 8);
            else
              qx[g] = rotate_chunk<T>(*reinterpret_cast<const uint4 *>(qp),
                                      *reinterpret_cast<const uint4 *>(qp + pc * 8), cs, sn, cl >= 8);
          }
        __syncthreads();
        if (mine && g0 == 0) *reinterpret_cast<uint4 *>(k + src) = kx;
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (mine && g0 + g < n_q) *reinterpret_cast<uint4 *>(q0 + (g0 + g) * D) = qx[g];
      }
    }
    if (mine) {
      *reinterpret_cast<uint4 *>(&kt[j][cl * 8]) = kx;
      *reinterpret_cast<uint4 *>(&vt[j][cl * 8]) = vx2[pass];
    }
  }
  __syncthreads();
  static_assert(kBack >= 16, "a window's tokens have a neighbour on either side in s_slot");
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1 && !two_passes) break;
    const int j = ja + 16 * pass + i;
    const int64_t slot = j < jb ? s_slot[j] : -1;
    if (slot >= 0) {
      const int64_t blk = slot >> bs_shift;
      const int o = static_cast<int>(slot) & (block_size - 1);
      // Element path for tokens that no run covers (a run starts at most 7 tokens back).
      const unsigned long long cover = in_win & (0xffull << (j > 7 ? j - 7 : 0)) & ~(~0ull << (j + 1));
      store16(&k_pool[(blk * (D / 8) + c) * block_size + o], *reinterpret_cast<const uint4 *>(&kt[j][c * 8]),
              rows_complete || ((lone_win >> j) & 1) != 0);
      if (cover == 0 && ((lone_win >> j) & 1) == 0) {
        uint16_t *vp = v_pool + (blk * D + c * 8) * block_size + o;
        const uint4 vx = *reinterpret_cast<const uint4 *>(&vt[j][c * 8]);
        const uint32_t w[4] = {vx.x, vx.y, vx.z, vx.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vp[(2 * e) * block_size] = static_cast<uint16_t>(w[e] & 0xffffu);
          vp[(2 * e + 1) * block_size] = static_cast<uint16_t>(w[e] >> 16);
        }
      }
    }
  }
  // V of tokens by themselves: 32 threads per token, 32 neighbouring dims of the block
  // per instruction, so that four lanes share a line.
  if (lone_win != 0) {
    for (int j = ja + static_cast<int>(threadIdx.x >> 5); j < jb; j += 8) {
      const int64_t slot = s_slot[j];
      if (((lone_win >> j) & 1) == 0) continue;
      const int l = threadIdx.x & 31;
      uint16_t *const vp = v_pool + ((slot >> bs_shift) * D + l) * block_size + (static_cast<int>(slot) & (block_size - 1));
#pragma unroll
      for (int e = 0; e < 4; ++e) __builtin_nontemporal_store(vt[j][l + 32 * e], &vp[32 * e * block_size]);
    }
  }
  // Up to three runs per window; thread (c, i) stores dim 8c + i%8 of runs i/8, i/8 + 2.
  for (int r = i >> 3; r < n_runs; r += 2) {
    unsigned long long m = in_win;
    for (int q = 0; q < r; ++q) m &= m - 1;                // drop the runs before run r
    const int jp = __ffsll(m) - 1;                         // bit, and LDS row, of the run's first token
    const int d = c * 8 + (i & 7);
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = static_cast<uint32_t>(vt[jp + 2 * e][d]) | (static_cast<uint32_t>(vt[jp + 2 * e + 1][d]) << 16);
    const int64_t slot0 = s_slot[jp];
    const int64_t b0 = slot0 >> bs_shift;
    const int o0 = static_cast<int>(slot0) & (block_size - 1);
    store16(v_pool + (b0 * D + d) * block_size + o0, make_uint4(w[0], w[1], w[2], w[3]), rows_complete);
  }
}

// Heads vary fastest over the workgroup ids: workgroups that run together read
// the neighbouring 256-byte head slices of the same k/v rows (one DRAM page)
// rather than one slice out of each of many rows.
template <typename T, bool ROPE, bool EARLY_Q>
__global__ __launch_bounds__(256) void reshape_and_cache_kernel(
    uint16_t *k, const uint16_t *__restrict__ v, int64_t row_stride,
    uint4 *__restrict__ k_pool, uint16_t *__restrict__ v_pool, int64_t num_blocks,
    const int64_t *__restrict__ slots, int64_t slot_stride, int num_tokens, int block_size, const RopeArgs R) {
  cache_write_window<T, ROPE, EARLY_Q>(k, v, row_stride, k_pool, v_pool, num_blocks, slots, slot_stride, num_tokens,
                                       block_size, R, blockIdx.x, blockIdx.y * 16);
}

// Several colocated models' cache writes of one step in one grid: the kernel
// argument carries one descriptor per model, a workgroup finds its model from
// the models' first workgroup ids and then does what the single-model kernel
// does (heads fastest within a model).
struct CacheWriteItemDev {
  uint16_t *k;
  const uint16_t *v;
  int64_t row_stride;
  const int64_t *slots;          // layer slice of the model's slot mapping
  int64_t slot_stride;
  RopeArgs rope;
  int32_t num_tokens;
  int32_t num_kv_heads;
  int32_t work_begin;            // first workgroup of this model
  int32_t per_xcd;               // rope_scatter_kernel: workgroups of this model per XCD; 0: rows packed token after token
};
struct MultiCacheWriteParams {
  CacheWriteItemDev it[MUXA_MAX_DECODE_ITEMS];
  uint4 *k_pool;
  uint16_t *v_pool;
  int64_t num_blocks;
  int32_t n_items;
  int32_t block_size;
};

template <typename T, bool ROPE, bool EARLY_Q>
__global__ __launch_bounds__(256) void multi_reshape_and_cache_kernel(const MultiCacheWriteParams P) {
  const int w = blockIdx.x;
  int ii = 0;
#pragma unroll
  for (int i = 1; i < MUXA_MAX_DECODE_ITEMS; ++i)
    if (i < P.n_items && w >= P.it[i].work_begin) ii = i;
  const CacheWriteItemDev I = P.it[ii];
  const int local = w - I.work_begin;
  const int ty = local / I.num_kv_heads;
  const int h = local - ty * I.num_kv_heads;
  cache_write_window<T, ROPE, EARLY_Q>(I.k, I.v, I.row_stride, P.k_pool, P.v_pool, P.num_blocks, I.slots, I.slot_stride,
                                       I.num_tokens, P.block_size, I.rope, h, ty * 16);
}

// What lane 0 (0x00), 1 (0x55), 2 (0xAA) or 3 (0xFF) of the quad holds.
template <int kCtrl>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t v) {
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xf, 0xf, true);
}

// The rotary form for steps of few tokens, where the chain of dependent loads is
// what counts: 32 lanes per (token, row), a row being a kv head (k rotated in
// place and scattered, v scattered) or a query head (rotated in place).  A lane
// holds both halves of its pairs, so nothing meets in LDS or at a barrier, and
// everything but the cos|sin row is requested at once: two memory latencies
// against the window kernel's five.  No runs are looked for (a decode step has
// none); a V store instruction covers 32 neighbouring dims of the block, four
// lanes to a 128-byte line.
//
// A token by itself - no neighbour in the batch goes to the slot beside its own, as in
// a decode step - is stored past the L2, here and in the window kernel (with rotation and
// without): it leaves a few bytes in each of 32 lines of V and 16 of K, and left in the L2
// those lines cost the attention behind the write more than the write itself.  us, kept /
// past the L2, over six sets of blocks and sixteen successive steps in turn: attention
// alone, 16 x 40 heads bf16 31.8 / 29.7, 56 tokens of three models 85.4 / 78.8, 256 x 32
// heads 318 / 280, 64 x 8 heads on 64 bf16 235.3 / 233.9; the write alone 5.3 / 5.0, 8.3 / 8.4,
// 22.5 / 25.1, 5.3 / 5.2; both as calls 37.8 / 35.3, 94.9 / 88.0, 341 / 307, 245.2 / 243.1; the
// plain write of 256 x 32 heads 20.8 / 23.5, with the attention 346 / 313; a mixed step (4
// prompts of 300, 64 decode rows, 32 heads) 128 / 120.  Blocks of 8 and 32 tokens alike (256
// x 32 heads 326 / 305, 350 / 335); contexts of some 30 tokens gain nothing.  The attention
// reads and writes the same bytes past the L2 either way (counters), so it is not traffic.
// On one state again and again, where the lines of the last pass are still at hand, the
// write alone looks worse (256 x 32 heads 13.3 / 24.1).  Tokens in a run (prompts) write
// the same lines again and keep the L2.
template <typename T>
__global__ __launch_bounds__(256) void rope_scatter_kernel(const MultiCacheWriteParams P) {
  constexpr int D = kHeadSize;
  const int w = blockIdx.x;
  int ii = 0;
#pragma unroll
  for (int i = 1; i < MUXA_MAX_DECODE_ITEMS; ++i)
    if (i < P.n_items && w >= P.it[i].work_begin) ii = i;
  const CacheWriteItemDev I = P.it[ii];
  const RopeArgs R = I.rope;
  // A kv head is followed by its query heads: all of a token's kv rows first
  // would put them, and the pool stores, on half of the XCDs where the rows of a
  // token are a multiple of 64 (32 + 32 heads, 256 tokens: 18.9 us).
  const int per_kv = R.q != nullptr ? R.ratio + 1 : 1;
  const int rows = I.num_kv_heads * per_kv;
  const int l = threadIdx.x & 31;
  int t, row;
  if (I.per_xcd == 0) {
    const int unit = (w - I.work_begin) * 8 + (threadIdx.x >> 5);
    t = unit / rows;
    row = unit - t * rows;
    if (t >= I.num_tokens) return;
  } else {
    const int local = w - I.work_begin;
    const int u = (local & 7) * I.per_xcd + (local >> 3);
    const int rows8 = u / I.num_tokens;
    t = u - rows8 * I.num_tokens;
    row = 8 * rows8 + (threadIdx.x >> 5);
    if (row >= rows) return;
  }
  const int h = row / per_kv, hq = row - h * per_kv - 1;
  const bool kv = hq < 0;
  int64_t pos = R.positions[t];
  uint32_t *const x = reinterpret_cast<uint32_t *>(
      kv ? I.k + static_cast<int64_t>(t) * I.row_stride + h * D
         : R.q + static_cast<int64_t>(t) * R.q_stride + (h * R.ratio + hq) * D);
  const uint32_t lo = x[l], hi = x[32 + l];
  int64_t slot = -1, before = -1, after = -1;
  uint16_t ve[4] = {0, 0, 0, 0};
  if (kv) {
    const int64_t *const sp = I.slots + static_cast<int64_t>(t) * I.slot_stride + h;
    slot = *sp;
    before = sp[t > 0 ? -I.slot_stride : 0];            // (its own slot where there is no neighbour)
    after = sp[t + 1 < I.num_tokens ? I.slot_stride : 0];
    const uint16_t *vp = I.v + static_cast<int64_t>(t) * I.row_stride + h * D + l;
#pragma unroll
    for (int e = 0; e < 4; ++e) ve[e] = vp[32 * e];
  }
  __builtin_amdgcn_sched_barrier(0);       // all of that is requested before the position is waited for
  pos = pos < 0 ? 0 : (pos >= R.max_position ? R.max_position - 1 : pos);
  const float2 cs = reinterpret_cast<const float2 *>(R.cos_sin + pos * D)[l];
  const float2 sn = reinterpret_cast<const float2 *>(R.cos_sin + pos * D + D / 2)[l];
  float x0, x1, y0, y1;
  if constexpr (__is_same(T, F16)) {
    const half2_t a = as_half2(lo), b = as_half2(hi);
    x0 = static_cast<float>(a.x); x1 = static_cast<float>(a.y);
    y0 = static_cast<float>(b.x); y1 = static_cast<float>(b.y);
  } else {
    x0 = bf16_lo(lo); x1 = bf16_hi(lo);
    y0 = bf16_lo(hi); y1 = bf16_hi(hi);
  }
  const uint32_t xo = to_storage2<T>(x0 * cs.x - y0 * sn.x, x1 * cs.y - y1 * sn.y);
  const uint32_t yo = to_storage2<T>(y0 * cs.x + x0 * sn.x, y1 * cs.y + x1 * sn.y);
  x[l] = xo;
  x[32 + l] = yo;
  // A chunk of the K pool (8 dims) is spread over four lanes: the first of them
  // stores the lower half's chunk, the second the upper half's (64 dims on).
  // (both are fetched before the choice: all four lanes take part)
  const uint32_t ka[4] = {quad_bcast<0x00>(xo), quad_bcast<0x55>(xo), quad_bcast<0xAA>(xo), quad_bcast<0xFF>(xo)};
  const uint32_t kb[4] = {quad_bcast<0x00>(yo), quad_bcast<0x55>(yo), quad_bcast<0xAA>(yo), quad_bcast<0xFF>(yo)};
  uint4 kc;
  kc.x = (l & 1) ? kb[0] : ka[0];
  kc.y = (l & 1) ? kb[1] : ka[1];
  kc.z = (l & 1) ? kb[2] : ka[2];
  kc.w = (l & 1) ? kb[3] : ka[3];
  if (slot >= 0 && slot < P.num_blocks * P.block_size) {
    const int bs = P.block_size;
    const int64_t blk = slot >> __builtin_ctz(static_cast<unsigned>(bs));
    const int o = static_cast<int>(slot) & (bs - 1);
    const bool alone = before != slot - 1 && after != slot + 1;
    if ((l & 2) == 0) store16(&P.k_pool[(blk * (D / 8) + (l >> 2) + 8 * (l & 1)) * bs + o], kc, alone);
    uint16_t *const vp = P.v_pool + (blk * D + l) * bs + o;
    if (alone) {
      // (written as an instruction, as in store16: the branches would be folded)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        asm volatile("global_store_short %0, %1, off nt" ::"v"(&vp[32 * e * bs]), "v"(static_cast<uint32_t>(ve[e])) : "memory");
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) vp[32 * e * bs] = ve[e];
    }
  }
}

}  // namespace mux

namespace mux {
namespace {

// Up to this many (token, kv head) pairs of all models of a call take
// rope_scatter_kernel.  us, window kernel -> scatter kernel, decode: 32 heads, 1
// token 3.3 -> 2.8, 16 4.7 -> 3.2, 80 7.9 -> 6.3; 52 heads, 48 tokens 7.7 -> 6.1; 64
// query heads on 8, 1 token 4.8 -> 2.5, 64 6.8 -> 3.5.  One prompt, whose V the
// window kernel writes as whole chunks: 45 tokens x 32 heads 4.1 -> 3.2, 80 x 32
// 4.2 -> 4.0, 64 x 40 4.2 -> 4.0, 45 x 52 4.3 -> 4.0, 320 x 8 4.2 -> 4.0, 320 x 8 of
// 64 8.8 -> 7.4; beyond the line prompts lose (128 x 32 4.7 -> 4.8, 512 x 32 8.0 ->
// 12.0), though decode goes on winning (256 x 32 23.0 -> 21.7).
constexpr int64_t kScatterPairs = 2560;

// From this many pairs on of kv heads with one query head each (and most pairs of
// the call being such), the window kernel requests the query rows early.  It takes
// 88 registers instead of 74 for that: five waves per SIMD instead of six, which
// pays where the rows come from memory.  Below the line they are what the projection
// has just left in the last-level cache (256 MB; q, k, v and pool lines of 262144
// pairs are 336 MB).  us, late -> early, f16, rows in that cache | in memory, prompts
// of two and three models: 83808 pairs 27.9 -> 29.7 | 39.5 -> 37.3, 226780 64.7 ->
// 65.3 | 90.5 -> 88.3, 340376 129.8 -> 128.5 | 131.1 -> 127.1, 829392 300.8 -> 290.2.
// With more query heads per kv head the registers are for nothing (64 / 8 heads,
// three prompts of 700 - 2000 tokens 41.0 -> 42.2; 16 / 4 heads, 2 x 2000 11.5 ->
// 12.3).
constexpr int64_t kEarlyQPairs = 262144;

hipError_t launch_rope_scatter(MultiCacheWriteParams &P, int32_t dtype, hipStream_t st) {
  int64_t work = 0;
  for (int i = 0; i < P.n_items; ++i) {
    CacheWriteItemDev &d = P.it[i];
    const int per_kv = d.rope.q != nullptr ? d.rope.ratio + 1 : 1;
    const int64_t rows = static_cast<int64_t>(d.num_kv_heads) * per_kv;
    // Eight rows to a workgroup (w runs on XCD w % 8: a model takes multiples of 8).
    // Packed token after token, a head's tokens come to one XCD where a token's rows
    // are a multiple of 64 and wander over the XCDs otherwise; the tokens of a prompt
    // then write their two bytes of a V line in different L2s (45 tokens x 52 heads
    // 5.4 us, the window kernel 4.3), unless query rows thin out the stores (64 query
    // heads on 8, where packed decode is 3 % faster).  Else eight rows of one token
    // per workgroup, and the workgroups of the same eight rows on one XCD or on two
    // neighbouring ones: 45 x 52 4.0 us, 64 tokens x 40 heads 4.9 -> 4.0.
    const bool packed = per_kv > 2 || rows % 64 == 0;
    d.per_xcd = packed ? 0 : static_cast<int32_t>(((rows + 7) / 8 * d.num_tokens + 7) / 8);
    d.work_begin = static_cast<int32_t>(work);
    work += 8 * (packed ? (d.num_tokens * rows + 63) / 64 : static_cast<int64_t>(d.per_xcd));
  }
  const dim3 grid(static_cast<unsigned>(work));
  if (dtype == MUXA_DTYPE_F16) hipLaunchKernelGGL(rope_scatter_kernel<F16>, grid, dim3(256), 0, st, P);
  else hipLaunchKernelGGL(rope_scatter_kernel<BF16>, grid, dim3(256), 0, st, P);
  return hipGetLastError();
}

}  // namespace
}  // namespace mux

extern "C" int32_t mux_reshape_and_cache(const void *k, const void *v, int64_t kv_row_stride,
                                         void *k_pool, void *v_pool, int64_t num_pool_blocks,
                                         const int64_t *slot_mapping, int32_t layer, int32_t num_layers,
                                         int32_t num_tokens, int32_t num_kv_heads, int32_t head_size,
                                         int32_t block_size, int32_t dtype, void *stream) {
  using namespace mux;
  const int32_t rc = check_cache_write(k, v, kv_row_stride, k_pool, v_pool, num_pool_blocks, slot_mapping, layer,
                                       num_layers, num_tokens, num_kv_heads, head_size, block_size, dtype);
  if (rc != MUXA_OK) return rc;
  if (num_tokens == 0) return MUXA_OK;
  const int64_t slot_stride = static_cast<int64_t>(num_layers) * num_kv_heads;
  const int64_t *slots = slot_mapping + static_cast<int64_t>(layer) * num_kv_heads;
  dim3 grid(num_kv_heads, (num_tokens + 15) / 16);
  // Without the rotary part the kernel only moves bytes and never writes k.
  hipLaunchKernelGGL((reshape_and_cache_kernel<F16, false, false>), grid, dim3(256), 0, static_cast<hipStream_t>(stream),
                     const_cast<uint16_t *>(static_cast<const uint16_t *>(k)), static_cast<const uint16_t *>(v),
                     kv_row_stride, static_cast<uint4 *>(k_pool), static_cast<uint16_t *>(v_pool), num_pool_blocks,
                     slots, slot_stride, num_tokens, block_size, RopeArgs{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e);
  return MUXA_OK;
}

extern "C" int32_t mux_rope_reshape_and_cache(const int64_t *positions, void *q, int64_t q_row_stride, void *k,
                                              const void *v, int64_t kv_row_stride, const float *cos_sin,
                                              int32_t max_position, int32_t rotary_dim, void *k_pool, void *v_pool,
                                              int64_t num_pool_blocks, const int64_t *slot_mapping, int32_t layer,
                                              int32_t num_layers, int32_t num_tokens, int32_t num_q_heads,
                                              int32_t num_kv_heads, int32_t head_size, int32_t block_size,
                                              int32_t dtype, void *stream) {
  using namespace mux;
  const int32_t rc = check_cache_write(k, v, kv_row_stride, k_pool, v_pool, num_pool_blocks, slot_mapping, layer,
                                       num_layers, num_tokens, num_kv_heads, head_size, block_size, dtype);
  if (rc != MUXA_OK) return rc;
  if ((num_tokens > 0 && (!positions || !cos_sin)) || max_position <= 0) return MUXA_EINVAL;
  if (rotary_dim != kHeadSize) return MUXA_EUNSUPPORTED;   // partial rotation: use mux_rotary_neox + mux_reshape_and_cache
  if (q != nullptr) {
    if (num_q_heads <= 0 || num_q_heads % num_kv_heads != 0) return MUXA_EINVAL;
    if (q_row_stride < static_cast<int64_t>(num_q_heads) * kHeadSize || q_row_stride % 8 != 0) return MUXA_EINVAL;
    if (reinterpret_cast<uintptr_t>(q) & 15u) return MUXA_EINVAL;
  }
  if (num_tokens == 0) return MUXA_OK;
  const int64_t slot_stride = static_cast<int64_t>(num_layers) * num_kv_heads;
  const int64_t *slots = slot_mapping + static_cast<int64_t>(layer) * num_kv_heads;
  RopeArgs R;
  R.q = static_cast<uint16_t *>(q);
  R.q_stride = q_row_stride;
  R.ratio = q ? num_q_heads / num_kv_heads : 0;
  R.positions = positions;
  R.cos_sin = cos_sin;
  R.max_position = max_position;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t pairs = static_cast<int64_t>(num_tokens) * num_kv_heads;
  if (pairs <= kScatterPairs) {
    MultiCacheWriteParams P = {};
    P.it[0] = {static_cast<uint16_t *>(k), static_cast<const uint16_t *>(v), kv_row_stride, slots, slot_stride, R,
               num_tokens, num_kv_heads, 0, 0};
    P.k_pool = static_cast<uint4 *>(k_pool);
    P.v_pool = static_cast<uint16_t *>(v_pool);
    P.num_blocks = num_pool_blocks;
    P.n_items = 1;
    P.block_size = block_size;
    const hipError_t e = launch_rope_scatter(P, dtype, st);
    return e == hipSuccess ? MUXA_OK : hip_fail(e);
  }
  dim3 grid(num_kv_heads, (num_tokens + 15) / 16);
  const bool early_q = R.ratio == 1 && pairs >= kEarlyQPairs;
  const auto kernel =
      dtype == MUXA_DTYPE_F16
          ? (early_q ? reshape_and_cache_kernel<F16, true, true> : reshape_and_cache_kernel<F16, true, false>)
          : (early_q ? reshape_and_cache_kernel<BF16, true, true> : reshape_and_cache_kernel<BF16, true, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, static_cast<uint16_t *>(k), static_cast<const uint16_t *>(v),
                     kv_row_stride, static_cast<uint4 *>(k_pool), static_cast<uint16_t *>(v_pool), num_pool_blocks, slots,
                     slot_stride, num_tokens, block_size, R);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e);
  return MUXA_OK;
}

extern "C" int32_t mux_multi_rope_reshape_and_cache(const MuxCacheWriteItem *items, int32_t n_items, void *k_pool,
                                                    void *v_pool, int64_t num_pool_blocks, int32_t head_size,
                                                    int32_t block_size, int32_t dtype, void *stream) {
  using namespace mux;
  if (!items || n_items <= 0 || n_items > MUXA_MAX_DECODE_ITEMS) return MUXA_EINVAL;
  MultiCacheWriteParams P = {};
  P.k_pool = static_cast<uint4 *>(k_pool);
  P.v_pool = static_cast<uint16_t *>(v_pool);
  P.num_blocks = num_pool_blocks;
  P.block_size = block_size;
  // Either every model of the call that has tokens rotates (positions given) or none does.
  bool rope = false;
  for (int i = 0; i < n_items; ++i)
    if (items[i].num_tokens > 0) {
      rope = items[i].positions != nullptr;
      break;
    }
  int64_t work = 0;
  for (int i = 0; i < n_items; ++i) {
    const MuxCacheWriteItem &it = items[i];
    const int32_t rc = check_cache_write(it.k, it.v, it.kv_row_stride, k_pool, v_pool, num_pool_blocks,
                                         it.slot_mapping, it.layer, it.num_layers, it.num_tokens, it.num_kv_heads,
                                         head_size, block_size, dtype);
    if (rc != MUXA_OK) return rc;
    if (it.num_tokens > 0 && (it.positions != nullptr) != rope) return MUXA_EINVAL;
    RopeArgs R{};
    if (rope && it.num_tokens > 0) {
      if ((it.num_tokens > 0 && !it.cos_sin) || it.max_position <= 0) return MUXA_EINVAL;
      if (it.rotary_dim != kHeadSize) return MUXA_EUNSUPPORTED;
      if (it.q != nullptr) {
        if (it.num_q_heads <= 0 || it.num_q_heads % it.num_kv_heads != 0) return MUXA_EINVAL;
        if (it.q_row_stride < static_cast<int64_t>(it.num_q_heads) * kHeadSize || it.q_row_stride % 8 != 0)
          return MUXA_EINVAL;
        if (reinterpret_cast<uintptr_t>(it.q) & 15u) return MUXA_EINVAL;
      }
      R.q = static_cast<uint16_t *>(it.q);
      R.q_stride = it.q_row_stride;
      R.ratio = it.q ? it.num_q_heads / it.num_kv_heads : 0;
      R.positions = it.positions;
      R.cos_sin = it.cos_sin;
      R.max_position = it.max_position;
    }
    if (it.num_tokens == 0) continue;
    CacheWriteItemDev &d = P.it[P.n_items++];
    d.k = static_cast<uint16_t *>(it.k);
    d.v = static_cast<const uint16_t *>(it.v);
    d.row_stride = it.kv_row_stride;
    d.slots = it.slot_mapping + static_cast<int64_t>(it.layer) * it.num_kv_heads;
    d.slot_stride = static_cast<int64_t>(it.num_layers) * it.num_kv_heads;
    d.rope = R;
    d.num_tokens = it.num_tokens;
    d.num_kv_heads = it.num_kv_heads;
    d.work_begin = static_cast<int32_t>(work);
    work += static_cast<int64_t>((it.num_tokens + 15) / 16) * it.num_kv_heads;
    if (work > 0x7fffffff) return MUXA_EUNSUPPORTED;
  }
  if (P.n_items == 0) return MUXA_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  int64_t pairs = 0, one_q_pairs = 0;
  for (int i = 0; i < P.n_items; ++i) {
    const int64_t n = static_cast<int64_t>(P.it[i].num_tokens) * P.it[i].num_kv_heads;
    pairs += n;
    if (P.it[i].rope.ratio == 1) one_q_pairs += n;
  }
  const bool early_q = one_q_pairs >= kEarlyQPairs && one_q_pairs > pairs / 2;
  if (rope && pairs <= kScatterPairs) {
    const hipError_t e = launch_rope_scatter(P, dtype, st);
    return e == hipSuccess ? MUXA_OK : hip_fail(e);
  }
  const dim3 grid(static_cast<unsigned>(work));
  const auto kernel =
      !rope ? multi_reshape_and_cache_kernel<F16, false, false>
      : dtype == MUXA_DTYPE_F16
          ? (early_q ? multi_reshape_and_cache_kernel<F16, true, true> : multi_reshape_and_cache_kernel<F16, true, false>)
          : (early_q ? multi_reshape_and_cache_kernel<BF16, true, true> : multi_reshape_and_cache_kernel<BF16, true, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, P);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e);
  return MUXA_OK;
}
