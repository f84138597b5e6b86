// Causal prefill attention on the fresh q, k, v of a batch of packed prompts,
// gfx950 MFMA (v_mfma_f32_32x32x16_{f16,bf16}).
//
// One workgroup = 128 query rows of one head of one prompt, 4 waves x 32 rows.
// Keys/values stream through LDS in tiles of 32 tokens shared by the 4 waves
// (32 rather than 64: 160 VGPRs and 34 KB of LDS let three workgroups share a
// CU instead of two, and the causal edge is cut at 32 keys; measured 8 %
// faster on ragged short prompts, 1 - 3 % on 2048-token prompts).
// Each wave keeps the TRANSPOSED problem so that probabilities never leave
// registers:
//     S^T[key][q] = K . Q^T      A = K tile   (LDS, row-major, 16-byte frags)
//                                B = Q^T      (registers, loaded once)
//     O^T[d][q]  += V^T . P^T    A = V^T      (the row-major V tile in LDS, read
//                                              with the transposing LDS read)
//                                B = P^T      = the S^T accumulators, converted
// In the 32x32 accumulator layout a lane owns ONE query column (q = lane%32)
// and 16 of the 32 keys of a block, so softmax statistics are per-lane scalars
// (one exchange with lane^32), the rescale of O^T is a per-lane multiply, and
// the accumulator registers of S^T are, in order, exactly the 8-element
// B-operand fragments of the P.V products - provided the V^T fragments use the
// same key order (two groups of four keys), which costs nothing because V^T is
// read from LDS anyway.
// The next tile's global loads are issued before the current tile's math.
//
// What bounds it: power.  With every CU busy the clock settles at 1.6 GHz; on half
// of the CUs 16 x 2048 tokens take 0.67 of the whole chip's CU time, on a quarter
// 0.63.  So what counts is work per score, in any unit: no maximum where the sum
// tells as much (attention of that shape 604 -> 588 us), fragment addresses that
// are registers or immediates (the tile loop is unrolled over its two buffers),
// waits for exactly the loads that are needed, two stores and no address
// arithmetic per 16 tokens for the pool (the step form 813 -> 793 us).  Fragments of
// V^T requested before the softmax, a third tile buffer, two chains of sums: no
// difference.
//
// The step form (STEP = true, mux_rope_prefill_and_cache) is a whole prompt step
// of the attention layer behind the rotation of k: it also rotates q and writes
// k and v to the pool.  As kernels of their own these passes are bound by
// memory and run 1:1 beside an attention that leaves the memory idle - at
// 16 x 2048 tokens, 32 heads: rotation of q and k 193 us, cache write 248 us,
// attention 600 us.  Here the query fragments are rotated in the registers they
// are loaded into (one workgroup reads each of them once; a lane holds both
// halves of a pair), and a workgroup scatters the 128 rows of K and V that its
// last four tiles bring into LDS anyway, so k and v are not read again and the
// stores go out under the matrix work.  Measured, whole step, both sides in turn
// on one machine: 16 x 2048 tokens f16 1052 -> 800 us (rotation of k 100, attention
// by itself 600, pool stores 55, rotation of q 45), three bf16 prompts of 700 - 4000
// tokens on 64 / 8 heads 548 -> 490 us.  Prompts of a few tokens lose in this form:
// 128 of 6 tokens, 32 heads, 47 us against 34 with rotation and cache write in a
// launch of their own, and 29.5 in the short form (SHORT, below), which one launch
// is: it waits for one chain of loads instead of two and reads k once; 16 prompts
// of 100 tokens, 32 heads, 30 -> 21 us, 64 of 128 101 -> 90.
#include "../prompt_step.h"
#include "cache_write.h"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace mux {

typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf16 __attribute__((ext_vector_type(8)));
typedef float v16f32 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBM = 128;                 // query rows per workgroup
constexpr int kBN = 32;                  // keys per tile (one MFMA row block)

// Query tiles listed in the kernel argument (its size limit is 4 KiB).
constexpr int kMaxPairs = 768;

// Tracing build (-DMUX_TRACE, libmuxattn_trace.so; never the shipped library):
// thread 0 of every workgroup that has work stamps the 100 MHz clock into a
// caller-provided table, 8 int64 per workgroup: [0] entry, [1] the prompt's
// place and length known, [2] first key tile landed and the workgroup met (end
// of the prologue), [3] last key tile done, [4] output stores issued (a wave
// does not wait for them before it ends, and neither does the stamp), [5] key
// tiles of the workgroup, [6] prompt length, [7] first query row.
#ifdef MUX_TRACE
__device__ long long *g_prefill_trace = nullptr;
__device__ long long g_prefill_trace_rows = 0;
#endif

union Frag {
  u32x4 u;
  v8f16 h;
  v8bf16 b;
};

template <typename T>
__device__ __forceinline__ v16f32 mfma(const Frag &a, const Frag &b, v16f32 c) {
  if constexpr (__is_same(T, F16)) return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, b.h, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
}

// Two fp32 -> one packed pair in storage type T, round to nearest even
// (one v_cvt_pk_f16_f32 / v_cvt_pk_bf16_f32).
typedef float float2_t __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const float2_t x = {lo, hi};
  if constexpr (__is_same(T, F16)) {
    union { half2_t h; uint32_t u; } c;
    c.h = __builtin_convertvector(x, half2_t);
    return c.u;
  } else {
    union { bf162_t h; uint32_t u; } c;
    c.h = __builtin_convertvector(x, bf162_t);
    return c.u;
  }
}

// One model's prompts (several colocated models can share a launch).
struct PrefillItemDev {
  uint16_t *out;
  const uint16_t *q, *k, *v;
  int64_t out_stride, q_stride, kv_stride;
  const int32_t *cu_seqlens;
  int32_t ratio;          // query heads per kv head
  int32_t num_kv_heads;
  int32_t num_prompts;
  int32_t kv_per_xcd;     // ceil(num_kv_heads / 8)
  float scale_log2;
  int32_t out_rows_16b;   // out and its row stride allow 16-byte stores
};

struct PrefillParams {
  PrefillItemDev it[MUXA_MAX_DECODE_ITEMS];
  const int32_t *prompt_order;   // dense grid, optional: prompts in the order their workgroups should start
  int32_t q_tiles;        // dense grid: 128-row query tiles per prompt (of the longest prompt)
  int32_t num_groups;     // dense grid: (prompt, kv head) pairs
  // Compact grid (the caller gave the prompt lengths on the host): the query
  // tiles that exist, the heaviest of all models first, as
  // model << 28 | prompt << 12 | tile; every pair takes slots_per_pair workgroups
  // on each XCD (the largest model's kv heads per XCD x query heads per kv head;
  // the surplus of smaller models leaves at once).  0 pairs = dense grid, one model.
  int32_t n_pairs;
  int32_t slots_per_pair;
  uint32_t pairs[kMaxPairs];
};

// The step form's part: one model's rotation and cache write.
struct PrefillStep {
  const int64_t *positions;
  const float *cos_sin;          // [max_position, 128] = [cos | sin]
  const int64_t *slots;          // layer slice of the slot mapping
  int64_t slot_stride;
  uint16_t *k_pool, *v_pool;
  int64_t pool_slots;
  int32_t max_position;
  int32_t block_size;
  int32_t short_waves;           // the host's choice of kernel: W of the short form, or 0
};
static_assert(sizeof(PrefillParams) + sizeof(PrefillStep) <= 4096, "kernel argument segment");
constexpr int kPairTileBits = 12;       // tile in bits 0-11, prompt in bits 12-27, model in bits 28-30

// K and V tiles go from global memory straight into LDS
// (global_load_lds_dwordx4: lane l's 16 bytes land at base + 16 l), row-major
// [key][128 dims] with the 16-byte chunks of a row XOR-swizzled by the row
// number so that fragment reads spread over the banks; V^T fragments come out of
// the row-major tile with the transposing read ds_read_b64_tr_b16.  No staging
// registers, no LDS stores, no byte permutes; two tile buffers per operand, one
// barrier per tile.
typedef short v4i16 __attribute__((ext_vector_type(4)));
// A wave raises its issue priority while it feeds the matrix cores and drops
// it for the softmax, so that of the two waves of a SIMD the one in its MFMA
// phase goes first (1 - 5 % on prompts of 1024 - 2048 tokens).
#define MUX_PF_PRIO(x) __builtin_amdgcn_s_setprio(x)
#define MUX_PF_PRIO_MFMA 1
#define MUX_PF_PRIO_VALU 0
constexpr int kTileElems = kBN * kHeadSize;          // one unpadded row-major tile
// The swizzle: the 16-byte chunk c of tile row r sits at chunk position
// c ^ swz(r), swz(r) = the low three bits of r rotated left by one.  LDS has 32
// banks of 4 bytes: a 256-byte row covers them twice, so only the low three bits
// of a chunk position choose the banks, and bit 3 of a chunk is left alone, an
// immediate offset of the reads.  The K fragments are read 8 rows at a time (one
// chunk each, ds_read_b128): the rotated bits of 8 consecutive rows are all
// different.  The V^T fragments are read 16 lanes at a time (ds_read_b64_tr_b16)
// over 4 consecutive rows x 2 neighbouring chunks x the two halves of a chunk: the
// rows' two low bits land in position bits 1-2 and the chunk pair in bit 0 - again
// all different.  (With the plain c ^ r the four rows and the chunk pair shared two
// position bits: a two-way conflict on every V^T read.)
__device__ __forceinline__ int swz(int row) { return ((row & 3) << 1) | ((row >> 2) & 1); }

// 16 tokens (rows row0 .. row0 + 15 of the K and V tile in LDS) to the pool, by
// the four waves of a workgroup together.  slot_at: LDS address of row0's slot, -1
// for none.  K: a thread stores one token's chunk, the 16 tokens of a chunk
// side by side, so a wave fills 1 KiB of a 16-token block.  V: the transposing
// read hands a lane 8 consecutive tokens of one dim, which is a chunk of the pool
// where those tokens are a run (consecutive slots from a multiple of 8: every
// prompt behind a block table, up to its last few tokens); the others go element
// by element.  The LDS reads are written out with their wait: for a transposing
// read of its own the compiler first waits for every load in flight, the next
// tile's among them.
// True if exactly two vector-memory instructions were issued (both 8-token
// halves are runs): the caller's wait for older loads can then leave them.
__device__ __forceinline__ bool write_tokens_to_pool(const uint16_t *Kt, const uint16_t *Vr, int row0, uint32_t slot_at,
                                                     int wave, int lane, const PrefillStep &S) {
  constexpr int D = kHeadSize;
  // (kept from the tile loop's registers: the compiler would hoist the addresses
  // below out of it and spill)
  asm volatile("" : "+v"(lane));
  typedef const __attribute__((address_space(3))) uint16_t lds_u16;
  const int bs = S.block_size, bs_shift = __builtin_ctz(static_cast<unsigned>(bs));
  const int i = lane & 15, c = 4 * wave + (lane >> 4);      // this thread's token and chunk (8 dims)
  const int kr = row0 + i;
  // Group of 16 lanes: dims 8 c .. 8 c + 7 of both halves.  Lane 4 j + m points at
  // four dims (m & 1) of token j (and j + 4) of half m >> 1, and receives dim
  // lane % 8 of half (lane / 8) % 2.
  const int j = i >> 2, m = i & 3;
  const int r0 = row0 + 8 * (m >> 1) + j, r1 = r0 + 4;
  const uint32_t ka = (uint32_t)(uintptr_t)(lds_u16 *)(Kt + kr * D + 8 * (c ^ swz(kr)));
  const uint32_t va0 = (uint32_t)(uintptr_t)(lds_u16 *)(Vr + r0 * D + 8 * (c ^ swz(r0)) + 4 * (m & 1));
  const uint32_t va1 = (uint32_t)(uintptr_t)(lds_u16 *)(Vr + r1 * D + 8 * (c ^ swz(r1)) + 4 * (m & 1));
  u32x4 kx;
  u32x2 v0, v1;
  int64_t slot;
  asm volatile("ds_read_b64 %3, %7\n\tds_read_b128 %0, %4\n\tds_read_b64_tr_b16 %1, %5\n\t"
               "ds_read_b64_tr_b16 %2, %6\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(kx), "=&v"(v0), "=&v"(v1), "=&v"(slot)
               : "v"(ka), "v"(va0), "v"(va1), "v"(slot_at + 8u * i)
               : "memory");
  // Runs: the previous lane's slot plus one, from a multiple of 8.
  const uint32_t slot_lo = static_cast<uint32_t>(slot), slot_hi = static_cast<uint32_t>(slot >> 32);
  const uint32_t prev_lo = __builtin_amdgcn_update_dpp(0, slot_lo, 0x111, 0xf, 0xf, true);      // row_shr:1
  const uint32_t prev_hi = __builtin_amdgcn_update_dpp(0, slot_hi, 0x111, 0xf, 0xf, true);
  const int64_t prev = static_cast<int64_t>((static_cast<uint64_t>(prev_hi) << 32) | prev_lo);
  const bool chained = slot >= 0 && ((lane & 7) == 0 ? (slot & 7) == 0 : slot == prev + 1);
  const uint32_t runs = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(chained));
  const bool run_a = (runs & 0xff) == 0xff, run_b = (runs & 0xff00) == 0xff00;      // (the four groups agree)
  auto slot_of = [&](int l) {
    const uint32_t lo = __builtin_amdgcn_readlane(slot_lo, l), hi = __builtin_amdgcn_readlane(slot_hi, l);
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
  };
  const int64_t a = slot_of(0), b = slot_of(8), base = i < 8 ? a : b;
  const int d = 8 * c + (lane & 7);
  uint16_t *const kp = S.k_pool + (((slot >> bs_shift) * (D / 8) + c) * bs + (slot & (bs - 1))) * 8;
  uint16_t *const vp = S.v_pool + ((base >> bs_shift) * D + d) * bs + (base & (bs - 1));
  const u32x4 vx = {v0.x, v0.y, v1.x, v1.y};
  if (run_a && run_b) {
    // (K rows are whole lines; V rows are where the halves fill the block's rows:
    // those stream past the L2, as in the cache-write kernel, and the wait states
    // between a 16-byte store and a write of its data are spelled out as there)
    asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 4" ::"v"(kp), "v"(kx) : "memory");
    if (bs == 8 || (bs == 16 && b == a + 8 && (a & 15) == 0))
      asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 4" ::"v"(vp), "v"(vx) : "memory");
    else
      asm volatile("global_store_dwordx4 %0, %1, off\n\ts_nop 4" ::"v"(vp), "v"(vx) : "memory");
    return true;
  }
  if (slot >= 0) *reinterpret_cast<u32x4 *>(kp) = kx;
  if (i < 8 ? run_a : run_b) {
    *reinterpret_cast<u32x4 *>(vp) = vx;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t sa = slot_of(e), sb = slot_of(8 + e), sl = i < 8 ? sa : sb;
      if (sl >= 0)
        S.v_pool[((sl >> bs_shift) * D + d) * bs + (sl & (bs - 1))] =
            static_cast<uint16_t>(vx[e >> 1] >> (16 * (e & 1)));
    }
  }
  return false;
}

// What a lane keeps for writing 16 tokens that fill (part of) one pool block in
// order, chunk c = 4 wave + lane / 16: LDS offsets of its K chunk and of its two V
// reads (see write_tokens_to_pool) in a tile, and its places in a K and V block.
struct BlockWriter {
  uint32_t k_lds, v_lds0, v_lds1, k_off, v_off;
  __device__ __forceinline__ BlockWriter(int wave, int lane, int bs) {
    constexpr int D = kHeadSize;
    const int i = lane & 15, c = 4 * wave + (lane >> 4), j = i >> 2, m = i & 3;
    const int r0 = 8 * (m >> 1) + j, r1 = r0 + 4;
    k_lds = 2 * (i * D + 8 * (c ^ swz(i)));
    v_lds0 = 2 * (r0 * D + 8 * (c ^ swz(r0)) + 4 * (m & 1));
    v_lds1 = 2 * (r1 * D + 8 * (c ^ swz(r1)) + 4 * (m & 1));
    k_off = 16 * (c * bs + i);
    v_off = 2 * ((8 * c + (lane & 7)) * bs + 8 * (i >> 3));
  }
};

// The first n of 16 rows of the tile (K at kt, V at vt, LDS addresses) to the n slots
// from `base`, a multiple of 16, of one block.  True if that took exactly two stores.
__device__ __forceinline__ bool write_block_to_pool(uint32_t kt, uint32_t vt, const BlockWriter &w, int64_t base, int n,
                                                    int lane, const PrefillStep &S) {
  constexpr int D = kHeadSize;
  u32x4 kx;
  u32x2 v0, v1;
  asm volatile("ds_read_b128 %0, %3\n\tds_read_b64_tr_b16 %1, %4\n\tds_read_b64_tr_b16 %2, %5\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(kx), "=&v"(v0), "=&v"(v1)
               : "v"(kt + w.k_lds), "v"(vt + w.v_lds0), "v"(vt + w.v_lds1)
               : "memory");
  const u32x4 vx = {v0.x, v0.y, v1.x, v1.y};
  const int bs_shift = __builtin_ctz(static_cast<unsigned>(S.block_size));
  const int64_t first = (base >> bs_shift) * (D << bs_shift);           // the block's first element
  const int64_t in_block = base & (S.block_size - 1);
  uint16_t *const kp = S.k_pool + first + 8 * in_block, *const vp = S.v_pool + first + in_block;
  if (n == 16) {
    // (as in write_tokens_to_pool: whole lines stream past the L2)
    asm volatile("global_store_dwordx4 %0, %1, %2 nt\n\ts_nop 4" ::"v"(w.k_off), "v"(kx), "s"(kp) : "memory");
    if (S.block_size == 16) asm volatile("global_store_dwordx4 %0, %1, %2 nt\n\ts_nop 4" ::"v"(w.v_off), "v"(vx), "s"(vp) : "memory");
    else asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 4" ::"v"(w.v_off), "v"(vx), "s"(vp) : "memory");
    return true;
  }
  if ((lane & 15) < n) *reinterpret_cast<u32x4 *>(reinterpret_cast<char *>(kp) + w.k_off) = kx;
  // V: this lane's 8 tokens of a dim, as many as there are, in pieces of 8, 4, 2 and 1.
  const int mine = n - (lane & 8);
  uint16_t *const v = reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(vp) + w.v_off);
  if (mine >= 8) {
    *reinterpret_cast<u32x4 *>(v) = vx;
  } else if (mine > 0) {
    const bool four = mine & 4;
    if (four) *reinterpret_cast<u32x2 *>(v) = u32x2{vx[0], vx[1]};
    const uint32_t next = four ? vx[2] : vx[0], last = four ? vx[3] : vx[1];
    uint16_t *const rest = v + (four ? 4 : 0);
    if (mine & 2) *reinterpret_cast<uint32_t *>(rest) = next;
    if (mine & 1) rest[mine & 2] = static_cast<uint16_t>((mine & 2) ? last : next);
  }
  return false;
}

// SHORT = W > 0: the step of prompts of at most 32 W tokens (W = 1, 2, 4) with as
// many kv heads as query heads, by workgroups of W waves.  A workgroup then holds all
// of a (prompt, head): it rotates k as well, in the registers its waves load their 32
// rows into, and the whole of K and V (W tiles each) sits in LDS, so that one launch
// does the step and its tile loop has one barrier in front of it.
template <typename T, bool STEP, int SHORT = 0>
__device__ __forceinline__ void prefill_body(const PrefillParams &P, const PrefillStep &S) {
  constexpr int D = kHeadSize;
  constexpr int W = SHORT > 0 ? SHORT : 4;     // waves
  constexpr int kRows = 32 * W;                // query rows
  // K[2], V[2] tile buffers (SHORT: W of each).  The epilogue reuses the memory for
  // the output rows (W waves x 32 rows of 272 bytes).
  constexpr int NBUF = SHORT > 0 ? W : 2;
  constexpr int kSmemElems =
      SHORT > 0 ? 2 * W * kTileElems + 4 * (kRows + kRows / 16) : std::max(4 * kTileElems, 4 * 32 * (D + 8));
  __shared__ __attribute__((aligned(16))) uint16_t smem[kSmemElems];

#ifdef MUX_TRACE
  const long long tr_entry = __builtin_amdgcn_s_memrealtime();
  long long tr_first = 0;
  long long *const tr_table = g_prefill_trace;   // read here, so that the write at the end waits for nothing
  const long long tr_rows = g_prefill_trace_rows;
#endif
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups are dealt to the 8 XCDs round-robin by id, and each XCD has its
  // own L2.  All workgroups that read the same K/V - the query tiles and query
  // heads of one (prompt, kv head) pair - are therefore given ids that are equal
  // mod 8.
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  int item = 0, prompt, hk, hq, q0, rem = 0;
  uint32_t pair = 0;
  if (P.n_pairs > 0) {
    // Compact grid: only query tiles that exist, the heaviest of the whole launch first.
    const int pi = slot / P.slots_per_pair;
    if (pi >= P.n_pairs) return;
    rem = slot - pi * P.slots_per_pair;
    pair = P.pairs[pi];
    item = min(static_cast<int>(pair >> 28), MUXA_MAX_DECODE_ITEMS - 1);
  }
  const PrefillItemDev I = P.it[item];
  if (P.n_pairs > 0) {
    // kv head hk of prompt p lives on XCD (hk + p) % 8 (rotated by the prompt so
    // that head counts that are no multiple of 8 load the XCDs evenly).
    if (rem >= I.kv_per_xcd * I.ratio) return;
    // (clamped: a malformed list costs results, never a stray read)
    prompt = min(static_cast<int>((pair >> kPairTileBits) & 0xffffu), I.num_prompts - 1);
    q0 = static_cast<int>(pair & ((1u << kPairTileBits) - 1)) * kBM;
    hk = ((xcd - prompt) & 7) + 8 * (rem / I.ratio);
    if (hk >= I.num_kv_heads) return;
    hq = hk * I.ratio + rem % I.ratio;
  } else {
    // Dense grid: every prompt gets the tiles of the longest one, heaviest first;
    // (prompt, kv head) groups go round-robin over the XCDs.
    const int per_group = I.ratio * P.q_tiles;
    const int group = (slot / per_group) * 8 + xcd;
    if (group >= P.num_groups) return;
    const int in_group = slot % per_group;
    const int prompt_rank = group / I.num_kv_heads;
    // (an entry outside the batch is clamped, as above)
    prompt = P.prompt_order ? min(max(P.prompt_order[prompt_rank], 0), I.num_prompts - 1) : prompt_rank;
    hk = group % I.num_kv_heads;
    hq = hk * I.ratio + in_group / P.q_tiles;
    q0 = (P.q_tiles - 1 - in_group % P.q_tiles) * kBM;
  }
  const int seq_begin = I.cu_seqlens[prompt];
  const int len = I.cu_seqlens[prompt + 1] - seq_begin;
  if (q0 >= len) return;
#ifdef MUX_TRACE
  asm volatile("s_nop 0" ::"s"(len));    // (the stamp waits for the loads of the two offsets)
  const long long tr_len = __builtin_amdgcn_s_memrealtime();
#endif

  const int qcol = lane & 31;            // this lane's query column / fragment row
  const int half = lane >> 5;            // which 8 of a fragment's 16 k-slots
  const int wq0 = q0 + wave * 32;        // first query row of this wave
  const int my_q = wq0 + qcol;           // this lane's query position inside the prompt

  // The query heads of a kv head share its K and V: the one whose turn it is by
  // the query tile writes them (each writes as many tiles as the others).
  bool writes_pool = false;
  if constexpr (STEP) writes_pool = hq - hk * I.ratio == (q0 / kBM) % I.ratio;

  // ---- Q^T fragments: Q[my_q][16 s + 8 half .. +7], s = 0..7 ------------------------
  Frag qf[8];
  if constexpr (!STEP) {
    const bool ok = my_q < len;
    const uint16_t *qp = I.q + static_cast<int64_t>(seq_begin + (ok ? my_q : 0)) * I.q_stride + hq * D + 8 * half;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s].u = ok ? *reinterpret_cast<const u32x4 *>(qp + 16 * s) : u32x4{0, 0, 0, 0};
  }

  v16f32 oacc[4];                        // O^T[d = 32 mb + ...][q]
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[mb][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  float neg_m = 0.f;                     // the reference as an exponent, kept beside m_run and changed with it

  // Keys needed by this workgroup: positions 0 .. min(len, q0 + 128) - 1.
  const int kv_end = min(len, q0 + kRows);
  const int n_tiles = (kv_end + kBN - 1) / kBN;

  // ---- tile staging -------------------------------------------------------------------
  const uint32_t row_bytes = static_cast<uint32_t>(I.kv_stride) * 2u;
  const char *kbase = reinterpret_cast<const char *>(I.k + static_cast<int64_t>(seq_begin) * I.kv_stride + hk * D);
  const char *vbase = reinterpret_cast<const char *>(I.v + static_cast<int64_t>(seq_begin) * I.kv_stride + hk * D);
  const uint32_t tile_bytes = kBN * row_bytes;
  const uint32_t last_row = static_cast<uint32_t>(len - 1) * row_bytes;
  // Rows past the prompt re-read its last row: finite data whose probability is
  // exactly 0 (such a key is in the future of every valid query).

  // Instruction i of wave w fills KiB W i + w of a tile = rows 4 (W i + w) .. +3;
  // lane l sits at row 4 (W i + w) + l/16, position l%16, and fetches chunk
  // position ^ swz(row) - with W > 1 the same for every i (rows 8 apart swizzle alike).
  constexpr int kLoads = kBN / (4 * W);    // such instructions per wave, tile and operand
  uint32_t koff[kLoads];
  const int row0 = 4 * wave + (lane >> 4);
  auto chunk_of = [&](int i) { return static_cast<uint32_t>((lane & 15) ^ swz(row0 + 4 * W * i)); };
#pragma unroll
  for (int i = 0; i < kLoads; ++i) koff[i] = static_cast<uint32_t>(row0 + 4 * W * i) * row_bytes + 16u * chunk_of(i);
  typedef const __attribute__((address_space(3))) uint16_t lds_u16;
  const uint32_t smem_at = (uint32_t)(uintptr_t)(lds_u16 *)smem;
  // The loads are written out (they have no destination registers), with the waits
  // for them in the loop: after a load to LDS of its own the compiler takes every
  // LDS access to be out of order, so that it waits for all fragments before the
  // first MFMA and for the next tile's loads before the V^T fragments (the step of
  // 16 x 2048 tokens 4 %, three bf16 prompts 3 % slower).
  auto dma_tile = [&](int t, int buf) {    // tile t into buffer buf
    const char *const kt = kbase + static_cast<uint64_t>(t) * tile_bytes, *const vt = vbase + static_cast<uint64_t>(t) * tile_bytes;
    const bool whole = (t + 1) * kBN <= len;
    const uint32_t omax = last_row - static_cast<uint32_t>(t) * tile_bytes;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint32_t o = whole ? koff[i] : min(koff[i], omax + 16u * chunk_of(i));
      const uint32_t kd = smem_at + 2 * (buf * kTileElems + (W * i + wave) * 512);
      if constexpr (SHORT == 0)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(kd), "v"(o), "s"(kt) : "memory", "m0");
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(kd + 2 * NBUF * kTileElems), "v"(o),
                   "s"(vt)
                   : "memory", "m0");
    }
  };

  // Lane-dependent part of the V^T fragment addresses (see read_v), in elements.
  int v_lane_base[2], k_lane_base[4];
  {
    const int jrow = (lane & 15) >> 2, m = lane & 3;
    const int rl = 4 * half + jrow, cl = 2 * ((lane >> 4) & 1) + (m >> 1);
    // rl < 8, cl < 4: the lane's part of the position is cl ^ swz(rl), below 8.
    v_lane_base[0] = rl * D + 8 * (cl ^ swz(rl)) + 4 * (m & 1);
    v_lane_base[1] = rl * D + 8 * (cl ^ swz(rl) ^ 4) + 4 * (m & 1);
#pragma unroll
    for (int f = 0; f < 4; ++f) k_lane_base[f] = qcol * D + 8 * ((2 * f + half) ^ swz(qcol));
  }
  if constexpr (SHORT > 0) {
    for (int t = 0; t < n_tiles; ++t) dma_tile(t, t);
  } else {
    dma_tile(0, 0);
  }
  // The slots of the workgroup's own rows, -1 for none, in LDS behind the tile
  // buffers (where only the epilogue's staging reaches): a load of them in the tile
  // loop would be waited for behind the previous tile's pool stores.
  // Behind them, for every 16 rows, (first slot << 5 | n) where the first n rows have
  // slots in order from a multiple of 16 inside one block and the others none (every
  // prompt behind a block table of 16 or more tokens), else -1.
  int64_t *const own_slots = reinterpret_cast<int64_t *>(smem + 2 * NBUF * kTileElems);
  static_assert(4 * NBUF * kTileElems + 8 * (kRows + kRows / 16) <= 2 * kSmemElems, "the slots fit behind the tile buffers");
  const BlockWriter writer(wave, lane, STEP && SHORT == 0 ? S.block_size : 0);
  if constexpr (STEP) {
    if (writes_pool && tid < kRows) {
      int64_t slot = -1;
      if (q0 + tid < len) slot = S.slots[static_cast<int64_t>(seq_begin + q0 + tid) * S.slot_stride + hk];
      if (slot >= S.pool_slots) slot = -1;
      own_slots[tid] = slot;
      const int64_t first = __shfl(slot, lane & 48);
      const uint32_t some = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(slot >= 0) >> (lane & 48)) & 0xffffu;
      const uint32_t fits = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(slot < 0 || slot == first + (lane & 15)) >> (lane & 48)) & 0xffffu;
      const bool in_order = fits == 0xffffu && (some & 1) && (some & (some + 1)) == 0 && (first & 15) == 0 && S.block_size >= 16;
      if ((lane & 15) == 0) own_slots[kRows + tid / 16] = in_order ? (first << 5 | __builtin_popcount(some)) : -1;
    }
  }
  if constexpr (SHORT > 0) {
    // The wave's 32 rows of q and of k, as below but 32 at a time: the rows of q pass
    // through the wave's own K tile, which then takes those of k.
#pragma unroll
    for (int f = 0; f < 8; ++f) qf[f].u = u32x4{0, 0, 0, 0};
    if (wq0 < len) {
      const int c = lane & 7, r8 = lane >> 3;
      u32x4 qlo[4], qhi[4], klo[4], khi[4];
      uint16_t *qp[4], *kp[4];
      int64_t pos[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int64_t row = seq_begin + min(wq0 + 8 * it + r8, len - 1);
        pos[it] = S.positions[row];
        qp[it] = const_cast<uint16_t *>(I.q) + row * I.q_stride + hq * D + 8 * c;
        kp[it] = const_cast<uint16_t *>(I.k) + row * I.kv_stride + hk * D + 8 * c;
        qlo[it] = *reinterpret_cast<const u32x4 *>(qp[it]);
        qhi[it] = *reinterpret_cast<const u32x4 *>(qp[it] + D / 2);
        klo[it] = *reinterpret_cast<const u32x4 *>(kp[it]);
        khi[it] = *reinterpret_cast<const u32x4 *>(kp[it] + D / 2);
      }
      uint16_t *const stage = smem + wave * kTileElems;
      auto rotate = [&](u32x4 &lo, u32x4 &hi, const float (&cs)[8], const float (&sn)[8], int r) {
        const uint4 x = make_uint4(lo.x, lo.y, lo.z, lo.w), y = make_uint4(hi.x, hi.y, hi.z, hi.w);
        const uint4 xr = rotate_chunk<T>(x, y, cs, sn, false), yr = rotate_chunk<T>(y, x, cs, sn, true);
        lo = u32x4{xr.x, xr.y, xr.z, xr.w};
        hi = u32x4{yr.x, yr.y, yr.z, yr.w};
      };
      auto to_stage = [&](const u32x4 (&lo)[4], const u32x4 (&hi)[4]) {
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const int r = 8 * it + r8;
          *reinterpret_cast<u32x4 *>(stage + r * D + 8 * (c ^ swz(r))) = lo[it];
          *reinterpret_cast<u32x4 *>(stage + r * D + 8 * ((c + 8) ^ swz(r))) = hi[it];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      };
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int64_t p = pos[it] < 0 ? 0 : (pos[it] >= S.max_position ? S.max_position - 1 : pos[it]);
        const u32x4 *row = reinterpret_cast<const u32x4 *>(S.cos_sin + p * D + 8 * c);
        const u32x4 c0 = row[0], c1 = row[1], s0 = row[D / 8], s1 = row[D / 8 + 1];
        float cs[8], sn[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          cs[e] = __uint_as_float(e < 4 ? c0[e] : c1[e & 3]);
          sn[e] = __uint_as_float(e < 4 ? s0[e] : s1[e & 3]);
        }
        rotate(qlo[it], qhi[it], cs, sn, 8 * it + r8);
        rotate(klo[it], khi[it], cs, sn, 8 * it + r8);
      }
      to_stage(qlo, qhi);
      if (my_q < len) {
#pragma unroll
        for (int f = 0; f < 8; ++f)
          qf[f].u = *reinterpret_cast<const u32x4 *>(stage + qcol * D + 8 * ((2 * f + half) ^ swz(qcol)));
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      to_stage(klo, khi);
      // (every load of this wave has landed before its stores go out: nothing waits
      // for the stores)
      __builtin_amdgcn_s_waitcnt(0x0070);
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        *reinterpret_cast<u32x4 *>(qp[it]) = qlo[it];
        *reinterpret_cast<u32x4 *>(qp[it] + D / 2) = qhi[it];
        *reinterpret_cast<u32x4 *>(kp[it]) = klo[it];
        *reinterpret_cast<u32x4 *>(kp[it] + D / 2) = khi[it];
      }
    } else {
      __builtin_amdgcn_s_waitcnt(0x0070);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  if constexpr (STEP && SHORT == 0) {
    // Rotation of the wave's 32 query rows: a lane takes the chunks c and c + 8
    // (the two halves of the same pairs) of one row, 8 rows at a time, so that
    // rows, table and the write-back go as whole lines, and the fragments come
    // back through the second tile buffers, 16 rows (4 KiB per wave) at a time.
    // Rows past the prompt stand for its last one (the same value stored twice,
    // by the one wave that holds the row, after all its loads); a wave that has
    // only such rows does nothing.
#pragma unroll
    for (int f = 0; f < 8; ++f) qf[f].u = u32x4{0, 0, 0, 0};
    if (wq0 < len) {
      const int c = lane & 7, r8 = lane >> 3;
      u32x4 lo[4], hi[4], cs4[4][2], sn4[4][2];
      int64_t pos[4];
      uint16_t *qp[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int64_t row = seq_begin + min(wq0 + 8 * it + r8, len - 1);
        pos[it] = S.positions[row];
        qp[it] = const_cast<uint16_t *>(I.q) + row * I.q_stride + hq * D + 8 * c;
        lo[it] = *reinterpret_cast<const u32x4 *>(qp[it]);
        hi[it] = *reinterpret_cast<const u32x4 *>(qp[it] + D / 2);
      }
      __builtin_amdgcn_sched_barrier(0);   // the rows are requested before the wait for the positions
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int64_t p = pos[it] < 0 ? 0 : (pos[it] >= S.max_position ? S.max_position - 1 : pos[it]);
        const u32x4 *row = reinterpret_cast<const u32x4 *>(S.cos_sin + p * D + 8 * c);
        cs4[it][0] = row[0];
        cs4[it][1] = row[1];
        sn4[it][0] = row[D / 8];
        sn4[it][1] = row[D / 8 + 1];
      }
      uint16_t *const stage = smem + (1 + 2 * (wave >> 1)) * kTileElems + (wave & 1) * (kTileElems / 2);
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int it = 2 * pass + h, r = 8 * h + r8;
          float cs[8], sn[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            cs[e] = __uint_as_float(cs4[it][e >> 2][e & 3]);
            sn[e] = __uint_as_float(sn4[it][e >> 2][e & 3]);
          }
          const uint4 x = make_uint4(lo[it].x, lo[it].y, lo[it].z, lo[it].w);
          const uint4 y = make_uint4(hi[it].x, hi[it].y, hi[it].z, hi[it].w);
          const uint4 xr = rotate_chunk<T>(x, y, cs, sn, false), yr = rotate_chunk<T>(y, x, cs, sn, true);
          const u32x4 xo = {xr.x, xr.y, xr.z, xr.w}, yo = {yr.x, yr.y, yr.z, yr.w};
          *reinterpret_cast<u32x4 *>(qp[it]) = xo;
          *reinterpret_cast<u32x4 *>(qp[it] + D / 2) = yo;
          *reinterpret_cast<u32x4 *>(stage + r * D + 8 * (c ^ swz(r))) = xo;
          *reinterpret_cast<u32x4 *>(stage + r * D + 8 * ((c + 8) ^ swz(r))) = yo;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int r = qcol & 15;
        const bool take = (qcol >> 4) == pass && my_q < len;
        if (take) {
#pragma unroll
          for (int f = 0; f < 8; ++f)
            qf[f].u = *reinterpret_cast<const u32x4 *>(stage + r * D + 8 * ((2 * f + half) ^ swz(r)));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
  }
  bool stores_counted = false;             // the previous tile's pool stores: exactly four, behind this tile's loads
  // (the compiler's own loads are behind it: a wait for them would be one for the tiles)
  if constexpr (SHORT == 0) __builtin_amdgcn_s_waitcnt(0x0070);
  auto tile = [&](int t, auto buffer) {
    constexpr int cur = decltype(buffer)::value;
    const int k0 = t * kBN;
    if constexpr (SHORT == 0) {
      // This wave's part of tile t has landed; after the barrier all of it has,
      // and everybody is done with the other buffer.  (The barrier by itself:
      // __syncthreads() would wait for the pool stores as well.)
      if (STEP && stores_counted) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
#ifdef MUX_TRACE
    if (t == 0) tr_first = __builtin_amdgcn_s_memrealtime();
#endif
    // A workgroup's own rows are its last four tiles: their K and V go to the pool
    // behind the tile's math.
    const bool to_pool = STEP && writes_pool && k0 >= q0;
    if (SHORT == 0 && t + 1 < n_tiles) dma_tile(t + 1, cur ^ 1);
    const uint16_t *const Kt = smem + cur * kTileElems;           // this tile's K
    const uint16_t *const Vr = smem + (NBUF + cur) * kTileElems;     // this tile's V (row-major)
    // (nothing to compute where every key of the tile is in this wave's future, or
    // all of the wave's rows are past the prompt's end)
    if (k0 <= wq0 + 31 && wq0 < len) {
      // ---- S^T = K . Q^T ------------------------------------------------------------------
      // LDS fragment reads run kDepth steps ahead of the MFMAs that consume them.
      // In the P.V product consecutive MFMAs go to different accumulators (4 dim
      // blocks); a single dependent chain, as here, runs at 3/4
      // of the rate.
      constexpr int kDepth = 4;
      v16f32 sacc;
#pragma unroll
      for (int i = 0; i < 16; ++i) sacc[i] = 0.f;
      {
        // Fragment j: dims 16 j + 8 half .. +7 of key row qcol.
        auto read_k = [&](int j) {
          Frag f;
          f.u = *reinterpret_cast<const u32x4 *>(Kt + k_lane_base[j & 3] + 64 * (j >> 2));
          return f;
        };
        Frag ring[kDepth];
#pragma unroll
        for (int j = 0; j < kDepth; ++j) ring[j] = read_k(j);
        __builtin_amdgcn_sched_barrier(0);   // keep the scheduler from sinking the reads to their uses
        MUX_PF_PRIO(MUX_PF_PRIO_MFMA);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          sacc = mfma<T>(ring[j % kDepth], qf[j], sacc);
          if (j + kDepth < 8) ring[j % kDepth] = read_k(j + kDepth);
          __builtin_amdgcn_sched_barrier(0);
        }
        MUX_PF_PRIO(MUX_PF_PRIO_VALU);
      }

      // ---- softmax over keys, per query column --------------------------------------
      // register i is key k0 + 8 (i/4) + 4 half + i%4.
      // Raw scores stay unscaled; scale (> 0) is folded into the exponent:
      // p = exp2(s * scale_log2 - m * scale_log2).
      // Exactly one tile per wave straddles the diagonal; only it pays for the mask.
      if (k0 + kBN - 1 > wq0) {
        const int rel = my_q - k0 - 4 * half;   // key offset inside the tile, less this lane's share
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i / 4) + (i % 4) > rel) sacc[i] = -INFINITY;
      }
      // The exponents' reference (m_run) stays where it is until a lane's
      // probabilities of a tile add up to more than kRescaleSum: a probability is then
      // kRescaleSum at most, well inside fp16 and fp32, and the 64 accumulators and the
      // running sum are rescaled rarely instead of whenever a maximum rises at all (with
      // 32 rows per wave, that is in most tiles of a prompt's first hundreds of keys).
      // Not further: the key that dominates a row is exact where it is the reference
      // itself, and rounded to 11 bits where the reference lags behind it.
      // The sum is needed anyway; the maxima are taken only where the reference moves:
      // there, in a wave's first tile, and wherever the sum is not a number.
      constexpr float kRescaleSum = 256.f;
      float p[16], psum;
      auto exponentials = [&] {
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = fast_exp2(__builtin_fmaf(sacc[i], I.scale_log2, neg_m));
        psum = p[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) psum += p[i];
      };
      bool moves = t == 0;                 // (no reference yet)
      if (!moves) {
        exponentials();
        moves = __builtin_amdgcn_ballot_w64(!(psum <= kRescaleSum)) != 0;
      }
      if (moves) {
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sacc[i]);
        const float m_new = fmaxf(m_run, max_with_lane_xor32(mx));
        // Rows past the prompt may have no valid key at all; keep them finite.
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2((m_run - m_use) * I.scale_log2);
        l_run *= alpha;
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[mb][i] *= alpha;
        m_run = m_use;
        neg_m = -m_use * I.scale_log2;
        exponentials();
      }
      l_run += psum;
      Frag pf[2];                                 // B fragments, 16 keys each
      // bf16 keeps only 8 mantissa bits of a probability, which alone would cost
      // more than the 2e-3 budget, so bf16 P is carried as hi + lo parts.
      constexpr bool kSplitP = __is_same(T, BF16);
      Frag pf_lo[kSplitP ? 2 : 1];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = pack2<T>(p[8 * st + 2 * j], p[8 * st + 2 * j + 1]);
        pf[st].u = u32x4{w[0], w[1], w[2], w[3]};
        if constexpr (kSplitP) {
          // The part of p that its bf16 rounding lost, as a second bf16.
          uint32_t lo[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            lo[j] = pack2<T>(p[8 * st + 2 * j] - bf16_lo(w[j]), p[8 * st + 2 * j + 1] - bf16_hi(w[j]));
          pf_lo[st].u = u32x4{lo[0], lo[1], lo[2], lo[3]};
        }
      }

      // ---- O^T += V^T . P^T ---------------------------------------------------------------
      // k-slot j of lane half h in step st is key 16 st + 8 (j/4) + 4 h + j%4
      {
        auto read_v = [&](int n) {         // fragment n = 4 ks + mb
          const int mb = n % 4, ks = n / 4;
          Frag f;
          // The transposing read works on groups of 16 lanes: lane 4 j + m of a
          // group points at dims 4 m .. 4 m + 3 of key row j, and lane i of the
          // group receives dim i of rows 0..3.  Here a group covers dims
          // 32 mb + 16 (lane/16 % 2) .. +15 and keys 16 ks + 4 half (+ 8) .. +3.
          // Address: row = 16 ks + 8 hsel + rl with rl = 4 half + jrow, chunk =
          // 4 mb + cl, position = chunk ^ swz(rl): cl ^ swz(rl) is below 8, so only
          // bit 2 of the constant part (mb odd) has to be folded into the lane's base:
          // two bases per lane, everything else is an immediate offset.
          typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
          u32x2 part[2];
#pragma unroll
          for (int hsel = 0; hsel < 2; ++hsel) {
            const uint16_t *src = Vr + v_lane_base[mb & 1] + (16 * ks + 8 * hsel) * D + 64 * (mb >> 1);
            const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16 *)src);
            union { v4i16 v; u32x2 u; } c;
            c.v = r;
            part[hsel] = c.u;
          }
          f.u = u32x4{part[0].x, part[0].y, part[1].x, part[1].y};
          return f;
        };
        Frag ring[kDepth];
#pragma unroll
        for (int j = 0; j < kDepth; ++j) ring[j] = read_v(j);
        __builtin_amdgcn_sched_barrier(0);
        MUX_PF_PRIO(MUX_PF_PRIO_MFMA);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          oacc[j % 4] = mfma<T>(ring[j % kDepth], pf[j / 4], oacc[j % 4]);
          if constexpr (kSplitP) oacc[j % 4] = mfma<T>(ring[j % kDepth], pf_lo[j / 4], oacc[j % 4]);
          if (j + kDepth < 8) ring[j % kDepth] = read_v(j + kDepth);
          __builtin_amdgcn_sched_barrier(0);
        }
        MUX_PF_PRIO(MUX_PF_PRIO_VALU);
      }
    }
    if constexpr (STEP) {
      stores_counted = to_pool;
      if (to_pool) {
#pragma unroll 1
        for (int r = 0; r < kBN; r += 16) {
          const uint32_t slots_at = smem_at + 4 * NBUF * kTileElems + 8 * (k0 - q0 + r);
          int64_t run;
          asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(run)
                       : "v"(smem_at + 4 * NBUF * kTileElems + 8 * (kRows + (k0 - q0 + r) / 16))
                       : "memory");
          const uint32_t run_lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(run));
          const uint32_t run_hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(run >> 32));
          run = static_cast<int64_t>((static_cast<uint64_t>(run_hi) << 32) | run_lo);
          const uint32_t kt = smem_at + 2 * (cur * kTileElems + r * D), vt = kt + 2 * NBUF * kTileElems;
          if constexpr (SHORT == 0) {
            if (run >= 0) stores_counted &= write_block_to_pool(kt, vt, writer, run >> 5, static_cast<int>(run & 31), lane, S);
            else stores_counted &= write_tokens_to_pool(Kt, Vr, r, slots_at, wave, lane, S);
          } else {
            for (int part = wave; part < 4; part += W) {      // (what the four waves of the other forms do)
              if (run >= 0)
                write_block_to_pool(kt, vt, BlockWriter(part, lane, S.block_size), run >> 5, static_cast<int>(run & 31), lane, S);
              else write_tokens_to_pool(Kt, Vr, r, slots_at, part, lane, S);
            }
          }
        }
      }
    }
  };
  if constexpr (SHORT > 0) {
    tile(0, std::integral_constant<int, 0>{});
    if constexpr (W > 1)
      if (n_tiles > 1) tile(1, std::integral_constant<int, 1>{});
    if constexpr (W > 2) {
      if (n_tiles > 2) tile(2, std::integral_constant<int, 2>{});
      if (n_tiles > 3) tile(3, std::integral_constant<int, 3>{});
    }
  } else {
    for (int t = 0; t < n_tiles; t += 2) {
      tile(t, std::integral_constant<int, 0>{});
      if (t + 1 < n_tiles) tile(t + 1, std::integral_constant<int, 1>{});
    }
  }

#ifdef MUX_TRACE
  const long long tr_loop = __builtin_amdgcn_s_memrealtime();
#endif
  // ---- normalise and store: register i of block mb is d = 32 mb + 8 (i/4) + 4 half + i%4 ------
  const float l_tot = sum_with_lane_xor32(l_run);
  const float inv = 1.f / l_tot;
  if (I.out_rows_16b) {
    // Through LDS, so that the rows go out as whole 256-byte runs (16 bytes per
    // lane, four rows per instruction) instead of 8-byte pieces of 32 rows: the
    // tile buffers are free once every wave has left the loop.
    constexpr int kORow = D + 8;         // 272-byte rows
    static_assert(W * 32 * kORow <= kSmemElems, "output staging fits the tile buffers");
    // (the barrier by itself, as in the loop: nothing waits for the pool stores)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    uint16_t *stage = smem + wave * 32 * kORow;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<u32x2 *>(&stage[qcol * kORow + 32 * mb + 8 * g + 4 * half]) =
            u32x2{pack2<T>(oacc[mb][4 * g] * inv, oacc[mb][4 * g + 1] * inv),
                  pack2<T>(oacc[mb][4 * g + 2] * inv, oacc[mb][4 * g + 3] * inv)};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int chunk = lane & 15;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int r = 4 * it + (lane >> 4);
      if (wq0 + r < len) {
        const u32x4 x = *reinterpret_cast<const u32x4 *>(&stage[r * kORow + 8 * chunk]);
        *reinterpret_cast<u32x4 *>(I.out + static_cast<int64_t>(seq_begin + wq0 + r) * I.out_stride + hq * D +
                                   8 * chunk) = x;
      }
    }
  } else if (my_q < len) {
    uint16_t *op = I.out + static_cast<int64_t>(seq_begin + my_q) * I.out_stride + hq * D + 4 * half;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint2 w2 = make_uint2(pack2<T>(oacc[mb][4 * g] * inv, oacc[mb][4 * g + 1] * inv),
                                    pack2<T>(oacc[mb][4 * g + 2] * inv, oacc[mb][4 * g + 3] * inv));
        *reinterpret_cast<uint2 *>(op + 32 * mb + 8 * g) = w2;
      }
  }
#ifdef MUX_TRACE
  if (tid == 0 && tr_table && blockIdx.x < tr_rows) {
    long long *row = tr_table + 8 * static_cast<long long>(blockIdx.x);
    row[0] = tr_entry, row[1] = tr_len, row[2] = tr_first, row[3] = tr_loop, row[4] = __builtin_amdgcn_s_memrealtime();
    row[5] = n_tiles, row[6] = len, row[7] = q0;
  }
#endif
}

template <typename T>
__global__ __launch_bounds__(256, 3) void prefill_causal_kernel(const PrefillParams P) {
  prefill_body<T, false>(P, PrefillStep{});
}
template <typename T>
__global__ __launch_bounds__(256, 3) void prefill_step_kernel(const PrefillParams P, const PrefillStep S) {
  prefill_body<T, true>(P, S);
}
template <typename T, int W>
__global__ __launch_bounds__(64 * W, 2) void prefill_short_step_kernel(const PrefillParams P, const PrefillStep S) {
  prefill_body<T, true, W>(P, S);
}

}  // namespace mux

namespace mux {
namespace {

int32_t check_prefill_item(const MuxPrefillItem &it, int32_t head_size) {
  // (pointers are only required when there is something to do)
  const bool work = it.num_prompts > 0 && it.max_prompt_len > 0;
  if (work && (!it.out || !it.q || !it.k || !it.v || !it.cu_seqlens)) return MUXA_EINVAL;
  if (it.num_prompts < 0 || it.max_prompt_len < 0 || it.num_q_heads <= 0 || it.num_kv_heads <= 0) return MUXA_EINVAL;
  if (it.num_q_heads % it.num_kv_heads != 0) return MUXA_EINVAL;
  if (head_size != kHeadSize) return MUXA_EUNSUPPORTED;
  if (it.q_row_stride < static_cast<int64_t>(it.num_q_heads) * kHeadSize ||
      it.out_row_stride < static_cast<int64_t>(it.num_q_heads) * kHeadSize ||
      it.kv_row_stride < static_cast<int64_t>(it.num_kv_heads) * kHeadSize)
    return MUXA_EINVAL;
  // 16-byte fragment loads and 8-byte output stores.
  if (it.q_row_stride % 8 || it.kv_row_stride % 8 || it.out_row_stride % 4) return MUXA_EINVAL;
  const uintptr_t a16 =
      reinterpret_cast<uintptr_t>(it.q) | reinterpret_cast<uintptr_t>(it.k) | reinterpret_cast<uintptr_t>(it.v);
  if ((a16 & 15u) || (reinterpret_cast<uintptr_t>(it.out) & 7u)) return MUXA_EINVAL;
  // K/V rows of one prompt are addressed with 32-bit byte offsets.
  if (static_cast<int64_t>(it.max_prompt_len + kBM + 2 * kBN) * it.kv_row_stride * 2 >= (int64_t{1} << 32))
    return MUXA_EUNSUPPORTED;
  if (it.prompt_lens_host != nullptr)
    for (int p = 0; p < it.num_prompts; ++p)
      if (it.prompt_lens_host[p] < 0 || it.prompt_lens_host[p] > it.max_prompt_len) return MUXA_EINVAL;
  return MUXA_OK;
}

PrefillItemDev device_item(const MuxPrefillItem &it) {
  PrefillItemDev d;
  d.out = static_cast<uint16_t *>(it.out);
  d.q = static_cast<const uint16_t *>(it.q);
  d.k = static_cast<const uint16_t *>(it.k);
  d.v = static_cast<const uint16_t *>(it.v);
  d.out_stride = it.out_row_stride;
  d.q_stride = it.q_row_stride;
  d.kv_stride = it.kv_row_stride;
  d.cu_seqlens = it.cu_seqlens;
  d.ratio = it.num_q_heads / it.num_kv_heads;
  d.num_kv_heads = it.num_kv_heads;
  d.num_prompts = it.num_prompts;
  d.kv_per_xcd = (it.num_kv_heads + 7) / 8;
  d.scale_log2 = it.scale * 1.4426950408889634f;
  d.out_rows_16b = (reinterpret_cast<uintptr_t>(it.out) & 15u) == 0 && it.out_row_stride % 8 == 0;
  return d;
}

hipError_t launch_prefill(const PrefillParams &P, const PrefillStep *S, int64_t n_wg, int32_t dtype, hipStream_t st) {
  const dim3 grid(static_cast<uint32_t>(n_wg));
  if (S != nullptr && S->short_waves > 0) {
#define MUX_PF_SHORT(W)                                                                                                  \
  do {                                                                                                                   \
    if (dtype == MUXA_DTYPE_F16) hipLaunchKernelGGL((prefill_short_step_kernel<F16, W>), grid, dim3(64 * W), 0, st, P, *S); \
    else hipLaunchKernelGGL((prefill_short_step_kernel<BF16, W>), grid, dim3(64 * W), 0, st, P, *S);                     \
  } while (0)
    if (S->short_waves == 1) MUX_PF_SHORT(1);
    else if (S->short_waves == 2) MUX_PF_SHORT(2);
    else MUX_PF_SHORT(4);
#undef MUX_PF_SHORT
  } else if (S != nullptr) {
    if (dtype == MUXA_DTYPE_F16) hipLaunchKernelGGL((prefill_step_kernel<F16>), grid, dim3(256), 0, st, P, *S);
    else hipLaunchKernelGGL((prefill_step_kernel<BF16>), grid, dim3(256), 0, st, P, *S);
  } else if (dtype == MUXA_DTYPE_F16) hipLaunchKernelGGL((prefill_causal_kernel<F16>), grid, dim3(256), 0, st, P);
  else hipLaunchKernelGGL((prefill_causal_kernel<BF16>), grid, dim3(256), 0, st, P);
  return hipGetLastError();
}

// One model on the grid sized by its longest prompt (no host-side lengths, or too
// many query tiles for the kernel argument).
int32_t launch_dense(const MuxPrefillItem &it, const int32_t *prompt_order, const PrefillStep *S, int32_t dtype,
                     hipStream_t st) {
  PrefillParams P = {};
  P.it[0] = device_item(it);
  P.prompt_order = prompt_order;
  P.q_tiles = (it.max_prompt_len + kBM - 1) / kBM;
  P.num_groups = it.num_prompts * it.num_kv_heads;
  const int64_t n_wg = static_cast<int64_t>((P.num_groups + 7) / 8) * 8 * P.it[0].ratio * P.q_tiles;
  if (n_wg > 0x7fffffff || P.q_tiles > 0xffff) return MUXA_EUNSUPPORTED;
  hipError_t e = launch_prefill(P, S, n_wg, dtype, st);
  if (e != hipSuccess) return hip_fail(e);
  return MUXA_OK;
}

// items[first .. first + n): one launch over the query tiles that exist, the
// heaviest (most keys) of all models first; false when they do not fit the
// kernel argument.  S: the step form (one item).
bool launch_compact(const MuxPrefillItem *items, int n, const PrefillStep *S, int32_t dtype, hipStream_t st,
                    int32_t *rc) {
  PrefillParams P = {};
  int64_t total = 0;
  int max_tiles = 0, slots = 0, n_dev = 0;
  int dev_of[MUXA_MAX_DECODE_ITEMS];
  for (int i = 0; i < n; ++i) {
    const MuxPrefillItem &it = items[i];
    dev_of[i] = -1;
    if (it.num_prompts == 0 || it.max_prompt_len == 0) continue;
    if (it.prompt_lens_host == nullptr || it.num_prompts > 0xffff) return false;
    int64_t tiles = 0;
    for (int p = 0; p < it.num_prompts; ++p) tiles += (it.prompt_lens_host[p] + kBM - 1) / kBM;
    if (tiles == 0) continue;
    total += tiles;
    max_tiles = std::max(max_tiles, (it.max_prompt_len + kBM - 1) / kBM);
    dev_of[i] = n_dev;
    P.it[n_dev] = device_item(it);
    slots = std::max(slots, P.it[n_dev].kv_per_xcd * P.it[n_dev].ratio);
    ++n_dev;
  }
  *rc = MUXA_OK;
  if (total == 0) return true;
  if (total > kMaxPairs || max_tiles > (1 << kPairTileBits)) return false;
  // Order: prompt by prompt, the longest prompt of all models first, and within a
  // prompt the heaviest query tile (most keys) first.  The query tiles and query
  // heads that read the same K/V then run at the same time on one XCD and walk
  // the keys from the start together, so a K/V tile is fetched from memory once
  // and found in that XCD's L2 by the others (tile by tile over the whole batch
  // instead - every stream of the batch live at once - the 16 x 2048-token shape
  // re-read K/V from memory at 4.6 TB/s and ran 1.2 x slower), and the launch
  // ends with the short prompts' small tiles.
  struct Group {
    int item, prompt, len;
  };
  std::vector<Group> groups;
  for (int i = 0; i < n; ++i) {
    if (dev_of[i] < 0) continue;
    for (int p = 0; p < items[i].num_prompts; ++p)
      if (items[i].prompt_lens_host[p] > 0) groups.push_back({i, p, items[i].prompt_lens_host[p]});
  }
  std::stable_sort(groups.begin(), groups.end(), [](const Group &a, const Group &b) { return a.len > b.len; });
  int np = 0;
  for (const Group &g : groups)
    for (int t = (g.len + kBM - 1) / kBM - 1; t >= 0; --t)
      P.pairs[np++] = (static_cast<uint32_t>(dev_of[g.item]) << 28) |
                      (static_cast<uint32_t>(g.prompt) << kPairTileBits) | static_cast<uint32_t>(t);
  P.n_pairs = np;
  P.slots_per_pair = slots;
  const int64_t n_wg = static_cast<int64_t>(np) * slots * 8;
  if (n_wg > 0x7fffffff) {
    *rc = MUXA_EUNSUPPORTED;
    return true;
  }
  hipError_t e = launch_prefill(P, S, n_wg, dtype, st);
  if (e != hipSuccess) *rc = hip_fail(e);
  return true;
}

}  // namespace
}  // namespace mux

extern "C" int32_t mux_multi_prefill_causal(const MuxPrefillItem *items, int32_t n_items, int32_t head_size,
                                            int32_t dtype, void *stream) {
  using namespace mux;
  if (!items || n_items <= 0 || n_items > MUXA_MAX_DECODE_ITEMS) return MUXA_EINVAL;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  for (int i = 0; i < n_items; ++i) {
    const int32_t rc = check_prefill_item(items[i], head_size);
    if (rc != MUXA_OK) return rc;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  int32_t rc = MUXA_OK;
  if (launch_compact(items, n_items, nullptr, dtype, st, &rc)) return rc;
  // Not all in one kernel argument: one launch per model, compact where possible.
  for (int i = 0; i < n_items; ++i) {
    if (items[i].num_prompts == 0 || items[i].max_prompt_len == 0) continue;
    if (!launch_compact(items + i, 1, nullptr, dtype, st, &rc))
      rc = launch_dense(items[i], nullptr, nullptr, dtype, st);
    if (rc != MUXA_OK) return rc;
  }
  return MUXA_OK;
}

extern "C" int32_t mux_prefill_causal(void *out, int64_t out_row_stride, const void *q, int64_t q_row_stride,
                                      const void *k, const void *v, int64_t kv_row_stride,
                                      const int32_t *cu_seqlens, const int32_t *prompt_order,
                                      const int32_t *prompt_lens_host, int32_t num_prompts,
                                      int32_t max_prompt_len, int32_t num_q_heads, int32_t num_kv_heads,
                                      int32_t head_size, float scale, int32_t dtype, void *stream) {
  using namespace mux;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  MuxPrefillItem it = {};
  it.out = out;
  it.out_row_stride = out_row_stride;
  it.q = q;
  it.q_row_stride = q_row_stride;
  it.k = k;
  it.v = v;
  it.kv_row_stride = kv_row_stride;
  it.cu_seqlens = cu_seqlens;
  it.prompt_lens_host = prompt_lens_host;
  it.num_prompts = num_prompts;
  it.max_prompt_len = max_prompt_len;
  it.num_q_heads = num_q_heads;
  it.num_kv_heads = num_kv_heads;
  it.scale = scale;
  const int32_t rc0 = check_prefill_item(it, head_size);
  if (rc0 != MUXA_OK) return rc0;
  if (num_prompts == 0 || max_prompt_len == 0) return MUXA_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  int32_t rc = MUXA_OK;
  if (launch_compact(&it, 1, nullptr, dtype, st, &rc)) return rc;
  return launch_dense(it, prompt_order, nullptr, dtype, st);
}

extern "C" int32_t mux_rope_prefill_and_cache(const MuxPrefillItem *attn, const MuxCacheWriteItem *write, void *k_pool,
                                              void *v_pool, int64_t num_pool_blocks, int32_t head_size,
                                              int32_t block_size, int32_t dtype, void *stream) {
  using namespace mux;
  if (!attn || !write) return MUXA_EINVAL;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  const MuxPrefillItem &it = *attn;
  const MuxCacheWriteItem &w = *write;
  int32_t rc = check_prefill_item(it, head_size);
  if (rc != MUXA_OK) return rc;
  rc = check_cache_write(w.k, w.v, w.kv_row_stride, k_pool, v_pool, num_pool_blocks, w.slot_mapping, w.layer,
                         w.num_layers, w.num_tokens, w.num_kv_heads, head_size, block_size, dtype);
  if (rc != MUXA_OK) return rc;
  // Both items describe the same q, k and v, and every token belongs to a prompt.
  if (it.q != w.q || it.k != w.k || it.v != w.v || it.q_row_stride != w.q_row_stride ||
      it.kv_row_stride != w.kv_row_stride || it.num_q_heads != w.num_q_heads || it.num_kv_heads != w.num_kv_heads)
    return MUXA_EINVAL;
  if (w.num_tokens > 0 && (!w.positions || !w.cos_sin || !it.prompt_lens_host)) return MUXA_EINVAL;
  if (w.max_position <= 0) return MUXA_EINVAL;
  if (w.rotary_dim != kHeadSize) return MUXA_EUNSUPPORTED;
  int64_t tokens = 0;
  for (int p = 0; p < it.num_prompts && it.prompt_lens_host; ++p) tokens += it.prompt_lens_host[p];
  if (tokens != w.num_tokens) return MUXA_EINVAL;
  if (tokens == 0) return MUXA_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  PrefillStep S = {};
  S.positions = w.positions;
  S.cos_sin = w.cos_sin;
  S.slots = w.slot_mapping + static_cast<int64_t>(w.layer) * w.num_kv_heads;
  S.slot_stride = static_cast<int64_t>(w.num_layers) * w.num_kv_heads;
  S.k_pool = static_cast<uint16_t *>(k_pool);
  S.v_pool = static_cast<uint16_t *>(v_pool);
  S.pool_slots = num_pool_blocks * block_size;
  S.max_position = w.max_position;
  S.block_size = block_size;
  S.short_waves = prompt_step_short_waves(it.prompt_lens_host, it.num_prompts, it.num_q_heads, it.num_kv_heads);
  if (S.short_waves == 0) {
    const hipError_t e = launch_rotary_k(w.positions, static_cast<uint16_t *>(w.k), w.kv_row_stride, w.cos_sin,
                                         w.max_position, w.num_tokens, w.num_kv_heads, dtype, st);
    if (e != hipSuccess) return hip_fail(e);
  }
  if (launch_compact(&it, 1, &S, dtype, st, &rc)) return rc;
  return launch_dense(it, nullptr, &S, dtype, st);
}

#ifdef MUX_TRACE
// Tracing build only: where the prefill kernel's workgroups write their stamps
// (DEVICE int64 [rows, 8], zero-filled by the caller; NULL switches it off).
extern "C" int32_t mux_prefill_trace_set(void *table, int64_t rows) {
  long long *p = static_cast<long long *>(table);
  long long n = table ? rows : 0;
  MUX_HIP_TRY(hipMemcpyToSymbol(HIP_SYMBOL(mux::g_prefill_trace), &p, sizeof(p)));
  MUX_HIP_TRY(hipMemcpyToSymbol(HIP_SYMBOL(mux::g_prefill_trace_rows), &n, sizeof(n)));
  return MUXA_OK;
}
#endif
