// Greedy sampling for gfx950: logits = hidden . embedding^T and the argmax over
// the vocabulary in one pass over the embedding matrix
// (muxserve/flexserver/sampler.py:15-35).  The logits are never written: a step
// reads the [vocab, hidden] matrix once (262 MB for a 7B model) and a few rows of
// hidden states, so the kernel is bound by HBM.
//
// lm_head_argmax_kernel<T, NB, NW>: a workgroup of NW waves owns 16 NW vocabulary
// rows (16 per wave) and up to 16 NB sampled rows of hidden states, and walks the
// hidden dimension in tiles of 128.
//   * Hidden states: the tile [16 NB][128] is staged in LDS, shared by the
//     waves, double-buffered, one barrier per tile.  Every workgroup reads all
//     of the sampled hidden states (from L2), so large vocabularies use 8 waves
//     per workgroup: half as many workgroups, half that traffic.
//   * Embedding rows: the MFMA A operand wants lane l to hold row l % 16
//     (v_mfma_f32_16x16x32: columns 8 (l / 16) .. +7 of a 32-column slice) -
//     loaded that way, every 16 lanes would touch 16 different rows with 16 bytes
//     each.  Instead a load instruction takes 4 rows x 256 contiguous bytes
//     (16 lanes per row), a tile ahead of their use (deeper makes no difference), and the wave regroups
//     its 4 KiB tile through a private LDS area: 16-byte chunk c of row r sits at
//     position c ^ r of the row, so both the row-wise writes and the
//     column-wise fragment reads are free of bank conflicts.
// Accumulators hold logits[vocab row 4 (l / 16) + i][sampled row l % 16]; each is
// rounded to the storage type (the reference compares logits of that type) and
// reduced to the workgroup's (max, lowest index) per sampled row, which goes to
// the workgroup's line of a table as a 64-bit key (ordered logit bits << 32 |
// ~index).  The last workgroup to arrive (a counter tells it) takes the maximum
// of every column of the table, writes the token ids and leaves the counter at
// zero for the next launch.  (Atomic max on one key per sampled row instead of
// the table serialises 16000 atomics on two cache lines: +30 us per launch.)
#include "mux_common.h"

namespace mux {

typedef _Float16 sm_v8f16 __attribute__((ext_vector_type(8)));
typedef __bf16 sm_v8bf16 __attribute__((ext_vector_type(8)));
typedef float sm_v4f32 __attribute__((ext_vector_type(4)));
typedef uint32_t sm_u32x4 __attribute__((ext_vector_type(4)));

union SmFrag {
  sm_u32x4 u;
  sm_v8f16 h;
  sm_v8bf16 b;
};

constexpr int kSmTile = 256;              // the hidden size must be a multiple of this
constexpr int kSmMaxRowsPerPass = 256;
// Up to 32 sampled rows the narrow kernel, beyond them the wide one.  32000 rows of
// 4096, us: the narrow one with 32 rows 43.5, the wide one with 33 to 64 rows 46 to
// 47.5 (the narrow one with four row blocks per wave took 52.3 to 53.5 there, and 107
// and 214 with 128 and 256 rows, passing over the matrix once per 64; the wide one 55
// and 76).  Small vocabularies too, though the wide kernel keeps its 128 rows per
// workgroup there: 16000 rows, 33 sampled 46.6 / 34.9, 64 48.0 / 38.1; 4000 rows
// 37.0 / 30.8 and 38.3 / 33.8.
constexpr int kSmNarrowRows = 32;
#ifndef MUX_SM_PREFETCH_TILES
#define MUX_SM_PREFETCH_TILES 2
#endif

struct LmHeadParams {
  const uint16_t *hidden;
  int64_t hidden_stride;
  const int32_t *row_index;               // sampled row r reads hidden row row_index[r]; null: row r
  const uint16_t *weight;
  int64_t weight_stride;
  int32_t hidden_size, vocab, num_rows;
  int32_t hidden_rows;                    // rows of `hidden`: row_index entries are clamped to it
  int32_t half_tiles;                     // the wide kernel: a large vocabulary, which the narrow one gives 8 waves
  uint32_t *counter;                      // workgroups arrived (and, behind it, per group of them), zero between launches
  unsigned long long *table;              // [workgroups][16 NB] keys, written before they are read
  int64_t *next_tokens;
};

// Float bits that compare like the floats as unsigned integers.
__device__ __forceinline__ uint32_t ordered_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

template <typename T>
__device__ __forceinline__ float sm_round(float f) {
  if constexpr (__is_same(T, F16)) return static_cast<float>(static_cast<_Float16>(f));
  else return __uint_as_float(static_cast<uint32_t>(f32_to_bf16_bits(f)) << 16);
}

// (value, index) pairs ordered by value, ties to the lower index.
__device__ __forceinline__ void take_better(float &v, int &i, float ov, int oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

// The workgroup's result per sampled row goes to its line of the table as a
// 64-bit key (ordered logit bits << 32 | ~index: a larger key is a better
// logit or, between equal logits, a lower index).
__device__ __forceinline__ void store_key(const LmHeadParams &P, int64_t at, float v, int i) {
  const unsigned long long key =
      (static_cast<unsigned long long>(ordered_bits(v)) << 32) | (0xffffffffu - static_cast<uint32_t>(i));
  __hip_atomic_store(&P.table[at], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Announces this workgroup's line of the table to the `expected` workgroups of a
// counter; true in the one that came last.  The table is written and read with device-coherent accesses (they
// bypass the per-XCD L2), so ordering them against the counter takes only a wait
// for this wave's table stores to be acknowledged before the workgroup meets
// and bumps the counter.  A device-scope fence would also write back and
// invalidate this XCD's L2, which holds the hidden states every other
// workgroup is still reading (measured: +30 us per launch).
__device__ __forceinline__ bool last_to_arrive(uint32_t *counter, uint32_t expected, int *s_last) {
  wait_own_vector_memory();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  if (threadIdx.x == 0)
    *s_last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == expected - 1;
  __syncthreads();
  if (!*s_last) return false;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  return true;
}

// Maximum over n lines of the table from `first`, `step` lines apart, per sampled
// row: thread -> (row tid % ROWS, slice tid / ROWS of the lines), sixteen loads in
// flight.  The result is whole in the threads below ROWS.  fin: THREADS keys of LDS.
template <int ROWS, int THREADS>
__device__ __forceinline__ unsigned long long reduce_lines(const LmHeadParams &P, int first, int n, int step,
                                                           unsigned long long *fin) {
  constexpr int SLICES = THREADS / ROWS;
  const int tid = threadIdx.x;
  const int row = tid % ROWS, slice = tid / ROWS;
  unsigned long long best = 0;
  for (int b0 = slice; b0 < n && slice < SLICES; b0 += 16 * SLICES) {
    unsigned long long v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int b = b0 + j * SLICES;
      v[j] = b < n ? __hip_atomic_load(&P.table[static_cast<int64_t>(first + b * step) * ROWS + row], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT)
                   : 0ull;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) best = v[j] > best ? v[j] : best;
  }
  fin[tid] = best;
  __syncthreads();
  if (tid < ROWS) {
#pragma unroll
    for (int sl = 1; sl < SLICES; ++sl) best = fin[sl * ROWS + tid] > best ? fin[sl * ROWS + tid] : best;
  }
  return best;
}

__device__ __forceinline__ void store_token(const LmHeadParams &P, int row, unsigned long long key) {
  const uint32_t idx = 0xffffffffu - static_cast<uint32_t>(key);
  P.next_tokens[row] = idx < static_cast<uint32_t>(P.vocab) ? idx : 0;   // every logit NaN: token 0
}

__device__ __forceinline__ void clear_counter(uint32_t *counter) {
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The last workgroup to arrive reduces the table.
template <int ROWS, int THREADS>
__device__ __forceinline__ void reduce_table(const LmHeadParams &P, unsigned long long *fin, int *s_last) {
  if (!last_to_arrive(P.counter, gridDim.x, s_last)) return;
  const unsigned long long key = reduce_lines<ROWS, THREADS>(P, 0, gridDim.x, 1, fin);
  if (static_cast<int>(threadIdx.x) < P.num_rows) store_token(P, threadIdx.x, key);
  clear_counter(P.counter);
}

template <typename T, int NB, int NW>
__global__ __launch_bounds__(64 * NW) void lm_head_argmax_kernel(const LmHeadParams P) {
  constexpr int KT = 128;                             // hidden elements per tile
  constexpr int ROWS = 16 * NB;                       // sampled rows held in LDS
  constexpr int CPR = KT / 8;                         // 16-byte chunks per tile row (16)
  constexpr int RPP = 4 * NW;                         // hidden-state rows staged per pass of the workgroup
  constexpr int SJ = (ROWS + RPP - 1) / RPP;          // staging chunks per thread
  constexpr int NF = KT / 32;                         // MFMA column slices per tile (4)
  constexpr int kHRow = KT + 8;     // LDS row pitch: 16 bytes of padding keep b128 reads off each other's banks
  __shared__ __attribute__((aligned(16))) uint16_t htile[2][ROWS * kHRow];
  __shared__ __attribute__((aligned(16))) uint16_t wtile[NW][16 * KT];  // 4 KiB per wave
  __shared__ float red_v[NW][ROWS];
  __shared__ int red_i[NW][ROWS];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int n_tiles = P.hidden_size / KT;
  // Workgroups start their walk over the hidden dimension at different tiles (a dot
  // product does not care about the order): with a row pitch that is a power of two
  // - 8 KiB at hidden size 4096 - workgroups walking in step would all be reading
  // the same few memory channels at any moment.  Large vocabularies (8 waves) start
  // at half tiles too, which spreads such a pitch better; one tile then consists of
  // the end and of the beginning of the hidden dimension, and a lane's column offset
  // is that of its half of the tile.  (32000 x 4096, one row 47.0 -> 43.0 us, 32 rows
  // 46.7 -> 43.5; small vocabularies wait for latencies and lose, 4000 x 5120 29.1 ->
  // 30.8.)
  // The start depends on the vocabulary and the vocabulary row alone (128 rows start
  // together, in both kernels and at both workgroup sizes), so that a logit, rounding
  // included, is the same whatever batch its row is sampled in.
  constexpr bool kHalfTiles = NW == 8;
  const int start = (kHalfTiles ? blockIdx.x % (2 * n_tiles) : 2 * (blockIdx.x / 2 % n_tiles)) * (KT / 2);
  const bool upper = r16 & 8;              // (of the chunks whose position in the row is r16)
  auto offset_of = [&](int t, bool upper_half) {
    int x = start + t * KT;
    if (x >= P.hidden_size) x -= P.hidden_size;
    if constexpr (!kHalfTiles) return x;
    const int wrapped = x + KT > P.hidden_size ? x - P.hidden_size : x;
    return upper_half ? wrapped : x;
  };

  // Embedding rows of this wave (rows past the vocabulary re-read its last row
  // and are masked at the end).  Load instruction j: lane l takes row
  // 4 j + l / 16, and of that row the chunk (l % 16) ^ row.
  const int vrow0 = blockIdx.x * (16 * NW) + 16 * wave;
  const uint16_t *wsrc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 4 * j + g;
    const int lrow = min(vrow0 + row, P.vocab - 1);
    wsrc[j] = P.weight + static_cast<int64_t>(lrow) * P.weight_stride + 8 * (r16 ^ row);
  }
  uint16_t *const wmine = &wtile[wave][0];

  // Hidden-state staging: thread -> (row tid / 16 + RPP j, 16-byte chunk tid % 16).
  const uint16_t *hsrc[SJ];
  bool hvalid[SJ], hstore[SJ];
#pragma unroll
  for (int j = 0; j < SJ; ++j) {
    const int row = (tid >> 4) + RPP * j;
    hstore[j] = row < ROWS;
    hvalid[j] = row < P.num_rows && hstore[j];
    const int src = hvalid[j] ? (P.row_index ? min(max(P.row_index[row], 0), P.hidden_rows - 1) : row) : 0;
    hsrc[j] = P.hidden + static_cast<int64_t>(src) * P.hidden_stride + 8 * (tid & 15);
  }
  const int hoff = (tid >> 4) * kHRow + 8 * (tid & 15);
  auto stage_load = [&](sm_u32x4 (&st)[SJ], int t) {
#pragma unroll
    for (int j = 0; j < SJ; ++j)
      st[j] = hvalid[j] ? *reinterpret_cast<const sm_u32x4 *>(hsrc[j] + offset_of(t, upper)) : sm_u32x4{0, 0, 0, 0};
  };
  auto stage_store = [&](const sm_u32x4 (&st)[SJ], int buf) {
#pragma unroll
    for (int j = 0; j < SJ; ++j)
      if (hstore[j]) *reinterpret_cast<sm_u32x4 *>(&htile[buf][hoff + RPP * j * kHRow]) = st[j];
  };
  auto load_w = [&](sm_u32x4 (&w)[4], int t) {
#pragma unroll
    for (int j = 0; j < 4; ++j)            // (row 4 j + g holds chunk r16 ^ row there)
      w[j] = __builtin_nontemporal_load(reinterpret_cast<const sm_u32x4 *>(wsrc[j] + offset_of(t, upper != (j >= 2))));
  };

  sm_v4f32 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = sm_v4f32{0.f, 0.f, 0.f, 0.f};
  // Regroup one embedding tile through the wave's LDS area, then multiply.
  auto consume = [&](const sm_u32x4 (&w)[4], int buf) {
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<sm_u32x4 *>(wmine + (4 * j) * KT + 8 * lane) = w[j];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    SmFrag a[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i)
      a[i].u = *reinterpret_cast<const sm_u32x4 *>(wmine + r16 * KT + 8 * ((4 * i + g) ^ r16));
    const uint16_t *base = &htile[buf][r16 * kHRow + 8 * g];
#pragma unroll
    for (int i = 0; i < NF; ++i) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        SmFrag b;
        b.u = *reinterpret_cast<const sm_u32x4 *>(base + 16 * nb * kHRow + 32 * i);
        if constexpr (__is_same(T, F16))
          acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i].h, b.h, acc[nb], 0, 0, 0);
        else
          acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].b, b.b, acc[nb], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();                    // fragment reads stay ahead of the next tile's writes
  };

  // PD tiles per wave are in flight: register sets used in rotation (unrolled,
  // so every set is addressed statically).  Loads return in order, so the
  // hidden-state part of a tile is requested together with - and just before -
  // its embedding part: waiting for one never waits for a younger tile.
  constexpr int PD = MUX_SM_PREFETCH_TILES;
  static_assert(PD % 2 == 0, "the hidden-state buffers alternate with the tile parity");
  sm_u32x4 w[PD][4], st[PD][SJ];
#pragma unroll
  for (int s2 = 0; s2 < PD; ++s2)
    if (s2 < n_tiles) {
      stage_load(st[s2], s2);
      load_w(w[s2], s2);
    }
  stage_store(st[0], 0);
  __syncthreads();
  for (int t0 = 0; t0 < n_tiles; t0 += PD) {
#pragma unroll
    for (int s2 = 0; s2 < PD; ++s2) {
      const int t = t0 + s2;
      if (t < n_tiles) {
        consume(w[s2], s2 & 1);
        if (t + 1 < n_tiles) stage_store(st[(s2 + 1) % PD], (s2 + 1) & 1);
        if (t + PD < n_tiles) {
          stage_load(st[s2], t + PD);
          load_w(w[s2], t + PD);
        }
        __syncthreads();
      }
    }
  }

  // Lane holds logits[vocab row vrow0 + 4 g + i][sampled row 16 nb + r16].
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    float bv = -__builtin_inff();
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int vr = vrow0 + 4 * g + i;
      const float val = sm_round<T>(acc[nb][i]);
      if (vr < P.vocab) take_better(bv, bi, val, vr);
    }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const float ov = __shfl_xor(bv, off);
      const int oi = __shfl_xor(bi, off);
      take_better(bv, bi, ov, oi);
    }
    if (g == 0) {
      red_v[wave][16 * nb + r16] = bv;
      red_i[wave][16 * nb + r16] = bi;
    }
  }
  __syncthreads();
  if (tid < ROWS) {
    float bv = red_v[0][tid];
    int bi = red_i[0][tid];
#pragma unroll
    for (int w = 1; w < NW; ++w) take_better(bv, bi, red_v[w][tid], red_i[w][tid]);
    store_key(P, static_cast<int64_t>(blockIdx.x) * ROWS + tid, bv, bi);
  }
  __shared__ unsigned long long fin[64 * NW];
  reduce_table<ROWS, 64 * NW>(P, fin, &s_last);
}

// ---------------------------------------------------------------------------
// More than 32 sampled rows: a matrix product with both operands through LDS.
// The kernel above reads one fragment of hidden states from LDS per MFMA (its
// waves are 16 vocabulary rows tall), which slows it from 33 rows on, and past
// 64 rows it would have to pass over the matrix once per 64.  Here eight waves
// share a tile of 128 vocabulary rows x 64 NB sampled rows as 2 x 4 waves of
// 64 x 16 NB, so that a fragment from LDS feeds NB (embedding) or four (hidden
// states) MFMAs.
//   * 128 rows per workgroup: a 32000-row vocabulary is 250 workgroups, one per
//     compute unit, one round.
//   * The hidden dimension is walked in tiles of 64 (a 128-byte line per row).  A
//     tile goes from global memory straight into LDS, NBUF - 1 tiles ahead, one
//     barrier per tile, 16-byte chunk c of a row at position c ^ (row % 8): no bank
//     conflicts.  NBUF is what 160 KB hold (at most 5).
// 32000 x 4096, us (tiles staged through registers and the reduction in one level / as
// here, both in turn on one machine): 33 rows 47.2 / 46.0, 64 rows 48.4 / 47.5, 128 rows
// 57.7 / 54.6, 192 rows 70 / 64, 256 rows 85.4 / 76.1; 16000 x 4096, 64 rows 37.7 / 37.9;
// 128256 x 4096 bf16, 256 rows 334 / 298.  Up to 64 rows it is bound by HBM (5.5 TB/s).  With 256 rows the clock is 1.66 GHz and LDS is the busiest unit: 128 KB
// of fragments and 48 KB of tiles in per 1024 cycles of MFMA and compute unit, at 128
// bytes a cycle.  Fewer fragment reads cost more than they save: four waves of 64 x
// 32 NB (a quarter less) 80, four waves of 128 x 16 NB with the hidden states straight
// from global memory in registers (half of it) 100 before the reduction, one wave per
// SIMD hides neither the barrier nor the latencies.
// The reduction is the one above with 64 NB columns per table line.  At 256 columns one
// workgroup reads 32 lines per round of loads (two slices of sixteen), the 250 lines of
// 32000 rows in 8 rounds; beyond 64 workgroups, 2 rounds at that width, it takes two
// levels: groups of 16, or 32 groups (one level / two: 32000 x 4096, 256 rows 84.5 / 79,
// 128 rows 56.2 / 54.3; 128256 x 4096, 256 rows 331 / 304; 9000 rows, 71 workgroups, 62.5 /
// 61.8).  Fewer columns read more lines per round, so there the line could lie higher.
constexpr size_t kSmCounterBytes = 256;    // the arrival counters, in front of the table
constexpr int kSmOneLevelWgs = 64, kSmGroupWgs = 16, kSmMaxGroups = 32;
template <typename T, int NB, int NBUF>
__global__ __launch_bounds__(512, 2) void lm_head_argmax_wide_kernel(const LmHeadParams P) {
  constexpr int KT = 64;                   // hidden elements per tile
  constexpr int ROWS = 64 * NB;            // sampled rows
  constexpr int VR = 128;                  // vocabulary rows
  constexpr int NW = 8;
  constexpr int kMfma = 0x8, kDsRead = 0x100;   // instruction classes of the scheduler
  constexpr int TILE = (VR + ROWS) * KT;   // elements of one LDS buffer: embedding rows, then hidden rows
  __shared__ __attribute__((aligned(16))) uint16_t tile[NBUF][TILE];
  __shared__ float red_v[2][ROWS];
  __shared__ int red_i[2][ROWS];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int r16 = lane & 15, g = lane >> 4;
  const int n_tiles = P.hidden_size / KT;
  // The same element as in the kernel above.
  const int t_start = P.half_tiles ? blockIdx.x % n_tiles : 2 * (blockIdx.x % (n_tiles / 2));
  const int vrow0 = blockIdx.x * VR;

  // Staging, global memory to LDS: instruction j of wave w fills 8 rows of a tile
  // (lane l's 16 bytes land at base + 16 l: row l / 8, position l % 8, which holds
  // chunk (l % 8) ^ (l / 8)).  Rows past the vocabulary re-read its last row (masked
  // at the end), sampled rows past the last re-read a valid one (not stored).
  const int srow = 8 * wave + (lane >> 3), schunk = (lane & 7) ^ (lane >> 3);
  const uint16_t *src[2 + NB];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    src[j] = P.weight + static_cast<int64_t>(min(vrow0 + srow + 64 * j, P.vocab - 1)) * P.weight_stride + 8 * schunk;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int row = min(srow + 64 * j, P.num_rows - 1);
    const int r = P.row_index ? min(max(P.row_index[row], 0), P.hidden_rows - 1) : row;
    src[2 + j] = P.hidden + static_cast<int64_t>(r) * P.hidden_stride + 8 * schunk;
  }
  typedef const __attribute__((address_space(3))) uint16_t lds_u16;
  const uint32_t tile_at = (uint32_t)(uintptr_t)(lds_u16 *)&tile[0][0];
  auto load = [&](int t, int buf) {
    int x = t + t_start;
    x = (x >= n_tiles ? x - n_tiles : x) * KT;
    const uint32_t at = tile_at + 2 * (buf * TILE + 8 * wave * KT);
#pragma unroll
    for (int j = 2; j < 2 + NB; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at + 2 * 64 * j * KT), "v"(src[j] + x)
                   : "memory", "m0");
#pragma unroll
    for (int j = 0; j < 2; ++j)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(at + 2 * 64 * j * KT), "v"(src[j] + x)
                   : "memory", "m0");
  };

  sm_v4f32 acc[4][NB];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = sm_v4f32{0.f, 0.f, 0.f, 0.f};
  // Fragments of one half (32 of the 64 hidden elements) of a tile, and their products.
  struct Half {
    SmFrag a[4], b[NB];
  };
  auto read_half = [&](Half &f, int buf, int kk) {
    const int chunk = 8 * ((4 * kk + g) ^ (r16 & 7));
    const uint16_t *const wt = &tile[buf][(64 * wm + r16) * KT + chunk];
    const uint16_t *const ht = &tile[buf][(VR + 16 * NB * wn + r16) * KT + chunk];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) f.a[mb].u = *reinterpret_cast<const sm_u32x4 *>(wt + 16 * mb * KT);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) f.b[nb].u = *reinterpret_cast<const sm_u32x4 *>(ht + 16 * nb * KT);
  };
  auto multiply = [&](const Half &f) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        if constexpr (__is_same(T, F16))
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.a[mb].h, f.b[nb].h, acc[mb][nb], 0, 0, 0);
        else
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[mb].b, f.b[nb].b, acc[mb][nb], 0, 0, 0);
      }
  };

#pragma unroll
  for (int t = 0; t < NBUF - 1; ++t)
    if (t < n_tiles) load(t, t);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  Half f0, f1;
  read_half(f0, 0, 0);
  int buf = 0;
  for (int t = 0; t < n_tiles; ++t) {
    const int next = buf + 1 == NBUF ? 0 : buf + 1;
    const bool more = t + NBUF - 1 < n_tiles;
    if (more) load(t + NBUF - 1, buf == 0 ? NBUF - 1 : buf - 1);
    read_half(f1, buf, 1);
    multiply(f0);
#pragma unroll
    for (int i = 0; i < 4 + NB; ++i) {
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kMfma, 4 * NB, 0);
    __builtin_amdgcn_sched_barrier(0);
    // This wave's part of the next tile has landed, and f1 has been read: behind the
    // barrier the other waves load into its buffer.
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * (2 + NB)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read_half(f0, next, 0);              // (behind the last tile: some buffer, not used)
    multiply(f1);
#pragma unroll
    for (int i = 0; i < 4 + NB; ++i) {
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kMfma, 4 * NB, 0);
    __builtin_amdgcn_sched_barrier(0);
    buf = next;
  }
  __syncthreads();

  // Lane holds logits[vocab row vrow0 + 64 wm + 16 mb + 4 g + i][sampled row 16 (NB wn + nb) + r16].
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    float bv = -__builtin_inff();
    int bi = 0x7fffffff;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vr = vrow0 + 64 * wm + 16 * mb + 4 * g + i;
        const float val = sm_round<T>(acc[mb][nb][i]);
        if (vr < P.vocab) take_better(bv, bi, val, vr);
      }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const float ov = __shfl_xor(bv, off);
      const int oi = __shfl_xor(bi, off);
      take_better(bv, bi, ov, oi);
    }
    if (g == 0) {
      red_v[wm][16 * (NB * wn + nb) + r16] = bv;
      red_i[wm][16 * (NB * wn + nb) + r16] = bi;
    }
  }
  __syncthreads();
  if (tid < ROWS) {
    float bv = red_v[0][tid];
    int bi = red_i[0][tid];
    take_better(bv, bi, red_v[1][tid], red_i[1][tid]);
    store_key(P, static_cast<int64_t>(blockIdx.x) * ROWS + tid, bv, bi);
  }
  unsigned long long *const fin = reinterpret_cast<unsigned long long *>(&tile[0][0]);
  const int n_wg = gridDim.x;
  if (n_wg <= kSmOneLevelWgs) {
    reduce_table<ROWS, 64 * NW>(P, fin, &s_last);
    return;
  }
  // Two levels: the last workgroup of a group leaves the group's maxima in the
  // group's first line (each thread in the column it has read itself), the last of
  // these reduces the groups' lines.
  const int per_group = max(kSmGroupWgs, (n_wg + kSmMaxGroups - 1) / kSmMaxGroups);
  const int group = blockIdx.x / per_group, first = group * per_group, groups = (n_wg + per_group - 1) / per_group;
  const int members = min(per_group, n_wg - first);
  uint32_t *const group_counter = P.counter + 1 + group;
  if (!last_to_arrive(group_counter, members, &s_last)) return;
  unsigned long long key = reduce_lines<ROWS, 64 * NW>(P, first, members, 1, fin);
  if (tid < ROWS)
    __hip_atomic_store(&P.table[static_cast<int64_t>(first) * ROWS + tid], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  clear_counter(group_counter);
  if (!last_to_arrive(P.counter, groups, &s_last)) return;
  key = reduce_lines<ROWS, 64 * NW>(P, 0, groups, per_group, fin);
  if (tid < P.num_rows) store_token(P, tid, key);
  clear_counter(P.counter);
}

__global__ void sampler_zero_kernel(uint32_t *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

static_assert(4 * (1 + kSmMaxGroups) <= kSmCounterBytes, "the counters fit in front of the table");
#ifndef MUX_SM_EIGHT_WAVE_MIN_WGS
#define MUX_SM_EIGHT_WAVE_MIN_WGS 192
#endif
constexpr int kSmEightWaveMinWgs = MUX_SM_EIGHT_WAVE_MIN_WGS;

}  // namespace mux

extern "C" size_t mux_greedy_sample_workspace_bytes(int32_t vocab_size) {
  if (vocab_size <= 0) return 0;
  // The largest table: 128 vocabulary rows per workgroup, a key per sampled row of a pass.
  const size_t n_wg = (static_cast<size_t>(vocab_size) + 127) / 128;
  return mux::kSmCounterBytes + n_wg * mux::kSmMaxRowsPerPass * sizeof(unsigned long long);
}

extern "C" int32_t mux_greedy_sample_workspace_init(void *workspace, size_t workspace_bytes, void *stream) {
  using namespace mux;
  if (!workspace || workspace_bytes < kSmCounterBytes || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return MUXA_EWORKSPACE;
  hipLaunchKernelGGL(sampler_zero_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<uint32_t *>(workspace), static_cast<int>(kSmCounterBytes / 4));
  MUX_HIP_TRY(hipGetLastError());
  return MUXA_OK;
}

extern "C" int32_t mux_greedy_sample(int64_t *next_tokens, const void *hidden_states, int64_t hidden_row_stride,
                                     int32_t num_hidden_rows, const int32_t *row_index, int32_t num_rows,
                                     const void *embedding,
                                     int64_t embedding_row_stride, int32_t embedding_rows, int32_t vocab_size,
                                     int32_t hidden_size, int32_t dtype, void *workspace, size_t workspace_bytes,
                                     void *stream) {
  using namespace mux;
  // (pointers are only required when there is something to do)
  if (num_rows > 0 && (!next_tokens || !hidden_states || !embedding)) return MUXA_EINVAL;
  if (num_rows < 0 || vocab_size <= 0 || hidden_size <= 0 || embedding_rows < vocab_size) return MUXA_EINVAL;
  if (num_hidden_rows < 1 || (!row_index && num_rows > num_hidden_rows)) return MUXA_EINVAL;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  if (hidden_size % kSmTile) return MUXA_EUNSUPPORTED;
  if (hidden_row_stride < hidden_size || embedding_row_stride < hidden_size || hidden_row_stride % 8 ||
      embedding_row_stride % 8)
    return MUXA_EINVAL;
  if ((reinterpret_cast<uintptr_t>(hidden_states) | reinterpret_cast<uintptr_t>(embedding)) & 15u)
    return MUXA_EINVAL;
  if (num_rows == 0) return MUXA_OK;
  if (!workspace || workspace_bytes < mux_greedy_sample_workspace_bytes(vocab_size) ||
      (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return MUXA_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // Up to 32 sampled rows: 128 vocabulary rows per workgroup (8 waves) once that
  // still gives the chip enough workgroups, else 64.
  const bool wide = (vocab_size + 127) / 128 >= kSmEightWaveMinWgs;
  const int rows_per_wg = wide ? 128 : 64;
  const int n_wg = (vocab_size + rows_per_wg - 1) / rows_per_wg;
  // At most 256 sampled rows per pass over the matrix; larger batches take
  // several passes, one after the other on the stream.
  for (int r0 = 0; r0 < num_rows; r0 += kSmMaxRowsPerPass) {
    const int rows = min(num_rows - r0, kSmMaxRowsPerPass);
    LmHeadParams P;
    P.hidden = static_cast<const uint16_t *>(hidden_states) + (row_index ? 0 : static_cast<int64_t>(r0) * hidden_row_stride);
    P.hidden_stride = hidden_row_stride;
    P.row_index = row_index ? row_index + r0 : nullptr;
    P.weight = static_cast<const uint16_t *>(embedding);
    P.weight_stride = embedding_row_stride;
    P.hidden_size = hidden_size;
    P.vocab = vocab_size;
    P.num_rows = rows;
    P.half_tiles = wide;
    P.hidden_rows = row_index ? num_hidden_rows : num_hidden_rows - r0;
    P.counter = static_cast<uint32_t *>(workspace);
    P.table = reinterpret_cast<unsigned long long *>(static_cast<char *>(workspace) + kSmCounterBytes);
    P.next_tokens = next_tokens + r0;
    const int nb = rows <= 16 ? 1 : 2;
    if (rows > kSmNarrowRows) {
      const dim3 wide_grid((vocab_size + 127) / 128);
#define MUX_LM_WIDE(TT)                                                                                            \
  do {                                                                                                            \
    if (rows <= 64) hipLaunchKernelGGL((lm_head_argmax_wide_kernel<TT, 1, 5>), wide_grid, dim3(512), 0, st, P);   \
    else if (rows <= 128) hipLaunchKernelGGL((lm_head_argmax_wide_kernel<TT, 2, 4>), wide_grid, dim3(512), 0, st, P); \
    else if (rows <= 192) hipLaunchKernelGGL((lm_head_argmax_wide_kernel<TT, 3, 3>), wide_grid, dim3(512), 0, st, P); \
    else hipLaunchKernelGGL((lm_head_argmax_wide_kernel<TT, 4, 3>), wide_grid, dim3(512), 0, st, P);              \
  } while (0)
      if (dtype == MUXA_DTYPE_F16) MUX_LM_WIDE(F16);
      else MUX_LM_WIDE(BF16);
#undef MUX_LM_WIDE
      continue;
    }
    const dim3 grid(n_wg);
#define MUX_LM_GO(TT, NBV, NWV) \
  hipLaunchKernelGGL((lm_head_argmax_kernel<TT, NBV, NWV>), grid, dim3(64 * NWV), 0, st, P)
#define MUX_LM_LAUNCH(TT)                    \
  do {                                       \
    if (!wide) {                             \
      if (nb == 1) MUX_LM_GO(TT, 1, 4);      \
      else MUX_LM_GO(TT, 2, 4);              \
    } else if (nb == 1) MUX_LM_GO(TT, 1, 8); \
    else MUX_LM_GO(TT, 2, 8);                \
  } while (0)
    if (dtype == MUXA_DTYPE_F16) MUX_LM_LAUNCH(F16);
    else MUX_LM_LAUNCH(BF16);
#undef MUX_LM_LAUNCH
#undef MUX_LM_GO
  }
  MUX_HIP_TRY(hipGetLastError());
  return MUXA_OK;
}
