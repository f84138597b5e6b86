// RMSNorm and SiluAndMul for gfx950: the two element-wise operators of a LLaMA
// layer next to the attention (muxserve/flexserver/models/llama.py:75-81,
// 200-232).  Both are bound by HBM: every input element is read once and every
// output element written once, in 16-byte pieces.
//
//   rms_norm      one workgroup (a wave for short rows) per token row at a time: the row
//                 stays in registers between the sum of squares and the scaling, so x
//                 is read once (with non-temporal loads), the weight once per workgroup.
//                 out = T(x * rsqrt(mean(x^2) + eps)) * w, the product in T.
//   silu_and_mul  one thread per 8 outputs: out = T(a / (1 + exp(-a))) * b for
//                 x = [a | b], the product in T.
#include <algorithm>

#include "mux_common.h"

namespace mux {

typedef uint32_t mo_u32x4 __attribute__((ext_vector_type(4)));

// Workgroups per compute unit of rms_norm.  4096 rows of 6656 f16: 2, 3, 4, 6, 8 of them
// 22.2, 20.8, 21.4, 21.6, 21.8 us, one workgroup per row 22.4; 2048 of 8192 14.2, 13.3, 14.2,
// 14.6, 14.7, 14.7.
constexpr int kRmsWgsPerCu = 3;
// A wave per row up to this row length, and up to twice that beyond 1024 rows; such
// workgroups per compute unit (2, 4, 8 of them, 8192 rows of 512 f16: 4.71, 4.44, 4.27 us).
// us, f16, a workgroup / a wave per row: 8192 rows of 512 7.5 / 4.3, of 1024 9.6 / 6.6, of 1536
// 12.0 / 10.0, of 2048 13.8 / 13.9; 4096 of 1032 6.0 / 4.7, of 2048 7.4 / 6.7; 256 of 1536 2.60 /
// 2.76, of 512 2.52 / 2.49.
constexpr int kRmsWaveHidden = 1024, kRmsWaveWgsPerCu = 8;

template <typename T>
__device__ __forceinline__ void unpack8(const mo_u32x4 v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (__is_same(T, F16)) {
      const half2_t h = as_half2(w[i]);
      f[2 * i] = static_cast<float>(h.x);
      f[2 * i + 1] = static_cast<float>(h.y);
    } else {
      f[2 * i] = bf16_lo(w[i]);
      f[2 * i + 1] = bf16_hi(w[i]);
    }
  }
}

template <typename T>
__device__ __forceinline__ float round_to(float f) {         // the value of f after one rounding to T
  if constexpr (__is_same(T, F16)) return static_cast<float>(static_cast<_Float16>(f));
  else return __uint_as_float(static_cast<uint32_t>(f32_to_bf16_bits(f)) << 16);
}

template <typename T>
__device__ __forceinline__ mo_u32x4 pack8(const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w[i] = to_storage2<T>(f[2 * i], f[2 * i + 1]);
  return mo_u32x4{w[0], w[1], w[2], w[3]};
}

// CPT = 16-byte chunks of a row that a thread keeps (thread t takes chunks t, t + 256,
// ...).  A workgroup walks rows blockIdx, blockIdx + gridDim, ... with the next row's
// loads issued before the current row is reduced and stored, so that across the chip
// reads and writes overlap instead of coming as one burst of each.  CPT = 0: rows of any
// length, x read twice.
// us, a wave per row (2048 of them, otherwise the same) / a workgroup per row: 64 rows of
// 8192 6.2 / 3.6, 1024 of 4096 6.6 / 5.9, 2048 of 5120 10.5 / 9.3, 16384 of 4096 53.5 / 49.7,
// 4096 of 6656 20.4 / 20.8 by themselves, 85.1 / 84.0 with silu_and_mul behind them.  Non-
// temporal stores make this kernel 6 - 19 % faster and the one that reads its output
// slower by more (4096 of 6656 and a read 37 / 40 us).
// WAVES per row: 4, the workgroup, or 1 for short rows, which leave most of a workgroup idle.
template <typename T, int CPT, int WAVES = 4>
__global__ __launch_bounds__(256) void rms_norm_kernel(uint16_t *__restrict__ out, int64_t out_stride,
                                                       const uint16_t *__restrict__ x, int64_t x_stride,
                                                       const uint16_t *__restrict__ weight, float eps, int hidden,
                                                       int num_rows) {
  __shared__ float part[2][4];             // the waves' sums, two rows
  constexpr int TPR = 64 * WAVES, RPW = 4 / WAVES;       // threads per row, rows per workgroup at a time
  const int tid = WAVES == 4 ? threadIdx.x : threadIdx.x & 63, nchunks = hidden >> 3;
  const int step = gridDim.x * RPW;
  const int first = WAVES == 4 ? blockIdx.x : blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (WAVES == 1 && first >= num_rows) return;
  const mo_u32x4 *wr = reinterpret_cast<const mo_u32x4 *>(weight);
  const float inv_n = 1.0f / static_cast<float>(hidden);
  // rsqrt(mean + eps) of a row from a thread's part of its sum of squares.  (The barrier
  // by itself: __syncthreads() would wait for the previous row's stores.)
  auto scale_of = [&](float ss, int buf) {
    ss = wave_sum(ss);
    if constexpr (WAVES == 1) return rsqrtf(ss * inv_n + eps);
    if ((tid & 63) == 0) part[buf][tid >> 6] = ss;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    return rsqrtf((part[buf][0] + part[buf][1] + part[buf][2] + part[buf][3]) * inv_n + eps);
  };
  auto scaled = [&](const mo_u32x4 v, const mo_u32x4 w, float s) {
    float f[8], g[8];
    unpack8<T>(v, f);
    unpack8<T>(w, g);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = round_to<T>(f[j] * s) * g[j];
    return pack8<T>(f);
  };
  auto add_squares = [](const mo_u32x4 v, float ss) {
    float f[8];
    unpack8<T>(v, f);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(f[j], f[j], ss);
    return ss;
  };
  if constexpr (CPT > 0) {
    const mo_u32x4 zero = {0, 0, 0, 0};
    auto load_row = [&](mo_u32x4 (&v)[CPT], int row) {
      const mo_u32x4 *xr = reinterpret_cast<const mo_u32x4 *>(x + row * x_stride);
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int c = tid + TPR * i;
        v[i] = c < nchunks ? __builtin_nontemporal_load(&xr[c]) : zero;
      }
    };
    mo_u32x4 w[CPT];
    auto finish_row = [&](const mo_u32x4 (&v)[CPT], int row, int buf) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < CPT; ++i) ss = add_squares(v[i], ss);
      const float s = scale_of(ss, buf);
      mo_u32x4 *outr = reinterpret_cast<mo_u32x4 *>(out + row * out_stride);
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int c = tid + TPR * i;
        if (c < nchunks) outr[c] = scaled(v[i], w[i], s);
      }
    };
    mo_u32x4 a[CPT], b[CPT];
    int row = first;
    load_row(a, row);
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + TPR * i;
      w[i] = c < nchunks ? wr[c] : zero;
    }
    for (; row < num_rows; row += 2 * step) {
      if (row + step < num_rows) load_row(b, row + step);
      finish_row(a, row, 0);
      if (row + step >= num_rows) break;
      if (row + 2 * step < num_rows) load_row(a, row + 2 * step);
      finish_row(b, row + step, 1);
    }
  } else {
    int buf = 0;
    for (int row = first; row < num_rows; row += step, buf ^= 1) {
      const mo_u32x4 *xr = reinterpret_cast<const mo_u32x4 *>(x + row * x_stride);
      mo_u32x4 *outr = reinterpret_cast<mo_u32x4 *>(out + row * out_stride);
      float ss = 0.f;
      for (int c = tid; c < nchunks; c += TPR) ss = add_squares(xr[c], ss);
      const float s = scale_of(ss, buf);
      for (int c = tid; c < nchunks; c += TPR) outr[c] = scaled(xr[c], wr[c], s);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(uint16_t *__restrict__ out, int64_t out_stride,
                                                           const uint16_t *__restrict__ x, int64_t x_stride,
                                                           int d8, int64_t total) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  const int64_t t = id / d8;
  const int c = static_cast<int>(id - t * d8);
  const mo_u32x4 *xr = reinterpret_cast<const mo_u32x4 *>(x + t * x_stride);
  const mo_u32x4 av = __builtin_nontemporal_load(&xr[c]), bv = __builtin_nontemporal_load(&xr[d8 + c]);
  float a[8], b[8];
  unpack8<T>(av, a);
  unpack8<T>(bv, b);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float e = fast_exp2(-1.4426950408889634f * a[j]);
    a[j] = round_to<T>(a[j] * __builtin_amdgcn_rcpf(1.0f + e)) * b[j];
  }
  reinterpret_cast<mo_u32x4 *>(out + t * out_stride)[c] = pack8<T>(a);
}

}  // namespace mux

extern "C" int32_t mux_rms_norm(void *out, int64_t out_row_stride, const void *x, int64_t x_row_stride,
                                const void *weight, float eps, int32_t num_tokens, int32_t hidden_size,
                                int32_t dtype, void *stream) {
  using namespace mux;
  // (pointers are only required when there is something to do)
  if (num_tokens > 0 && (!out || !x || !weight)) return MUXA_EINVAL;
  if (num_tokens < 0 || hidden_size <= 0 || !(eps >= 0.f)) return MUXA_EINVAL;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  if (hidden_size % 8) return MUXA_EUNSUPPORTED;
  if (out_row_stride < hidden_size || x_row_stride < hidden_size || out_row_stride % 8 || x_row_stride % 8)
    return MUXA_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight)) & 15u)
    return MUXA_EINVAL;
  if (num_tokens == 0) return MUXA_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // At most so many workgroups per CU; rows beyond that are walked in sequence.
  static const int cus = [] {                      // compute units of the current device, asked once
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      return v;
    return 256;
  }();
  const bool wave = hidden_size <= kRmsWaveHidden || (hidden_size <= 2 * kRmsWaveHidden && num_tokens > 1024);
  const dim3 grid(wave ? std::min((num_tokens + 3) / 4, cus * kRmsWaveWgsPerCu) : std::min(num_tokens, cus * kRmsWgsPerCu));
  const dim3 block(256);
  uint16_t *o = static_cast<uint16_t *>(out);
  const uint16_t *xi = static_cast<const uint16_t *>(x), *w = static_cast<const uint16_t *>(weight);
  const int nchunks = hidden_size / 8;
#define MUX_RMS_LAUNCH(...)                                                                              \
  hipLaunchKernelGGL((rms_norm_kernel<__VA_ARGS__>), grid, block, 0, st, o, out_row_stride, xi, x_row_stride, w, \
                     eps, hidden_size, num_tokens)
#define MUX_RMS_PICK(TT)                              \
  do {                                                \
    if (wave && nchunks <= 64 * 1) MUX_RMS_LAUNCH(TT, 1, 1); \
    else if (wave && nchunks <= 64 * 2) MUX_RMS_LAUNCH(TT, 2, 1); \
    else if (wave) MUX_RMS_LAUNCH(TT, 4, 1);            \
    else if (nchunks <= 256 * 1) MUX_RMS_LAUNCH(TT, 1); \
    else if (nchunks <= 256 * 2) MUX_RMS_LAUNCH(TT, 2); \
    else if (nchunks <= 256 * 3) MUX_RMS_LAUNCH(TT, 3); \
    else if (nchunks <= 256 * 4) MUX_RMS_LAUNCH(TT, 4); \
    else MUX_RMS_LAUNCH(TT, 0);                       \
  } while (0)
  if (dtype == MUXA_DTYPE_F16) MUX_RMS_PICK(F16);
  else MUX_RMS_PICK(BF16);
#undef MUX_RMS_PICK
#undef MUX_RMS_LAUNCH
  MUX_HIP_TRY(hipGetLastError());
  return MUXA_OK;
}

extern "C" int32_t mux_silu_and_mul(void *out, int64_t out_row_stride, const void *x, int64_t x_row_stride,
                                    int32_t num_tokens, int32_t d, int32_t dtype, void *stream) {
  using namespace mux;
  if (num_tokens > 0 && (!out || !x)) return MUXA_EINVAL;
  if (num_tokens < 0 || d <= 0) return MUXA_EINVAL;
  if (dtype != MUXA_DTYPE_F16 && dtype != MUXA_DTYPE_BF16) return MUXA_EUNSUPPORTED;
  if (d % 8) return MUXA_EUNSUPPORTED;
  if (out_row_stride < d || x_row_stride < 2 * static_cast<int64_t>(d) || out_row_stride % 8 || x_row_stride % 8)
    return MUXA_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(x)) & 15u) return MUXA_EINVAL;
  if (num_tokens == 0) return MUXA_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int d8 = d / 8;
  const int64_t total = static_cast<int64_t>(num_tokens) * d8;
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffffLL) return MUXA_EUNSUPPORTED;
  const dim3 grid(static_cast<uint32_t>(blocks)), block(256);
  if (dtype == MUXA_DTYPE_F16)
    hipLaunchKernelGGL(silu_and_mul_kernel<F16>, grid, block, 0, st, static_cast<uint16_t *>(out), out_row_stride,
                       static_cast<const uint16_t *>(x), x_row_stride, d8, total);
  else
    hipLaunchKernelGGL(silu_and_mul_kernel<BF16>, grid, block, 0, st, static_cast<uint16_t *>(out), out_row_stride,
                       static_cast<const uint16_t *>(x), x_row_stride, d8, total);
  MUX_HIP_TRY(hipGetLastError());
  return MUXA_OK;
}
