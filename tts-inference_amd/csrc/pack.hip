// Weight packers and per-token activation quantization.
//
// Load-time packers (int8, e4m3) and the run-time fp8 and int8 activation quantizers.  One
// workgroup of 256 threads owns one row: a coalesced pass finds the row's absmax,
// a second pass divides, rounds and stores; the 16-bit aligned rows have vector forms that hold the
// row in registers between the two (the packers': one wave a row).  All arithmetic is IEEE fp32 (hipcc's
// default correctly-rounded division; no fast-math), so results are bit-exact with
// the reference's torch expressions (see the oracle tests).
#include "common.h"

namespace qtts {

constexpr int kPackThreads = 256;

template <typename T>
__device__ __forceinline__ float row_absmax(const T* __restrict__ row, int64_t k, float* red) {
  float m = 0.0f;
  for (int64_t c = threadIdx.x; c < k; c += kPackThreads) m = fmaxf(m, fabsf(to_f32(row[c])));
  m = wave_max(m);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return m;
}

// quantize_weight_per_channel, qtts/quant/int8.py:45-56 (+ stored scale cast, :105).
template <typename SrcT, typename StoreT>
__global__ __launch_bounds__(kPackThreads) void pack_int8_kernel(
    const SrcT* __restrict__ src, int64_t k, int64_t ld, int8_t* __restrict__ q,
    StoreT* __restrict__ scale_out, float* __restrict__ scale_f32, int div_mode) {
  __shared__ float red[4];
  const int64_t r = blockIdx.x;
  const SrcT* row = src + r * ld;
  float amax = row_absmax(row, k, red);
  amax = fmaxf(amax, 1e-12f);  // clamp_min(1e-12)
  const float scale = scalar_div(amax, 127.0f, div_mode);
  int8_t* qrow = q + r * k;
  for (int64_t c = threadIdx.x; c < k; c += kPackThreads) {
    float v = __builtin_rintf(to_f32(row[c]) / scale);  // round half to even
    v = fminf(fmaxf(v, -127.0f), 127.0f);
    qrow[c] = (int8_t)(int)v;
  }
  if (threadIdx.x == 0) {
    scale_out[r] = from_f32<StoreT>(scale);
    if (scale_f32) scale_f32[r] = scale;
  }
}

// quantize_weight_fp8, qtts/quant/fp8.py:45-49.
template <typename SrcT>
__global__ __launch_bounds__(kPackThreads) void pack_fp8_kernel(
    const SrcT* __restrict__ src, int64_t k, int64_t ld, uint8_t* __restrict__ q,
    float* __restrict__ scale_out, int div_mode) {
  __shared__ float red[4];
  const int64_t r = blockIdx.x;
  const SrcT* row = src + r * ld;
  float amax = fmaxf(row_absmax(row, k, red), 1e-12f);
  const float scale = scalar_div(amax, 448.0f, div_mode);
  uint8_t* qrow = q + r * k;
  for (int64_t c = threadIdx.x; c < k; c += kPackThreads) qrow[c] = (uint8_t)e4m3_encode(to_f32(row[c]) / scale);
  if (threadIdx.x == 0) scale_out[r] = scale;
}

// Vector form of the two packers: 16-bit rows of up to 8192 columns, 16-byte aligned, k % 8 == 0.  One wave
// a row, 4 rows a workgroup; lane l holds vectors l, l + 64, ... (8 elements each) of the row in
// registers, so the row is read once, in one round trip, and no workgroup barrier stands between the absmax and the
// codes.  The quotients are the IEEE ones, from the row's reciprocal and one FMA correction (div_by); a row
// whose sum of squares is not finite (an infinity, a NaN, values past 2^63) divides and encodes as the scalar
// kernel does.  Bound by HBM: 12288 x 2048 bf16 moves 75.6 MB, 14.7 us at a copy's 5.1 TB/s; int8 / e4m3 46.0 / 53.7 us
// with the scalar kernel, 17.4 / 14.3 with this one.
template <typename SrcT, int V, bool FP8, typename StoreT>
__global__ __launch_bounds__(kPackThreads) void pack_vec_kernel(const SrcT* __restrict__ src, int64_t n, int k, int64_t ld,
                                                                uint8_t* __restrict__ q, StoreT* __restrict__ scale_out,
                                                                float* __restrict__ scale_f32, int div_mode) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * (kPackThreads / 64) + (threadIdx.x >> 6);
  if (r >= n) return;
  const int nv = k >> 3;
  const SrcT* row = src + r * ld;
  i32x4_t v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = *(const i32x4_t*)(row + 8 * min(lane + 64 * j, nv - 1));  // clamped: repeats the last
  float mx = 0.0f, ss = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t p = (uint32_t)v[j][e];
      mx = fmaxf(mx, fmaxf(fabsf(to_f32(SrcT{(uint16_t)p})), fabsf(to_f32(SrcT{(uint16_t)(p >> 16)}))));
      ss = sq2_acc<SrcT>(p, ss);
    }
  const bool finite = !__any(!(ss <= 3.402823466e38f));
  mx = fmaxf(group_max<64>(mx), 1e-12f);  // clamp_min(1e-12)
  const float scale = scalar_div(mx, FP8 ? 448.0f : 127.0f, div_mode), rs = 1.0f / scale;
  auto store = [&](auto div, auto plain) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int idx = lane + 64 * j;
      if (idx >= nv) continue;
      uint32_t w[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t p0 = (uint32_t)v[j][2 * h], p1 = (uint32_t)v[j][2 * h + 1];
        const float f[4] = {div(to_f32(SrcT{(uint16_t)p0})), div(to_f32(SrcT{(uint16_t)(p0 >> 16)})),
                            div(to_f32(SrcT{(uint16_t)p1})), div(to_f32(SrcT{(uint16_t)(p1 >> 16)}))};
        uint32_t o = 0;
        if constexpr (FP8 && decltype(plain)::value) {
#pragma unroll
          for (int i = 0; i < 4; ++i) o |= e4m3_encode(f[i]) << (8 * i);
        } else if constexpr (FP8) {
          o = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false) & 0xffffu;
          o |= (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], 0, false) << 16;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {  // round half to even, clamp
            const int c = (int)fminf(fmaxf(__builtin_rintf(f[i]), -127.0f), 127.0f);
            o |= ((uint32_t)c & 0xffu) << (8 * i);
          }
        }
        w[h] = o;
      }
      *(uint2*)(q + r * k + 8 * idx) = make_uint2(w[0], w[1]);
    }
  };
  if (finite) store([&](float x) { return div_by(x, scale, rs); }, std::false_type{});
  else store([&](float x) { return x / scale; }, std::true_type{});
  if (lane == 0) {
    scale_out[r] = from_f32<StoreT>(scale);
    if (scale_f32) scale_f32[r] = scale;
  }
}

// Activation half of Fp8Method.apply, qtts/quant/fp8.py:77-78.  The absmax and the
// 1e-6 clamp happen in the activation dtype (exact for max/abs; the clamp value is
// 1e-6 rounded to that dtype), then the scale is formed in fp32.
template <typename XT>
__global__ __launch_bounds__(kPackThreads) void quant_act_fp8_kernel(
    const XT* __restrict__ x, int64_t k, int64_t ld, uint8_t* __restrict__ qx,
    float* __restrict__ sx, int div_mode) {
  __shared__ float red[4];
  const int64_t r = blockIdx.x;
  const XT* row = x + r * ld;
  const float floor_v = round_through<XT>(1e-6f);
  const float amax = fmaxf(row_absmax(row, k, red), floor_v);
  const float s = scalar_div(amax, 448.0f, div_mode);
  uint8_t* qrow = qx + r * k;
  for (int64_t c = threadIdx.x; c < k; c += kPackThreads) qrow[c] = (uint8_t)e4m3_encode(to_f32(row[c]) / s);
  if (threadIdx.x == 0) sx[r] = s;
}

// Vectorized quant_act_fp8_kernel for 16-bit activations with 16-byte aligned rows and
// k % 8 == 0: every thread loads up to V 8-element vectors of its row at once (one
// memory round trip), the row maximum goes through one LDS exchange, and the codes
// come from a correctly rounded quotient (the row's reciprocal plus one FMA
// correction) and v_cvt_pk_fp8_f32 -- the same codes as the scalar kernel.
template <typename XT, int V>
__global__ __launch_bounds__(kPackThreads) void quant_act_fp8_vec_kernel(
    const XT* __restrict__ x, int64_t k, int64_t ld, uint8_t* __restrict__ qx,
    float* __restrict__ sx, int div_mode) {
  __shared__ float red[kPackThreads / 64];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int nv = (int)(k >> 3);
  const XT* row = x + r * ld;
  i32x4_t v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int idx = tid + kPackThreads * j;
    v[j] = *(const i32x4_t*)(row + 8 * (int64_t)min(idx, nv - 1));  // clamped: in the row
  }
  float mx = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    if (tid + kPackThreads * j < nv) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t pr = (uint32_t)v[j][e];
        mx = fmaxf(mx, fmaxf(fabsf(to_f32(XT{(uint16_t)pr})), fabsf(to_f32(XT{(uint16_t)(pr >> 16)}))));
      }
    }
  }
  mx = group_max<64>(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPackThreads / 64; ++w) mx = fmaxf(mx, red[w]);
  const float s = scalar_div(fmaxf(mx, round_through<XT>(1e-6f)), 448.0f, div_mode);
  const float rs = 1.0f / s;
  uint8_t* qrow = qx + r * k;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int idx = tid + kPackThreads * j;
    if (idx < nv) {
      uint32_t w[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t p0 = (uint32_t)v[j][2 * h], p1 = (uint32_t)v[j][2 * h + 1];
        const uint32_t c01 = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(
            div_by(to_f32(XT{(uint16_t)p0}), s, rs), div_by(to_f32(XT{(uint16_t)(p0 >> 16)}), s, rs), 0, false);
        const uint32_t c23 = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(
            div_by(to_f32(XT{(uint16_t)p1}), s, rs), div_by(to_f32(XT{(uint16_t)(p1 >> 16)}), s, rs), 0, false);
        w[h] = (c01 & 0xffffu) | (c23 << 16);
      }
      *(uint2*)(qrow + 8 * (int64_t)idx) = make_uint2(w[0], w[1]);
    }
  }
  if (tid == 0) sx[r] = s;
}

// ---- int8 activations: Int8Method.apply, qtts/quant/int8.py:147-149 ----------------
// Everything happens in the activation dtype XT: the absmax, the 1e-6 clamp, the
// division by 127 (div_mode) and the quotient x / scale, each rounded to XT as torch
// rounds an XT tensor op; .round() is half-to-even on that XT value.  The scale is
// stored widened to fp32 (exact).  A NaN quotient (0 / 0, which the fp16 scale of a
// row with absmax below ~3.8e-6 produces, since that scale rounds to zero) stores
// code 0, what the reference's float -> int8 cast gives it.

template <typename XT>
__global__ __launch_bounds__(kPackThreads) void quant_act_int8_kernel(
    const XT* __restrict__ x, int64_t k, int64_t ld, int8_t* __restrict__ qx, float* __restrict__ sx,
    int div_mode) {
  __shared__ float red[4];
  const int64_t r = blockIdx.x;
  const XT* row = x + r * ld;
  const float s = int8_act_scale<XT>(row_absmax(row, k, red), div_mode);
  int8_t* qrow = qx + r * k;
  for (int64_t c = threadIdx.x; c < k; c += kPackThreads) qrow[c] = (int8_t)int8_act_code<XT>(to_f32(row[c]), s);
  if (threadIdx.x == 0) sx[r] = s;
}

// Vectorized form for 16-bit activations with 16-byte aligned rows and k % 8 == 0:
// each thread holds up to V 8-element vectors of the row in registers across both
// passes, so the row is read once.
template <typename XT, int V>
__global__ __launch_bounds__(kPackThreads) void quant_act_int8_vec_kernel(
    const XT* __restrict__ x, int64_t k, int64_t ld, int8_t* __restrict__ qx, float* __restrict__ sx,
    int div_mode) {
  __shared__ float red[kPackThreads / 64];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int nv = (int)(k >> 3);
  const XT* row = x + r * ld;
  i32x4_t v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int idx = tid + kPackThreads * j;
    v[j] = *(const i32x4_t*)(row + 8 * (int64_t)min(idx, nv - 1));  // clamped: in the row
  }
  float mx = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    if (tid + kPackThreads * j < nv) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t pr = (uint32_t)v[j][e];
        mx = fmaxf(mx, fmaxf(fabsf(to_f32(XT{(uint16_t)pr})), fabsf(to_f32(XT{(uint16_t)(pr >> 16)}))));
      }
    }
  }
  mx = group_max<64>(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPackThreads / 64; ++w) mx = fmaxf(mx, red[w]);
  const float s = int8_act_scale<XT>(mx, div_mode);
  int8_t* qrow = qx + r * k;
  auto store = [&](auto code) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int idx = tid + kPackThreads * j;
      if (idx < nv) {
        uint32_t w[2] = {0u, 0u};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t pr = (uint32_t)v[j][e];
          const uint32_t c0 = (uint32_t)code(to_f32(XT{(uint16_t)pr})) & 0xffu;
          const uint32_t c1 = (uint32_t)code(to_f32(XT{(uint16_t)(pr >> 16)})) & 0xffu;
          w[e >> 1] |= (c0 | (c1 << 8)) << (16 * (e & 1));
        }
        *(uint2*)(qrow + 8 * (int64_t)idx) = make_uint2(w[0], w[1]);
      }
    }
  };
  // The quotient from the row's reciprocal, correctly rounded (div_by): an IEEE division an element was half of
  // this kernel's time at 1500 rows (four int8 linears of a talker layer 167.9 -> 164.6 us).  A zero scale
  // (fp16) or an infinite one divides plainly.
  if (s > 0.0f && s <= 3.402823466e38f) {
    const float rs = 1.0f / s;
    store([&](float x) { return int8_code_of(round_through<XT>(div_by(x, s, rs))); });
  } else {
    store([&](float x) { return int8_act_code<XT>(x, s); });
  }
  if (tid == 0) sx[r] = s;
}

}  // namespace qtts

using namespace qtts;

namespace {

// The vector packer where it takes the call: false otherwise.
template <bool FP8, typename SrcT, typename StoreT>
bool pack_vec(const void* src, int64_t n, int64_t k, int64_t ld, void* q, void* scale_out, float* scale_f32, int div_mode,
              hipStream_t st) {
  const int64_t nv = k / 8, blocks = (n + kPackThreads / 64 - 1) / (kPackThreads / 64);
  if (k <= 0 || k % 8 != 0 || nv > 16 * 64 || n > (1 << 24) || (uintptr_t)src % 16 != 0 || ld % 8 != 0 ||
      (uintptr_t)q % 8 != 0)
    return false;
#define QTTS_PACK_VEC(V)                                                                                           \
  qtts::launch(&pack_vec_kernel<SrcT, V, FP8, StoreT>, dim3((unsigned)blocks), dim3(kPackThreads), 0, st,          \
               (const SrcT*)src, n, (int)k, ld, (uint8_t*)q, (StoreT*)scale_out, scale_f32, div_mode)
  if (nv <= 2 * 64) QTTS_PACK_VEC(2);
  else if (nv <= 4 * 64) QTTS_PACK_VEC(4);
  else if (nv <= 6 * 64) QTTS_PACK_VEC(6);
  else if (nv <= 12 * 64) QTTS_PACK_VEC(12);
  else QTTS_PACK_VEC(16);
#undef QTTS_PACK_VEC
  return true;
}

}  // namespace

int qtts_launch_pack_int8(const void* src, int src_dtype, int64_t n, int64_t k, int64_t ld, int8_t* q,
                          void* scale_out, int scale_dtype, float* scale_f32, int div_mode, hipStream_t st) {
  dim3 grid((unsigned)n), block(kPackThreads);
  bool done = false;
#define QTTS_PACK_I8V(ST)                                                                                           \
  (scale_dtype == QTTS_F32    ? pack_vec<false, ST, float>(src, n, k, ld, q, scale_out, scale_f32, div_mode, st)  \
   : scale_dtype == QTTS_BF16 ? pack_vec<false, ST, bf16_t>(src, n, k, ld, q, scale_out, scale_f32, div_mode, st) \
                              : pack_vec<false, ST, f16_t>(src, n, k, ld, q, scale_out, scale_f32, div_mode, st))
  if (src_dtype == QTTS_BF16) done = QTTS_PACK_I8V(bf16_t);
  else if (src_dtype == QTTS_F16) done = QTTS_PACK_I8V(f16_t);
#undef QTTS_PACK_I8V
  if (done) return qtts_check_launch("pack_int8_rowwise");
#define QTTS_PACK_I8(ST, DT)                                                                         \
  do {                                                                                               \
    if (scale_dtype == QTTS_F32)                                                                     \
      qtts::launch(&pack_int8_kernel<ST, float>, dim3(grid), dim3(block), 0, st, (const ST*)src, k, ld, q, (float*)scale_out, \
                                                          scale_f32, div_mode);                      \
    else if (scale_dtype == QTTS_BF16)                                                               \
      qtts::launch(&pack_int8_kernel<ST, bf16_t>, dim3(grid), dim3(block), 0, st, (const ST*)src, k, ld, q, (bf16_t*)scale_out, \
                                                           scale_f32, div_mode);                     \
    else                                                                                             \
      qtts::launch(&pack_int8_kernel<ST, f16_t>, dim3(grid), dim3(block), 0, st, (const ST*)src, k, ld, q, (f16_t*)scale_out, \
                                                          scale_f32, div_mode);                      \
  } while (0)
  if (src_dtype == QTTS_F32) QTTS_PACK_I8(float, 0);
  else if (src_dtype == QTTS_BF16) QTTS_PACK_I8(bf16_t, 1);
  else QTTS_PACK_I8(f16_t, 2);
#undef QTTS_PACK_I8
  return qtts_check_launch("pack_int8_rowwise");
}

int qtts_launch_pack_fp8(const void* src, int src_dtype, int64_t n, int64_t k, int64_t ld, uint8_t* q,
                         float* scale, int div_mode, hipStream_t st) {
  if ((src_dtype == QTTS_BF16 && pack_vec<true, bf16_t, float>(src, n, k, ld, q, scale, nullptr, div_mode, st)) ||
      (src_dtype == QTTS_F16 && pack_vec<true, f16_t, float>(src, n, k, ld, q, scale, nullptr, div_mode, st)))
    return qtts_check_launch("pack_fp8_e4m3_rowwise");
  dim3 grid((unsigned)n), block(kPackThreads);
  if (src_dtype == QTTS_F32) qtts::launch(&pack_fp8_kernel<float>, dim3(grid), dim3(block), 0, st, (const float*)src, k, ld, q, scale, div_mode);
  else if (src_dtype == QTTS_BF16) qtts::launch(&pack_fp8_kernel<bf16_t>, dim3(grid), dim3(block), 0, st, (const bf16_t*)src, k, ld, q, scale, div_mode);
  else qtts::launch(&pack_fp8_kernel<f16_t>, dim3(grid), dim3(block), 0, st, (const f16_t*)src, k, ld, q, scale, div_mode);
  return qtts_check_launch("pack_fp8_e4m3_rowwise");
}

int qtts_launch_quant_act_fp8(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ld, uint8_t* qx,
                              float* sx, int div_mode, hipStream_t st) {
  dim3 grid((unsigned)m), block(kPackThreads);
  const int64_t nv = k / 8;
  if (x_dtype != QTTS_F32 && k % 8 == 0 && k > 0 && (uintptr_t)x % 16 == 0 && ld % 8 == 0 && (uintptr_t)qx % 8 == 0 &&
      nv <= 4 * kPackThreads) {
#define QTTS_QA_VEC(XT)                                                                                          \
  do {                                                                                                           \
    if (nv <= kPackThreads)                                                                                      \
      qtts::launch(&quant_act_fp8_vec_kernel<XT, 1>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
    else if (nv <= 2 * kPackThreads)                                                                             \
      qtts::launch(&quant_act_fp8_vec_kernel<XT, 2>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
    else                                                                                                         \
      qtts::launch(&quant_act_fp8_vec_kernel<XT, 4>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
  } while (0)
    if (x_dtype == QTTS_BF16) QTTS_QA_VEC(bf16_t);
    else QTTS_QA_VEC(f16_t);
#undef QTTS_QA_VEC
    return qtts_check_launch("quant_act_fp8_rows");
  }
  if (x_dtype == QTTS_F32) qtts::launch(&quant_act_fp8_kernel<float>, dim3(grid), dim3(block), 0, st, (const float*)x, k, ld, qx, sx, div_mode);
  else if (x_dtype == QTTS_BF16) qtts::launch(&quant_act_fp8_kernel<bf16_t>, dim3(grid), dim3(block), 0, st, (const bf16_t*)x, k, ld, qx, sx, div_mode);
  else qtts::launch(&quant_act_fp8_kernel<f16_t>, dim3(grid), dim3(block), 0, st, (const f16_t*)x, k, ld, qx, sx, div_mode);
  return qtts_check_launch("quant_act_fp8_rows");
}

int qtts_launch_quant_act_int8(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ld, int8_t* qx,
                               float* sx, int div_mode, hipStream_t st) {
  dim3 grid((unsigned)m), block(kPackThreads);
  const int64_t nv = k / 8;
  if (x_dtype != QTTS_F32 && k % 8 == 0 && k > 0 && (uintptr_t)x % 16 == 0 && ld % 8 == 0 && (uintptr_t)qx % 8 == 0 &&
      nv <= 4 * kPackThreads) {
#define QTTS_QA8_VEC(XT)                                                                                          \
  do {                                                                                                            \
    if (nv <= kPackThreads)                                                                                       \
      qtts::launch(&quant_act_int8_vec_kernel<XT, 1>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
    else if (nv <= 2 * kPackThreads)                                                                              \
      qtts::launch(&quant_act_int8_vec_kernel<XT, 2>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
    else                                                                                                          \
      qtts::launch(&quant_act_int8_vec_kernel<XT, 4>, grid, block, 0, st, (const XT*)x, k, ld, qx, sx, div_mode); \
  } while (0)
    if (x_dtype == QTTS_BF16) QTTS_QA8_VEC(bf16_t);
    else QTTS_QA8_VEC(f16_t);
#undef QTTS_QA8_VEC
    return qtts_check_launch("quant_act_int8_rows");
  }
  if (x_dtype == QTTS_F32)
    qtts::launch(&quant_act_int8_kernel<float>, grid, block, 0, st, (const float*)x, k, ld, qx, sx, div_mode);
  else if (x_dtype == QTTS_BF16)
    qtts::launch(&quant_act_int8_kernel<bf16_t>, grid, block, 0, st, (const bf16_t*)x, k, ld, qx, sx, div_mode);
  else
    qtts::launch(&quant_act_int8_kernel<f16_t>, grid, block, 0, st, (const f16_t*)x, k, ld, qx, sx, div_mode);
  return qtts_check_launch("quant_act_int8_rows");
}
