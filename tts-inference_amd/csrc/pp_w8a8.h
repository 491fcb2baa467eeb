// W8A8 GEMM (fp8 and int8, strip weights) for prefill rows on larger tiles than pipe_w8a8.h's, chosen
// where they fill whole rounds of compute units better: the same operands, LDS stages of 128
// columns and MFMAs in the same order per output, on another schedule.
//
// In pipe_w8a8.h all waves wait at one barrier a stage, read their operands and multiply, so the
// LDS reads and the matrix cores take turns.  Here the eight waves (a WM x 8 / WM grid over the tile)
// form two groups of four, one wave of each on every SIMD, half a stage apart: while one group reads
// its stage's operands into registers and issues the loads of a later one, the other multiplies, and a
// workgroup barrier hands over twice a stage.  Group 1 starts with one barrier more, group 0 ends with one more.
//   * Stage i is read by group 0 in phase 2 i and by group 1 in phase 2 i + 1; every wave waits for its
//     own loads of stage i before the barrier that ends phase 2 i - 1 (group 0 after multiplying stage
//     i - 1, group 1 after reading it).
//   * The loads of stage i + P - 1 reuse the buffer of stage i - 1, which group 1 finished reading in phase
//     2 i - 1; they go out at the start of a group's read of stage i, in phase 2 i or later.
// Measured on the talker's linears (three weights in turn, us, pipe_w8a8.h's choice -> this one): int8
// gate_up at 512 / 1024 / 1500 / 2048 rows 22.9 / 41.3 / 58.2 / 61.0 -> 19.0 / 29.5 / 48.8 / 54.5, qkv at 1024 /
// 1500 15.1 / 22.4 -> 14.0 / 18.4, o_proj at 1500 / 2048 14.4 / 15.5 -> 13.5 / 14.4, down_proj 32.0 / 33.8 -> 28.0 /
// 29.4; fp8 gate_up at 1024 / 1500 42.0 / 59.6 -> 36.6 / 57.3, qkv at 1500 22.9 -> 21.3 (at 2048 rows all four fp8
// linears fill whole rounds of pipe_w8a8.h's tiles and stay there).  An ablation of
// gate_up at 1024 rows (int8, 31.3 us under it): 26.5 without the global loads, 29.9 without the LDS reads, 23.6
// without the MFMAs: no single one bounds it; about 10 us are the launch, the first stages and the
// 25 MB of output that a single round writes at its end.
#pragma once

#include "pipe_w8a8.h"

namespace qtts {

template <typename Kind, typename OT, int BM, int BN, int WM, int P>
__global__ __launch_bounds__(512) void w8a8_pp_kernel(
    const typename Kind::code_t* __restrict__ qx, const float* __restrict__ sx, int M, int K, int64_t ldqx,
    const typename Kind::code_t* __restrict__ qw, int N, const float* __restrict__ sw, const OT* __restrict__ bias,
    OT* __restrict__ y, int64_t ldy, int ntiles) {
  typedef typename Kind::acc_t acc_t;
  constexpr int WN = 8 / WM, MB = BM / 16 / WM, NB = BN / 16 / WN;
  constexpr int XF = BM / 8, F = XF + BN / 8, FPW = F / 8, SB = F * 1024;
  static_assert(F % 8 == 0 && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "the waves must share the tile evenly");
  static_assert(P >= 2 && P * SB + 4 * (BM + 2 * BN) <= kLdsBytes && (P - 2) * FPW < 64, "LDS ring, 6-bit vmcnt");
  static_assert(BM <= 512 && BN <= 512, "a thread carries one row's and one column's scale");
  __shared__ __align__(1024) uint8_t ring[P * SB];
  __shared__ uint32_t epi_sx[BM], epi_sw[BN], epi_bi[BN];
  const int nt = blockIdx.x % ntiles, mt = blockIdx.x / ntiles;
  const int m0 = mt * BM, n0 = nt * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 2;
  const int wm = wave / WN, wn = wave % WN;
  const int c16 = lane & 15, g = lane >> 4;
  const int nk = K >> 7, strips = (N + 15) >> 4;

  // Epilogue operands first, as raw bits, parked in LDS once they land.
  const int ec = min(n0 + tid, N - 1);
  const uint32_t my_sx = load_out_bits(sx + min(m0 + tid, M - 1)), my_sw = load_out_bits(sw + ec);
  const uint32_t my_bi = load_out_bits((bias ? bias : (const OT*)sw) + (bias ? ec : 0));

  const uint8_t* src[FPW];
  int stride[FPW];
#pragma unroll
  for (int j = 0; j < FPW; ++j) {
    const int f = wave * FPW + j;
    if (f < XF) {
      const int row = 8 * f + (lane >> 3);
      src[j] = (const uint8_t*)qx + (int64_t)min(m0 + row, M - 1) * ldqx + 16 * swizzle8(row, lane & 7);
      stride[j] = 128;
    } else {
      const int s = min(n0 / 16 + ((f - XF) >> 1), strips - 1);
      src[j] = (const uint8_t*)qw + (int64_t)s * nk * 2048 + ((f - XF) & 1) * 1024 + lane * 16;
      stride[j] = 2048;
    }
  }
  auto issue = [&](int i) __attribute__((always_inline)) {
    uint8_t* stage = ring + (i % P) * SB + wave * FPW * 1024;
#pragma unroll
    for (int j = 0; j < FPW; ++j) load_to_lds16(src[j] + (int64_t)i * stride[j], stage + j * 1024);
  };
  acc_t acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = acc_t{0, 0, 0, 0};
  i32x4_t x0[MB], x1[MB], w0[NB], w1[NB];
  const int xoff0 = c16 * 128 + 16 * swizzle8(c16, Kind::col(g, 0) >> 4);
  const int xoff1 = c16 * 128 + 16 * swizzle8(c16, Kind::col(g, 1) >> 4);
  auto read = [&](int i) __attribute__((always_inline)) {
    const uint8_t* stage = ring + (i % P) * SB;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const uint8_t* ws = stage + (XF + 2 * (wn * NB + nb)) * 1024 + lane * 16;
      w0[nb] = *(const i32x4_t*)ws;
      w1[nb] = *(const i32x4_t*)(ws + 1024);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      x0[mb] = *(const i32x4_t*)(stage + (wm * MB + mb) * 2048 + xoff0);
      x1[mb] = *(const i32x4_t*)(stage + (wm * MB + mb) * 2048 + xoff1);
    }
  };

#pragma unroll
  for (int p = 0; p < P - 1; ++p)
    if (p < nk) issue(p);
  if (tid < BM) epi_sx[tid] = my_sx;
  if (tid < BN) {
    epi_sw[tid] = my_sw;
    epi_bi[tid] = my_bi;
  }
  wait_stages<FPW, P - 2>(nk - 1);
  wait_lgkmcnt0();
  barrier_only();
  if (group) barrier_only();
  for (int i = 0; i < nk; ++i) {
    if (i + P - 1 < nk) issue(i + P - 1);
    read(i);
    if (group) wait_stages<FPW, P - 2>(nk - 2 - i);
    wait_lgkmcnt0();
    __builtin_amdgcn_sched_barrier(0);
    barrier_only();
    // The multiplying group goes first on its SIMD (the scheduling barriers keep the MFMAs inside).
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = Kind::mma(w0[nb], w1[nb], x0[mb], x1[mb], acc[nb][mb]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    if (!group) wait_stages<FPW, P - 2>(nk - 2 - i);
    barrier_only();
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!group) barrier_only();

  // D of each 16x16 MFMA: lane (c16, g) holds rows 4g..4g+3 (weight rows n) of column c16 (activation row m).
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int col = (wn * NB + nb) * 16 + 4 * g, nbase = n0 + col;
    float swv[4], biv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      swv[t] = __uint_as_float(epi_sw[col + t]);
      biv[t] = out_bits_to_f32<OT>(epi_bi[col + t]);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = (wm * MB + mb) * 16 + c16, m = m0 + row;
      if (m >= M) continue;
      const float sxv = __uint_as_float(epi_sx[row]);
      OT* yr = y + (int64_t)m * ldy;
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = Kind::template out<OT>(acc[nb][mb][t], sxv, swv[t], biv[t], bias != nullptr);
      if constexpr (std::is_same<OT, float>::value) {
        if (nbase + 3 < N && ((uintptr_t)(yr + nbase) & 15) == 0) {
          *(f32x4_t*)(yr + nbase) = f32x4_t{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (nbase + t < N) yr[nbase + t] = v[t];
        }
      } else {
        const uint32_t lo = pack2_f32<OT>(v[0], v[1]), hi = pack2_f32<OT>(v[2], v[3]);
        if (nbase + 3 < N && ((uintptr_t)(yr + nbase) & 7) == 0) {
          *(uint2*)(yr + nbase) = make_uint2(lo, hi);
        } else {
          const uint16_t o[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (nbase + t < N) yr[nbase + t] = OT{o[t]};
        }
      }
    }
  }
}

// The tile of this kernel for an automatic call, or bm = 0 for pipe_w8a8.h's choice: past 256 rows,
// whichever finishes first at one workgroup a compute unit: rounds of 256 times a tile's time.  The times
// are us at K = 2048 (they scale with K alike), from the sweep above; 64 x 128 is the one small tile where pipe_w8a8.h
// stays ahead, and its 128 x 256 stays where it fills its rounds.
struct PpTile { int bm, bn; float us; };

template <typename Kind> inline PpTile pp_tile(int64_t m, int64_t n, int64_t k) {
  PpTile none{0, 0, 0.0f};
  if (m <= 256) return none;
  const W8A8PipeCfg old = w8a8_cfg(m, n, k, 0, 0, 0);
  if (old.nw != 8 || old.S != 1) return none;
  auto rounds = [&](int bm, int bn) {
    return (float)((((m + bm - 1) / bm) * ((n + bn - 1) / bn) + 255) / 256);
  };
  constexpr bool i8 = std::is_same<Kind, PipeI8>::value;
  const float old_us = old.bn == 128 ? 8.8f : (old.bm == 64 ? 15.1f : 21.0f);
  static const PpTile tiles[] = {{128, 128, i8 ? 14.0f : 15.9f}, {192, 128, i8 ? 18.0f : 20.0f},
                                 {128, 192, i8 ? 18.0f : 20.3f}, {256, 192, i8 ? 28.5f : 36.0f}};
  PpTile best = none;
  float best_us = 0.97f * old_us * rounds(old.bm, old.bn);
  for (const PpTile& t : tiles) {
    const float us = t.us * rounds(t.bm, t.bn);
    if (us < best_us) {
      best = t;
      best_us = us;
    }
  }
  return best;
}

template <typename Kind, typename OT> bool launch_pp(const PpTile& t, const W8A8Args<Kind>& a, hipStream_t st) {
  const int64_t mt = (a.m + t.bm - 1) / t.bm, nt = (a.n + t.bn - 1) / t.bn;
  if (mt * nt >= (1 << 22)) return false;
#define QTTS_PP(BM, BN, WM, P)                                                                                       \
  if (t.bm == BM && t.bn == BN) {                                                                                    \
    qtts::launch(&w8a8_pp_kernel<Kind, OT, BM, BN, WM, P>, dim3((unsigned)(mt * nt)), dim3(512), 0, st, a.qx, a.sx,  \
                 (int)a.m, (int)a.k, a.ldqx, a.qw, (int)a.n, a.sw, (const OT*)a.bias, (OT*)a.y, a.ldy, (int)nt);      \
    return true;                                                                                                     \
  }
  QTTS_PP(128, 128, 4, 4)
  QTTS_PP(192, 128, 4, 3)
  QTTS_PP(128, 192, 2, 3)
  QTTS_PP(256, 192, 4, 2)
#undef QTTS_PP
  return false;
}

// An automatic call: true when it was launched here.
template <typename Kind> bool try_pp(const W8A8Args<Kind>& a, int out_dtype, hipStream_t st) {
  const PpTile t = pp_tile<Kind>(a.m, a.n, a.k);
  if (t.bm == 0) return false;
  if (out_dtype == QTTS_BF16) return launch_pp<Kind, bf16_t>(t, a, st);
  if (out_dtype == QTTS_F16) return launch_pp<Kind, f16_t>(t, a, st);
  return launch_pp<Kind, float>(t, a, st);
}

}  // namespace qtts
