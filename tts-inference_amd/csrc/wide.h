// The W8A16 kernels for 5 to 128 rows of weights that fill the GPU once (decode batches, the code predictor's prefix walk, short
// prompts) on strip weights, and for more rows of very few strips; the rule, row by row, is wide_rule.h.
//
// These calls are bound by latency and by the bytes each compute unit pulls through L2, not by the
// matrix cores: a ring of LDS stages (tile_w8a16.h) spends a wait and a barrier on each of its 8-48
// stages.  Here a workgroup owns 16 MB rows x 16 NB columns and all of K; its W waves split K into
// runs of up to CPW chunks, and a wave issues every load of its run before it consumes any: the activation
// rows straight to its own LDS block in whole cache lines (16-byte pieces swizzled, as pipe.h's
// stages), the weights to registers.  A call is one memory round trip and one reduction
// through LDS.  (Activation operands loaded to registers in MFMA lane order, as the decode kernel's
// direct form does, touch each line twice at half width: 0.5-1.5 us a call slower at 32 rows.)
//
// Measured in graphs over distinct weights (5 of the predictor's, 12 of the talker's), us a call, the former automatic choice ->
// this kernel, at the row counts of 16 / 32 / 64 / 128 that come here: the talker's qkv 4.33 / 6.34 / 7.39 / 7.94 -> 3.82 / 4.28 /
// 5.44 / 6.74, o_proj from 32 rows 5.20 / 7.37 / 7.32 -> 3.65 / 4.41 / 5.06, gate_up at 16 / 32 9.52 / 10.17 -> 7.04 / 7.96, down_proj at
// 32 / 64 9.36 / 9.54 -> 6.37 / 7.54; the predictor's qkv and gate_up at 16 / 32 3.21 / 4.10 -> 2.73 / 3.29 and 4.44 / 6.08 -> 3.31 / 3.78, its
// o_proj from 32 rows 3.72 / 4.80 / 7.06 -> 3.10 / 3.34 / 4.11, down_proj 4.83 / 7.00 / 7.68 -> 3.59 / 3.83 / 4.83.  With the RMSNorm inside
// against the norm before the GEMM (or the decode kernel's): predictor qkv 5.58 / 6.64 / 7.96 / 8.36 -> 3.72 / 4.14 / 4.87 / 6.42, talker
// qkv to 64 rows 6.53 / 9.67 / 10.87 -> 5.83 / 6.30 / 7.62; gate_up with norm and activation to 64 rows 7.24 / 10.74 / 10.54 -> 4.46 /
// 4.92 / 6.35 (predictor), at 16 13.08 -> 9.42 (talker).  The floor of a call is the 1.6 us launch, one memory round trip and 2-13 MB
// at 5.1 TB/s.
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "layout.h"
#include "pipe.h"
#include "skinny.h"
#include "tile_w8a16.h"
#include "wide_rule.h"

namespace qtts {

// v + v of the lanes 16 and 32 away: the four lanes that share a row in the MFMA operand layout.
__device__ __forceinline__ float add_row_lanes(float v) {
  auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// EPI: tile_w8a16.h's epilogues.  NORM: the input is RMSNorm(x) with weight aux and epsilon eps,
// rounded as the reference rounds it (skinny.h: kProRmsNorm): each wave sums x^2 over its run, the
// waves meet at one fence-free barrier while the weights stay in flight, and each scales its operands.
// FIT: K = 64 W CPW, every run a constant (the norm with K = 2048 at 32 / 64 rows 6.5 / 7.7 us, 6.8 / 8.3 with the runs computed).
// CL: chunks of a run that go through LDS; the rest load to registers in lane order (LDS holds no more).
// NT: the weight policy, as in skinny.h (alone, streaming loads measure 0.1-0.8 us a call slower; in a 12-layer
// talker step they win, 32 rows 382.0 -> 379.0 us, 8 rows 289.2 -> 280.7 with the half strips below).
template <typename XT, int MB, int NB, int W, int CPW, int CL, int EPI, bool NORM, bool F8W, bool NT, bool FIT>
__global__ __launch_bounds__(W * 64) void w8a16_wide_kernel(
    const int8_t* __restrict__ qs, const XT* __restrict__ x, const void* scale, const XT* bias, const XT* aux, int ldx,
    int M, int N, int kdt, float eps, XT* y, int64_t ldy, const XT* res, int64_t ldr) {
  typedef mfma16<XT> MM;
  typedef typename MM::vec V;
  constexpr int XI = 2 * MB * CL, P = 8 * CL;  // direct loads a wave, 16-byte pieces a row of its block
  static_assert(CL <= CPW && (CL % 2 == 0 || CL == 1 || CL == 3), "pieces in groups of 16, or of 8");
  __shared__ __align__(1024) uint8_t lds[W][1024 * (2 * MB * CL > MB * NB ? 2 * MB * CL : MB * NB)];
  __shared__ uint32_t epi_sc[16 * NB], epi_bi[16 * NB];  // scale and bias bits, column by column
  __shared__ float nss[NORM ? W : 1][NORM ? 16 * MB : 1];
  const int strips = (N + 15) >> 4;
  const int s0 = blockIdx.x * NB, y0 = blockIdx.z * (16 * MB);
  if (s0 >= strips) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int chunks = FIT ? W * CPW : kdt >> 8, sdt = kdt & 0xff;  // K / 64, the scales' type
  // The wave's run of K: run chunks from wc0 (0 to CPW; the runs of a call differ by one at most).  A run shorter
  // than CPW loads its last chunk again in the slots past it, and leaves them out of the sums.
  const int wc0 = FIT ? wave * CPW : wave * (chunks / W) + min(wave, chunks % W);
  const int run = FIT ? CPW : chunks / W + (wave < chunks % W ? 1 : 0);
  const int last = min(max(run, 1), chunks - wc0) - 1;  // of the run, counted from wc0 (-1: a wave of no chunks)
  auto at = [&](int u) { return FIT ? u : min(u, last); };

  // Position of piece p of a row in the wave's block (an involution): conflict-free operand reads.
  auto swz = [](int row, int p) { return CL % 2 == 0 ? p ^ (row & 15) : ((p & ~7) | swizzle8(row, p & 7)); };
  const XT* xw = x + wc0 * 64;
  auto load_rows = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int flat = i * 64 + lane, row = flat / P, p = swz(row, flat % P);
      const int col = decltype(whole)::value ? 8 * p : at(p >> 3) * 64 + 8 * (p & 7);
      load_to_lds16(xw + (int64_t)min(y0 + row, M - 1) * ldx + col, &lds[wave][i * 1024]);
    }
  };
  if (FIT || run >= CL) load_rows(std::true_type{});
  else load_rows(std::false_type{});
  i32x4_t w[CPW][NB], xa[CPW][MB], xb[CPW][MB], nw[NORM ? CPW : 1][2];
#pragma unroll
  for (int u = CL; u < CPW; ++u)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const XT* p = x + (int64_t)min(y0 + 16 * mb + r, M - 1) * ldx + (wc0 + at(u)) * 64 + 16 * g;
      xa[u][mb] = *(const i32x4_t*)p;
      xb[u][mb] = *(const i32x4_t*)(p + 8);
    }
  if constexpr (NORM) {
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      nw[u][0] = *(const i32x4_t*)(aux + (wc0 + at(u)) * 64 + 16 * g);
      nw[u][1] = *(const i32x4_t*)(aux + (wc0 + at(u)) * 64 + 16 * g + 8);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int s = min(s0 + nb, strips - 1);
    const int8_t* wp;
    if constexpr (EPI == kEpiPair) {  // (N % 32 == 0: both halves sit in whole strips)
      const int R = 8 * s + (r & 7) + (r < 8 ? 0 : (N >> 1));
      wp = qs + ((int64_t)(R >> 4) * chunks + wc0) * 1024 + ((R & 15) + 16 * g) * 16;
    } else {
      wp = qs + ((int64_t)s * chunks + wc0) * 1024 + lane * 16;
    }
#pragma unroll
    for (int u = 0; u < CPW; ++u) w[u][nb] = load_weight<NT>(wp + at(u) * 1024);
  }
  __builtin_amdgcn_sched_barrier(0);

  // The epilogue is shared by the waves: unit u (wave u % W) is two of the four rows a lane holds of
  // block u / 2 (kEpiPair: a block's 16 x 8 outputs, two a lane).  Its operands are raw bits, fetched after
  // the weights and not needed before the end; thread t < 16 NB takes column t's scale and bias
  // (every thread loads: a branch here would end in a wait).
  constexpr int UNITS = EPI == kEpiPair ? NB * MB : 2 * NB * MB;
  constexpr int UPW = (UNITS + W - 1) / W;
  uint32_t my_sc, my_bi, rb[EPI == kEpiRes ? UPW : 1][2];
  {
    const int t = min((int)threadIdx.x, 16 * NB - 1), s = s0 + (t >> 4), i = t & 15;
    const int n = min(EPI == kEpiPair ? 8 * s + (i & 7) + (i < 8 ? 0 : (N >> 1)) : 16 * s + i, N - 1);
    my_sc = load_scale_bits(scale, sdt, n);
    my_bi = load_bits((bias ? bias : x) + (bias ? n : 0));
    if constexpr (EPI == kEpiRes) {
#pragma unroll
      for (int j = 0; j < UPW; ++j) {
        const int u = min(wave + j * W, UNITS - 1), q = u >> 1;
        const XT* row = res + (int64_t)min(y0 + 16 * (q % MB) + r, M - 1) * ldr;
#pragma unroll
        for (int e = 0; e < 2; ++e)
          rb[j][e] = load_bits(row + min(16 * (s0 + q / MB) + 4 * g + 2 * (u & 1) + e, N - 1));
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load in flight before the first wait

  wait_vmcnt<CPW * NB>();  // the rows have landed; at least the weights issued after them may be in flight
#pragma unroll
  for (int u = 0; u < CL; ++u)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = 16 * mb + r;
      xa[u][mb] = *(const i32x4_t*)&lds[wave][(row * P + swz(row, 8 * u + 2 * g)) * 16];
      xb[u][mb] = *(const i32x4_t*)&lds[wave][(row * P + swz(row, 8 * u + 2 * g + 1)) * 16];
    }
  if constexpr (NORM) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float ss = 0.0f;
#pragma unroll
      for (int u = 0; u < CPW; ++u) {
        if (!FIT && u >= run) break;
#pragma unroll
        for (int i = 0; i < 4; ++i) ss = sq2_acc<XT>((uint32_t)xb[u][mb][i], sq2_acc<XT>((uint32_t)xa[u][mb][i], ss));
      }
      ss = add_row_lanes(ss);
      if (g == 0) nss[wave][16 * mb + r] = ss;
    }
    wait_lgkmcnt0();
    barrier_only();
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float t = 0.0f;
#pragma unroll
      for (int v = 0; v < W; ++v) t += nss[v][16 * mb + r];
      const float inv = 1.0f / __builtin_sqrtf(t / (float)(64 * chunks) + eps);
#pragma unroll
      for (int u = 0; u < CPW; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          i32x4_t& v = h ? xb[u][mb] : xa[u][mb];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t p = (uint32_t)v[i], q = (uint32_t)nw[u][h][i];
            const float a = to_f32(XT{(uint16_t)p}), b = to_f32(XT{(uint16_t)(p >> 16)});
            v[i] = (int)pack2_f32<XT>((a * inv) * to_f32(XT{(uint16_t)q}), (b * inv) * to_f32(XT{(uint16_t)(q >> 16)}));
          }
        }
    }
  }

  f32x4_t acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    if (!FIT && u >= run) break;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const V wlo = wcvt<F8W, XT>((uint32_t)w[u][nb][0], (uint32_t)w[u][nb][1]);
      const V whi = wcvt<F8W, XT>((uint32_t)w[u][nb][2], (uint32_t)w[u][nb][3]);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = MM::mma(wlo, __builtin_bit_cast(V, xa[u][mb]), acc[nb][mb]);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = MM::mma(whi, __builtin_bit_cast(V, xb[u][mb]), acc[nb][mb]);
    }
  }

  // Each wave's sums over its own rows block (its reads of it are done: the MFMAs above waited for them).
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) *(f32x4_t*)&lds[wave][((nb * MB + mb) * 64 + lane) * 16] = acc[nb][mb];
  if ((int)threadIdx.x < 16 * NB) {
    epi_sc[threadIdx.x] = my_sc;
    epi_bi[threadIdx.x] = my_bi;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < UPW; ++j) {  // sums in wave order
    const int u = wave + j * W;
    if (u >= UNITS) break;
    const int q = EPI == kEpiPair ? u : u >> 1;
    const int nb = q / MB, s = s0 + nb, m = y0 + 16 * (q % MB) + r;
    uint16_t o[2];
    int n;
    if constexpr (EPI == kEpiPair) {
      // lane (r, g): columns 2 g, 2 g + 1 of the strip's 8; the gate sums sit in lane (r, g / 2), the up sums 32 lanes on
      const int src = (q * 64 + r + 16 * (g >> 1)) * 16 + 8 * (g & 1);
      float a[2] = {0.0f, 0.0f}, b[2] = {0.0f, 0.0f};
#pragma unroll
      for (int v = 0; v < W; ++v)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          a[e] += ((const float*)&lds[v][src])[e];
          b[e] += ((const float*)&lds[v][src + 512])[e];
        }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int cg = 16 * nb + 2 * g + e, cu = cg + 8;
        float gv = a[e] * scale_bits_to_f32(epi_sc[cg], sdt), uv = b[e] * scale_bits_to_f32(epi_sc[cu], sdt);
        if (bias) {
          gv += xbits_to_f32<XT>(epi_bi[cg]);
          uv += xbits_to_f32<XT>(epi_bi[cu]);
        }
        o[e] = from_f32<XT>(silu_mul<XT>(round_through<XT>(gv), round_through<XT>(uv))).bits;
      }
      n = 8 * s + 2 * g;
    } else {
      const int src = (q * 64 + lane) * 16 + 8 * (u & 1);
      float a[2] = {0.0f, 0.0f};
#pragma unroll
      for (int v = 0; v < W; ++v)
#pragma unroll
        for (int e = 0; e < 2; ++e) a[e] += ((const float*)&lds[v][src])[e];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int c = 16 * nb + 4 * g + 2 * (u & 1) + e;
        float f = a[e] * scale_bits_to_f32(epi_sc[c], sdt);
        if (bias) f += xbits_to_f32<XT>(epi_bi[c]);
        if constexpr (EPI == kEpiRes) f = xbits_to_f32<XT>(rb[j][e]) + round_through<XT>(f);
        o[e] = from_f32<XT>(f).bits;
      }
      n = 16 * s + 4 * g + 2 * (u & 1);
    }
    const int cols = EPI == kEpiPair ? N >> 1 : N;
    if (m >= M) continue;
    XT* yr = y + (int64_t)m * ldy + n;
    if (n + 1 < cols && ((uintptr_t)yr & 3) == 0) {
      *(uint32_t*)yr = o[0] | ((uint32_t)o[1] << 16);
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if (n + e < cols) yr[e] = XT{o[e]};
    }
  }
}

// The same for up to 8 rows a workgroup on few strips: a workgroup takes half a strip (8 weight rows) of one
// 8-row part of the call, so 64 or 128 strips still spread over the GPU.  One MFMA covers two chunks ("a unit"), as
// skinny.h's half strips: A rows 0-7 and B columns 0-7 hold the even chunk, rows 8-15 and columns 8-15 the odd
// one, and the two diagonal blocks of D are added in the epilogue.  What it has over the half strips
// of skinny.h: the rows go straight to LDS (no registers, no LDS writes) and 8-12 waves share a row's loads.
// Measured as above, us a call, skinny.h's half strips (9-16 rows: the kernel above) -> this one, with the
// residual add, at 8 / 16 rows: the talker's o_proj 3.51 -> 3.23 at 8, its down_proj 6.11 -> 4.62; the predictor's
// o_proj 4.37 / 4.60 -> 3.92 / 4.07, its down_proj 5.07 / 5.02 -> 4.14 / 4.35; its 1-stream frame 1243 -> 1158.
template <typename XT, int W, int UPW, int EPI, bool F8W, bool NT, bool FIT>
__global__ __launch_bounds__(W * 64) void w8a16_wide_half_kernel(
    const int8_t* __restrict__ qs, const XT* __restrict__ x, const void* scale, const XT* bias, int ldx, int M, int N, int kdt,
    XT* y, int64_t ldy, const XT* res, int64_t ldr) {
  typedef mfma16<XT> MM;
  typedef typename MM::vec V;
  constexpr int P = 16 * UPW, XI = 2 * UPW;
  __shared__ __align__(1024) uint8_t lds[W][XI * 1024];
  const int strip = blockIdx.x >> 1, part = (blockIdx.x & 1) * 8, y0 = blockIdx.z * 8;
  if (strip * 16 + part >= N) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int units = FIT ? W * UPW : kdt >> 8, sdt = kdt & 0xff;  // K / 128, the scales' type
  // The wave's run of units, as the kernel above's of chunks
  const int u0 = FIT ? wave * UPW : wave * (units / W) + min(wave, units % W);
  const int run = FIT ? UPW : units / W + (wave < units % W ? 1 : 0);
  const int last = min(max(run, 1), units - u0) - 1;
  auto at = [&](int u) { return FIT ? u : min(u, last); };
  const XT* xw = x + u0 * 128;
  auto load_rows = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int flat = i * 64 + lane, row = flat / P, p = flat % P ^ row;
      const int col = decltype(whole)::value ? 8 * p : at(p >> 4) * 128 + 8 * (p & 15);
      load_to_lds16(xw + (int64_t)min(y0 + row, M - 1) * ldx + col, &lds[wave][i * 1024]);
    }
  };
  if (FIT || run == UPW) load_rows(std::true_type{});
  else load_rows(std::false_type{});
  __builtin_amdgcn_sched_barrier(0);
  i32x4_t w[UPW];
  const int8_t* wp = qs + ((int64_t)strip * 2 * units + 2 * u0 + (r >> 3)) * 1024 + (part + (r & 7) + 16 * g) * 16;
#pragma unroll
  for (int u = 0; u < UPW; ++u) w[u] = load_weight<NT>(wp + at(u) * 2048);
  __builtin_amdgcn_sched_barrier(0);
  // output (row m, column n) of lane: n = lane % 8, m = lane / 8
  const int on = min(strip * 16 + part + (lane & 7), N - 1), om = min(y0 + (lane >> 3), M - 1);
  const uint32_t sc = load_scale_bits(scale, sdt, on);
  const uint32_t bi = load_bits((bias ? bias : x) + (bias ? on : 0));
  uint32_t rb = 0;
  if constexpr (EPI == kEpiRes) rb = load_bits(res + (int64_t)om * ldr + on);
  __builtin_amdgcn_sched_barrier(0);
  wait_vmcnt<UPW>();
  V xa[UPW], xb[UPW];
#pragma unroll
  for (int u = 0; u < UPW; ++u) {
    const int row = r & 7, p = 16 * u + 8 * (r >> 3) + 2 * g;
    xa[u] = *(const V*)&lds[wave][(row * P + (p ^ row)) * 16];
    xb[u] = *(const V*)&lds[wave][(row * P + ((p + 1) ^ row)) * 16];
  }
  f32x4_t acc = {0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < UPW; ++u) {
    if (!FIT && u >= run) break;
    acc = MM::mma(wcvt<F8W, XT>((uint32_t)w[u][0], (uint32_t)w[u][1]), xa[u], acc);
    acc = MM::mma(wcvt<F8W, XT>((uint32_t)w[u][2], (uint32_t)w[u][3]), xb[u], acc);
  }
  *(f32x4_t*)&lds[wave][lane * 16] = acc;
  __syncthreads();
  if (wave > 0) return;
  const int n = lane & 7, m = lane >> 3;
  const int src = (m + 16 * (n >> 2)) * 16 + 4 * (n & 3), src2 = ((m + 16 * (n >> 2)) ^ 40) * 16 + 4 * (n & 3);
  float a = 0.0f, b = 0.0f;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    a += *(const float*)&lds[v][src];
    b += *(const float*)&lds[v][src2];
  }
  float f = (a + b) * scale_bits_to_f32(sc, sdt);
  if (bias) f += xbits_to_f32<XT>(bi);
  if constexpr (EPI == kEpiRes) f = xbits_to_f32<XT>(rb) + round_through<XT>(f);
  if (y0 + m < M && strip * 16 + part + n < N) y[(int64_t)(y0 + m) * ldy + strip * 16 + part + n] = from_f32<XT>(f);
}

struct WideArgs {
  const void* x; int64_t m, k, ldx; const int8_t* qs; int64_t n; const void* scale; int sdt; const void* bias;
  const void* aux; float eps; const void* res; int64_t ldr; void* y; int64_t ldy; hipStream_t st;
};

// One launch of tile I of kWideTiles (wide_rule.h) in its form.
template <typename XT, int EPI, bool NORM, bool F8W, int FORM, int I> inline void launch_wide_tile(const WideArgs& a) {
  if constexpr ((kWideTiles[I].forms & FORM) != 0) {
    constexpr WideTile t = kWideTiles[I];
    const int64_t strips = (a.n + 15) / 16, blocks = (a.m + 16 * t.mb - 1) / (16 * t.mb);
    const dim3 grid((unsigned)wide_grid_x((strips + t.nb - 1) / t.nb, blocks), 1, (unsigned)blocks);
    auto run = [&](auto fit, auto nt) {
      qtts::launch(&w8a16_wide_kernel<XT, t.mb, t.nb, t.waves, t.cpw, t.cl, EPI, NORM, F8W, decltype(nt)::value, decltype(fit)::value>,
                   grid, dim3(t.waves * 64), 0, a.st, a.qs, (const XT*)a.x, a.scale, (const XT*)a.bias, (const XT*)a.aux,
                   (int)a.ldx, (int)a.m, (int)a.n, (int)(a.k / 64) << 8 | a.sdt, a.eps, (XT*)a.y, a.ldy,
                   (const XT*)a.res, a.ldr);
    };
    qtts::launch_by_policy<std::is_same<XT, bf16_t>::value>([&](auto nt) {
      if (a.k == 64 * t.waves * t.cpw) run(std::true_type{}, nt);
      else run(std::false_type{}, nt);
    });
  }
}

template <typename XT, int EPI, bool NORM, bool F8W, int... I>
inline void launch_wide(int tile, const WideArgs& a, std::integer_sequence<int, I...>) {
  constexpr int form = F8W ? kWideFp8 : (EPI == kEpiPair ? (NORM ? kWideNormPair : kWidePair) : (NORM ? kWideNorm : kWidePlain));
  (void)((I == tile && (launch_wide_tile<XT, EPI, NORM, F8W, form, I>(a), true)) || ...);
}

// tile: what wide_cfg gives for the form.
template <typename XT, int EPI, bool NORM, bool F8W> inline void launch_wide(int tile, const WideArgs& a) {
  launch_wide<XT, EPI, NORM, F8W>(tile, a, std::make_integer_sequence<int, kWideTileCount>{});
}

// One launch of a configuration of half_cfg (wide_rule.h).
template <typename XT, int EPI, bool F8W> inline bool launch_half(const HalfCfg& c, const WideArgs& a) {
  const dim3 grid((unsigned)((a.n + 15) / 16 * 2), 1, (unsigned)((a.m + 7) / 8));
#define QTTS_HALF(W, UPW)                                                                                       \
  if (c.waves == W && c.upw == UPW) {                                                                           \
    auto run = [&](auto fit, auto nt) {                                                                         \
      qtts::launch(&w8a16_wide_half_kernel<XT, W, UPW, EPI, F8W, decltype(nt)::value, decltype(fit)::value>, grid, \
                   dim3(W * 64), 0, a.st, a.qs, (const XT*)a.x, a.scale, (const XT*)a.bias, (int)a.ldx, (int)a.m, \
                   (int)a.n, (int)(a.k / 128) << 8 | a.sdt, (XT*)a.y, a.ldy, (const XT*)a.res, a.ldr);          \
    };                                                                                                          \
    qtts::launch_by_policy<std::is_same<XT, bf16_t>::value>([&](auto nt) {                                      \
      if (a.k == 128 * W * UPW) run(std::true_type{}, nt);                                                      \
      else run(std::false_type{}, nt);                                                                          \
    });                                                                                                         \
    return true;                                                                                                \
  }
  QTTS_HALF(8, 2)
  QTTS_HALF(8, 3)
  QTTS_HALF(12, 4)
#undef QTTS_HALF
  return false;
}

}  // namespace qtts
