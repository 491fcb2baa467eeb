// Building blocks of the LDS-pipelined GEMM kernels (tile.hip, tile_fp8.hip): direct
// global -> LDS loads, vmcnt waits by stage, and a fence-free workgroup barrier.
#pragma once

#include "common.h"

namespace qtts {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void gbl_void_t;

// One 16-byte-per-lane direct load: lane l's 16 bytes land at lds_wave + 16 l.
__device__ __forceinline__ void load_to_lds16(const void* src, void* lds_wave) {
  __builtin_amdgcn_global_load_lds((gbl_void_t*)src, (lds_void_t*)lds_wave, 16, 0, 0);
}

// s_waitcnt vmcnt(N), expcnt and lgkmcnt left at their maxima.
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// s_waitcnt lgkmcnt(0), vmcnt and expcnt left at their maxima: this wave's LDS
// accesses are complete (before a barrier that publishes them to other waves).
__device__ __forceinline__ void wait_lgkmcnt0() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Workgroup barrier without a memory fence: stage visibility is established by each
// wave's own vmcnt wait before it; the signal fences keep the compiler from moving
// LDS accesses across it.
__device__ __forceinline__ void barrier_only() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// vmcnt(A * FPW) for the largest A <= min(ahead, AMAX): wait until at most `ahead`
// stages of this wave's loads are still in flight.
template <int FPW, int AMAX> __device__ __forceinline__ void wait_stages(int ahead) {
  if constexpr (AMAX > 0) {
    if (ahead >= AMAX) {
      wait_vmcnt<AMAX * FPW>();
      return;
    }
    wait_stages<FPW, AMAX - 1>(ahead);
  } else {
    wait_vmcnt<0>();
  }
}

// Activation rows of a stage in LDS: 128 bytes a row (64 16-bit or 128 8-bit columns), eight 16-byte
// pieces, piece p of row r at position swizzle8(r, p).  A direct load of 1 KiB then covers eight whole
// 128-byte rows (the lane at position p of row r fetches piece swizzle8(r, p): an involution), where MFMA
// lane order took half of each of 16 lines.  The table keeps the operand reads free of bank conflicts:
// ds_read_b128 serves lanes 0-3, 12-15, 20-23, 24-27 together, then 4-11 with 16-19 and 28-31 (and the
// upper half wave alike), so rows 0-3 and 12-15 of one piece meet rows 4-11 of the next (piece + 2, or
// + 1 for int8): the two groups of row pairs take the two halves of the eight positions.  By counter: no
// conflicts, one cycle for every 256 bytes read; with (row >> 1) in place of the table half the reads'
// cycles were conflicts and fp16 fp8-weight-only prefill lost 2.5%.  Measured against lane order: the
// four linears of a talker layer at 640 rows (fp8 weight-only, fp16) 105.1 -> 94.8 us, at 1500 rows
// (int8 W8A8) 172.6 -> 168.0, at 2048 (fp8 W8A8) 182.1 -> 174.7.
__device__ __forceinline__ int swizzle8(int row, int piece) {
  return piece ^ (int)((0x32765410u >> (4 * ((row >> 1) & 7))) & 7);
}

constexpr int kLdsBytes = 160 * 1024;  // LDS per workgroup on gfx950

}  // namespace qtts
