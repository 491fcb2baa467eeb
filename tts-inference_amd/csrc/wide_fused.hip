// The wide W8A16 kernel (wide.h) with the RMSNorm inside, GatedMLP's activation, or both.
#include "wide.h"

using namespace qtts;

// x [m, k] 16-bit, 16-byte aligned rows; nw: the norm's weight (16-byte aligned) or NULL; pair: the activation
// of a fused gate_up weight (n % 32 == 0), y [m, n / 2].  Returns as qtts_launch_w8a16_wide.
int qtts_launch_w8a16_wide_fused(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const void* nw, float eps,
                                 const int8_t* qs, int64_t n, const void* scale, int sdt, const void* bias, bool pair,
                                 void* y, int64_t ldy, hipStream_t st) {
  const int tile = wide_cfg(m, n, k, pair ? (nw ? kWideNormPair : kWidePair) : kWideNorm);
  if (tile < 0 || ldx > INT32_MAX) return 1;
  const WideArgs a{x, m, k, ldx, qs, n, scale, sdt, bias, nw, eps, nullptr, 0, y, ldy, st};
  if (x_dtype == QTTS_BF16) {
    if (!pair) launch_wide<bf16_t, kEpiNone, true, false>(tile, a);
    else if (nw) launch_wide<bf16_t, kEpiPair, true, false>(tile, a);
    else launch_wide<bf16_t, kEpiPair, false, false>(tile, a);
  } else {
    if (!pair) launch_wide<f16_t, kEpiNone, true, false>(tile, a);
    else if (nw) launch_wide<f16_t, kEpiPair, true, false>(tile, a);
    else launch_wide<f16_t, kEpiPair, false, false>(tile, a);
  }
  return qtts_check_launch("w8a16_wide_fused");
}
