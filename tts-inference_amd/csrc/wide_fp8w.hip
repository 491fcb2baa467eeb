// The wide kernels (wide.h) on e4m3 codes: the fp8 weight-only calls that wide_rule.h names.
#include "wide.h"

using namespace qtts;

// As qtts_launch_w8a16_wide, with fp32 scales and no residual.
int qtts_launch_fp8w_wide(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const uint8_t* qs, int64_t n,
                          const float* scale, const void* bias, void* y, int64_t ldy, hipStream_t st) {
  const HalfCfg h = half_cfg(m, n, k);
  const int tile = wide_cfg(m, n, k, kWideFp8);
  if ((h.waves == 0 && tile < 0) || ldx > INT32_MAX) return 1;
  const WideArgs a{x, m, k, ldx, (const int8_t*)qs, n, scale, QTTS_F32, bias, nullptr, 0.0f, nullptr, 0, y, ldy, st};
  if (h.waves > 0) {
    const bool done = x_dtype == QTTS_BF16 ? launch_half<bf16_t, kEpiNone, true>(h, a) : launch_half<f16_t, kEpiNone, true>(h, a);
    return done ? qtts_check_launch("fp8w_wide_half") : 1;
  }
  if (x_dtype == QTTS_BF16) launch_wide<bf16_t, kEpiNone, false, true>(tile, a);
  else launch_wide<f16_t, kEpiNone, false, true>(tile, a);
  return qtts_check_launch("fp8w_wide");
}
