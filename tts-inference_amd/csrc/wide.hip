// The wide W8A16 kernel (wide.h), plain and with the residual add.
#include "wide.h"

using namespace qtts;

// x [m, k] 16-bit, 16-byte aligned rows; strip weights; res [m, n] (row stride ldr) or NULL, may be y.
// Returns QTTS_OK, 1 when the call is not this kernel's (wide_rule.h), or an error status.
int qtts_launch_w8a16_wide(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const int8_t* qs, int64_t n,
                           const void* scale, int sdt, const void* bias, const void* res, int64_t ldr, void* y,
                           int64_t ldy, hipStream_t st) {
  const HalfCfg h = half_cfg(m, n, k);
  const int tile = wide_cfg(m, n, k, kWidePlain);
  if ((h.waves == 0 && tile < 0) || ldx > INT32_MAX) return 1;
  const WideArgs a{x, m, k, ldx, qs, n, scale, sdt, bias, nullptr, 0.0f, res, ldr, y, ldy, st};
  if (h.waves > 0) {
    bool ok;
    if (x_dtype == QTTS_BF16) ok = res ? launch_half<bf16_t, kEpiRes, false>(h, a) : launch_half<bf16_t, kEpiNone, false>(h, a);
    else ok = res ? launch_half<f16_t, kEpiRes, false>(h, a) : launch_half<f16_t, kEpiNone, false>(h, a);
    return ok ? qtts_check_launch("w8a16_wide_half") : 1;
  }
  if (x_dtype == QTTS_BF16) res ? launch_wide<bf16_t, kEpiRes, false, false>(tile, a) : launch_wide<bf16_t, kEpiNone, false, false>(tile, a);
  else res ? launch_wide<f16_t, kEpiRes, false, false>(tile, a) : launch_wide<f16_t, kEpiNone, false, false>(tile, a);
  return qtts_check_launch("w8a16_wide");
}
