// The W8A16 tile kernel (tile_w8a16.h) with an epilogue of the decoder layer: the residual add after
// o_proj and down_proj, or GatedMLP's activation after gate_up_proj (qtts/models/talker.py:270-271,
// qtts/layers/activation.py:142-147), for the automatic choice past the decode rows.  As separate
// kernels the add cost 4.9 us and the activation 5.0 (32 rows) to 7.8 us (1003 rows) a launch, reading
// back what the GEMM had just written; fused, a 12-layer talker step of 32 rows went from 514.4 to
// 469.7 us, the predictor's 8-stream frame from 2652 to 2326 and two prefill layers of 1003 rows from
// 311.1 to 288.0.  Built for the tiles the automatic choice takes.
#include "tile_w8a16.h"

using namespace qtts;

namespace {

template <typename XT, int BM, int BN, int P, bool PF, int NW, int CPS, int EPI>
void launch_epi(const PipeCfg& c, const PipeArgs& a, const void* res, int64_t ldr, unsigned blocks, hipStream_t st) {
  qtts::launch(&w8a16_pipe_kernel<XT, BM, BN, P, 1, false, PF, NW, CPS, EPI>, dim3(blocks), dim3(NW * 64), 0, st,
               (const XT*)a.x, (int)a.m, (int)a.k, a.ldx, a.qs, (int)a.n, a.scale, a.sdt, (const XT*)a.bias, (XT*)a.y,
               a.ldy, a.part, a.counters, c.mtiles, c.ntiles, c.S, c.cps, (const XT*)res, ldr);
}

// False when the tile is not built here.
template <typename XT, int EPI>
bool launch_cfg(const PipeCfg& c, const PipeArgs& a, const void* res, int64_t ldr, unsigned blocks, hipStream_t st) {
  if (c.wm != 1) return false;
  if (c.nw == 4 && c.bm == 32 && c.bn == 64 && c.P == 4 && c.pf) {
    if (c.cps2) launch_epi<XT, 32, 64, 4, true, 4, 2, EPI>(c, a, res, ldr, blocks, st);
    else launch_epi<XT, 32, 64, 4, true, 4, 1, EPI>(c, a, res, ldr, blocks, st);
    return true;
  }
  if (c.nw != 8) return false;
  if (c.bm == 64 && c.bn == 128 && c.P == 4 && c.pf) launch_epi<XT, 64, 128, 4, true, 8, 1, EPI>(c, a, res, ldr, blocks, st);
  else if (c.bm == 64 && c.bn == 256 && c.P == 4 && c.pf) launch_epi<XT, 64, 256, 4, true, 8, 1, EPI>(c, a, res, ldr, blocks, st);
  else if (c.bm == 128 && c.bn == 256 && c.P == 4 && c.pf) launch_epi<XT, 128, 256, 4, true, 8, 1, EPI>(c, a, res, ldr, blocks, st);
  else if (c.bm == 128 && c.bn == 384 && c.P == 3 && !c.pf) launch_epi<XT, 128, 384, 3, false, 8, 1, EPI>(c, a, res, ldr, blocks, st);
  else return false;
  return true;
}

}  // namespace

// One automatic tile launch with the residual (res != NULL) or the SiLU-pair epilogue (res == NULL:
// n % 32 == 0, y [m, n / 2]).  x [m, k] 16-bit, 16-byte aligned rows, k % 64 == 0, strip weights.
// Returns QTTS_OK, 1 when the tile is not built (the caller runs the separate kernels), or an error.
int qtts_launch_w8a16_pipe_epi(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const int8_t* qs,
                               int64_t n, const void* scale, int sdt, const void* bias, const void* res, int64_t ldr,
                               void* y, int64_t ldy, void* ws, int64_t ws_bytes, hipStream_t st) {
  PipeCfg c = pipe_cfg(m, n, k, 0, 0);
  const int64_t need = pipe_ws(c);
  if (need > ws_bytes || (need > 0 && !ws)) c = pipe_cfg(m, n, k, 1, 0);  // as the plain launch
  const int64_t blocks = ((int64_t)c.mtiles * c.ntiles + 7) / 8 * 8 * c.S;
  if (blocks <= 0 || blocks >= ((int64_t)1 << 31)) return 1;
  const PipeArgs a{x, m, k, ldx, qs, n, scale, sdt, bias, y, ldy,
                   ws ? (float*)((char*)ws + kCounterBytes) : nullptr, (unsigned*)ws};
  bool ok;
  if (x_dtype == QTTS_BF16)
    ok = res ? launch_cfg<bf16_t, kEpiRes>(c, a, res, ldr, (unsigned)blocks, st)
             : launch_cfg<bf16_t, kEpiPair>(c, a, res, ldr, (unsigned)blocks, st);
  else
    ok = res ? launch_cfg<f16_t, kEpiRes>(c, a, res, ldr, (unsigned)blocks, st)
             : launch_cfg<f16_t, kEpiPair>(c, a, res, ldr, (unsigned)blocks, st);
  return ok ? qtts_check_launch("w8a16_pipe_epilogue") : 1;
}
