// Which calls the wide kernels (wide.h) take, and in which tile.
#pragma once

#include <stdint.h>

namespace qtts {

// The forms of a call: kWidePlain with and without the residual, kWideFp8 the plain form on e4m3 codes.
enum : int { kWidePlain = 1, kWideNorm = 2, kWidePair = 4, kWideNormPair = 8, kWideFp8 = 16 };

// A workgroup of `waves` waves, up to cpw chunks (64 columns) of K each, cl of them through LDS; 16 mb rows, nb strips;
// forms: those that it is built for, the ones that wide_cfg chooses it in.
struct WideTile { int mb, nb, waves, cpw, cl, forms; };

constexpr WideTile kWideTiles[] = {
    {1, 1, 8, 2, 2, 31}, {1, 2, 8, 2, 2, 31}, {1, 3, 8, 2, 2, 31}, {1, 4, 8, 2, 2, 31}, {2, 2, 8, 2, 2, 14},
    {2, 3, 8, 2, 2, 31}, {2, 4, 8, 2, 2, 31}, {4, 3, 8, 2, 2, 4},
    {1, 1, 16, 2, 2, 31}, {1, 2, 16, 2, 2, 31}, {1, 3, 16, 2, 2, 31}, {1, 4, 16, 2, 2, 31}, {2, 2, 16, 2, 2, 21},
    {2, 3, 16, 2, 2, 21}, {2, 4, 16, 2, 2, 21},
    {1, 1, 8, 4, 4, 31}, {1, 2, 8, 4, 4, 31}, {2, 2, 8, 4, 4, 21},
    {1, 1, 8, 6, 6, 21}, {1, 2, 8, 6, 6, 21},
    {1, 1, 16, 6, 4, 21}, {1, 2, 16, 6, 4, 21}};
constexpr int kWideTileCount = (int)(sizeof(kWideTiles) / sizeof(kWideTiles[0]));

// The grid's x for `cols` columns of tiles in `blocks` row blocks.  Workgroups go to the eight dies (32 compute units and an L2
// each) in turn, so with x a multiple of 8 a column's row blocks meet on one die and read its weights through one L2; of 4 or 2,
// on two or four.  The largest of these that leaves every die at most 32 of the workgroups that have a tile, else x = cols:
// 85 columns x 3 blocks, 255 workgroups, would be 33 on five dies at x = 88 (39 rows of 5408 x 1536 with the norm: 12.8 us, 9.4 at
// x = 85).  41 columns x 6 blocks (90 rows of 1312 x 6144) 12.0 us at x = 41, 9.9 at 42; 33 x 7 (100 of 1056 x 6144) 11.6 at 33, 8.1 at 36.
inline int64_t wide_grid_x(int64_t cols, int64_t blocks) {
  for (int64_t step = 8; step > 1; step /= 2) {
    const int64_t x = (cols + step - 1) / step * step;
    int64_t extra[8] = {0}, most = 0;
    for (int64_t b = 0; b < blocks; ++b)
      for (int64_t c = 0; c < cols % 8; ++c) most = most > ++extra[(b * x + c) % 8] ? most : extra[(b * x + c) % 8];
    if (cols / 8 * blocks + most <= 32) return x;
  }
  return cols;
}

// Whether the decode kernel keeps a call of 9 to 16 rows on up to 128 strips, where this kernel has at most 128 workgroups.
// 65 to 128 strips: the two row parts (skinny.h) make 256 of 8 staged rows.  Measured at N = 1040 .. 2048, us a call, decode kernel -> wide:
// K = 6144 plain at 12 / 16 rows 5.64 / 5.60 -> 6.08 / 6.40, residual 6.17 / 6.19 -> 6.67 / 7.06 (K = 4096 and 5120 alike: 0.3 to 2.1
// slower); K = 2048 with the norm 4.81 -> 5.38, with the activation 3.56 -> 3.86, residual 3.63 -> 3.88, plain the same (K = 1536: norm 0.2
// slower, the rest within 0.2); K <= 1024 and 2560 .. 3072 0.2 to 0.6 faster, and the norm with the activation 0.6 to 1.7 everywhere.
// Up to 64 strips: K in whole units of 128 has the half strips below (with the norm the decode kernel takes two launches: 6.9 -> 5.3).  Odd
// chunks, N = 224 .. 1024, 9 / 16 rows: K = 3136 plain 4.7 -> 5.4 / 6.0, residual 4.9 -> 5.8 / 6.7, 6080 at 16 rows 5.8 -> 6.4, K <= 3008
// 0.1 to 0.5 faster; the norm at 1600 / 1984 5.0 -> 5.2 / 5.4, at 1088 5.0 -> 4.9.
// The activation alone at 3072 < K <= 4096: 1.1 to 1.9 slower on up to 64 strips too (longer K has no decode form: 0.8 to 1.4 faster).
inline bool decode_keeps(int64_t m, int64_t strips, int64_t k, int form) {
  if (m > 16 || strips > 128 || form == kWideNormPair) return false;
  if (form == kWidePair && k > 3072) return k <= 4096;
  if (strips > 64) return k > 3072 || (k > 1024 && k <= 2048);
  return k % 128 != 0 && form != kWidePair && k > (form == kWideNorm ? 1280 : 3072);
}

// The tile of kWideTiles for the automatic choice of an [m, k] x [n, k] call on strip weights, or -1: 9 to 128 rows (8 and
// fewer stay with the decode kernel, whose half strips and row staging are faster there; with the norm inside and K <= 1024 from 5
// rows: 8 rows of the predictor's qkv 5.50 -> 5.00 us, of its gate_up with the activation 6.59 -> 5.65) and 512 < K <= 6144
// (shorter K within 0.2 us of the kernels that have it, either way, on wide weights; longer K would not fit the built runs),
// where one of the built tiles covers the call in a single round of workgroups on the 256 compute units.
// The waves share the K / 64 chunks, so that every K takes the group of tiles with the shortest runs that hold it: 2 chunks a
// wave up to K = 1024, up to K = 2048 16 waves of 2 on more than 128 strips and 8 of 4 on fewer (32 rows: talker qkv 4.49 against
// 4.84 us, o_proj + residual 4.43 against 4.19), 8 waves of 6 up to 3072, 16 of 6 beyond.  Measured off the tiles' full runs,
// former automatic choice -> this, plain, N = 2048, 27 / 48 / 100 rows: K = 1088 5.80 / 6.14 / 6.30 -> 3.16 / 3.61 / 4.47, 1984 6.07 /
// 7.57 / 7.76 -> 3.63 / 4.18 / 5.08, 2560 7.80 / 7.57 -> 4.09 / 4.89, 5120 9.03 / 8.85 -> 6.12 / 7.16.
// Of the group's tiles the one that reads the fewest bytes a workgroup:
// a second round costs more than any tile's extra bytes (the talker's gate_up past 32 rows, 512 workgroups,
// 12.9 us at 48 rows against the tile kernel's 11.7).
// With the norm inside every workgroup repeats its rows' normalization, so the tile of the
// fewest rows is taken and at most 32768 elements (16 rows of 2048): past them the norm's own launch
// (about 2.7 us) is cheaper (talker gate_up at 32 rows 12.0 inside against 8.3 + 2.7; predictor gate_up
// at 128 10.7 against 7.5 + 2.9, and inside up to 64 rows, 7.48 against 8.6).
// K <= 1024 past 48 rows: plain and residual calls stay with the tile kernel and the decode kernel's half strips, because the
// automatic choice is held to the tile kernel's bits there (64 rows of 4096 x 1024; they would gain 0.1-3.8 us a call), and
// e4m3 codes with them, one line for both.
inline int wide_cfg(int64_t m, int64_t n, int64_t k, int form) {
  const bool norm = (form & (kWideNorm | kWideNormPair)) != 0;
  if ((form == kWidePlain || form == kWideFp8) && k <= 1024 && m > 48) return -1;
  if (m < (norm && k <= 1024 ? 5 : 9) || m > 128 || n <= 0 || n > (1 << 30) || k % 64 != 0 || k <= 512 || k > 6144) return -1;
  const int64_t strips = (n + 15) / 16, chunks = k / 64;
  if (decode_keeps(m, strips, k, form)) return -1;
  int waves, cpw;
  if (chunks <= 16) waves = 8, cpw = 2;
  else if (chunks <= 32) waves = strips > 128 ? 16 : 8, cpw = strips > 128 ? 2 : 4;
  else waves = chunks <= 48 ? 8 : 16, cpw = 6;
  int best = -1;
  int64_t best_cost = 0;
  for (int i = 0; i < kWideTileCount; ++i) {
    const WideTile& t = kWideTiles[i];
    if (t.waves != waves || t.cpw != cpw || !(t.forms & form)) continue;
    if (16 * t.mb >= m + 16) continue;  // a row block with no row of the call
    if ((strips + t.nb - 1) / t.nb * ((m + 16 * t.mb - 1) / (16 * t.mb)) > 256) continue;
    if (norm && (16 * t.mb * k > 32768 || k > 2048)) continue;
    const int64_t cost = norm ? 8 * t.mb + t.nb : 2 * t.mb + t.nb;  // bytes a workgroup over 16 K
    if (best < 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return best;
}

struct HalfCfg { int waves, upw; };  // waves == 0: not this kernel

// Half strips in 8-row parts (wide.h): from 5 rows, 512 < K <= 6144 and K % 128 == 0, where the strips times two times the parts make one
// round of at most 256 workgroups: 8 rows on 128 strips, 16 on 64, 32 on 32, and so on to 1024 rows on one.  Measured over that
// whole line, no call slower than with the former choice; us a call at K = 1024 / 2048 / 6144, plain: N = 2048, 8 rows 3.80 / 3.74 / 5.35 ->
// 3.03 / 3.49 / 4.62; N = 1024, 16 rows 3.79 / 3.49 / 5.00 -> 3.05 / 3.15 / 4.26; N = 512, 32 rows 3.79 / 3.47 / 4.93 -> 3.04 / 3.15 / 4.11; N = 200,
// 72 rows 5.94 / 6.53 / 8.68 -> 3.06 / 3.15 / 4.19; N = 64, 256 rows 5.84 / 6.41 / 12.10 -> 3.05 / 3.14 / 3.97; N = 16, 1024 rows 8.35 / 9.50 /
// 13.03 -> 3.01 / 3.10 / 3.97 (e4m3 codes alike, the residual 0.1 to 2 more saved).  The waves share the K / 128 units as the chunks above.  Below 5 rows
// skinny.h stages fewer rows, and whole steps run faster on it: 10 predictor layers at 2 / 4 rows 155.1 / 165.3 us
// against 160.7 / 167.9 with these (8 rows: 187.1 against 177.9), 4 talker layers 85.9 / 91.6 against 87.6 / 92.0
// (8 rows: 107.0 against 103.0).
inline HalfCfg half_cfg(int64_t m, int64_t n, int64_t k) {
  if (m < 5 || n < 1 || (n + 15) / 16 * 2 * ((m + 7) / 8) > 256 || k % 128 != 0 || k <= 512 || k > 6144) return HalfCfg{0, 0};
  if (k <= 2048) return HalfCfg{8, 2};
  return k <= 3072 ? HalfCfg{8, 3} : HalfCfg{12, 4};
}

// Whether the automatic choice runs a plain (or residual) call on the wide kernels.
inline bool wide_takes(int64_t m, int64_t n, int64_t k) {
  return half_cfg(m, n, k).waves > 0 || wide_cfg(m, n, k, kWidePlain) >= 0;
}

}  // namespace qtts
