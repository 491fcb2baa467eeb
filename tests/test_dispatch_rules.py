"""The dispatch rules that are plain host headers (csrc/*_rule.h), compiled alone and read here on the CPU."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tts-inference_amd", "csrc")


def _run(tmp_path, source: str) -> list[list[int]]:
    """The rows of whole numbers that a program on these headers prints."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return [[int(v) for v in line.split()] for line in out.splitlines()]


def test_rms_norm_rows_of_every_size_take_a_vector_kernel(tmp_path):
    """16-bit aligned rows: in registers where they fit, in vectors past that (never element by element); the others not."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include "norm_rule.h"
int main() {
  const long long ks[] = {8, 512, 520, 1024, 1032, 2048, 2056, 4096, 4104, 8192, 8200, 16384, 1 << 20};
  const long long ms[] = {1, 1003, 1 << 22, (1 << 22) + 1, 1 << 25};
  for (long long k : ks)
    for (long long m : ms)
      for (int vec = 0; vec < 2; ++vec) {
        const qtts::NormForm f = qtts::norm_form(vec, m, k);
        printf("%lld %lld %d %d %d\\n", m, k, vec, f.threads, f.vectors);
      }
}
""")
    assert len(rows) == 13 * 5 * 2
    for m, k, vec, threads, vectors in rows:
        if not vec:
            assert threads == 0, (m, k)
        elif k <= 8192 and m <= 1 << 22:
            assert threads * vectors * 8 >= k and threads * m < 1 << 32, (m, k)
            assert threads in (64, 128, 256) and (vectors == 1 or threads == 256), (m, k)
        else:
            assert (threads, vectors) == (64, 0), (m, k)


def test_wide_tiles_are_built_in_the_forms_that_the_rule_chooses(tmp_path):
    """The launcher builds each tile in the forms its line names, and the rule takes tiles from those lines alone: every line's
    forms are the ones that some call chooses it in, no more (a kernel nothing reaches) and no fewer."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include "wide_rule.h"
using namespace qtts;
int main() {
  int chosen[kWideTileCount] = {0};
  for (int k = 64; k <= 6400; k += 64)
    for (int n = 32; n <= 20000; n += 32)
      for (int m = 1; m <= 140; ++m)
        for (int form = 1; form <= 16; form *= 2) {
          const bool pair = form == kWidePair || form == kWideNormPair, plain = form == kWidePlain || form == kWideFp8;
          if (pair && n % 32) continue;
          if (plain && half_cfg(m, n, k).waves) continue;  // the half strips come first
          const int t = wide_cfg(m, n, k, form);
          if (t >= 0) chosen[t] |= form;
        }
  for (int i = 0; i < kWideTileCount; ++i) printf("%d %d\\n", kWideTiles[i].forms, chosen[i]);
}
""")
    assert rows and all(built == chosen for built, chosen in rows), rows


def test_decode_row_parts_keep_9_to_16_rows_of_few_strips(tmp_path):
    """65 to 128 strips at 9-16 rows, where two row parts of the decode kernel fill the GPU and the wide kernel does not: the
    K at which they measured faster stay there, and the lines lie at 16 rows and 64 / 128 strips."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include "wide_rule.h"
using namespace qtts;
int main() {
  const int ks[] = {1024, 2048, 3072, 6144}, ns[] = {1024, 1056, 2048, 2080}, ms[] = {9, 12, 16, 17};
  for (int k : ks)
    for (int n : ns)
      for (int m : ms)
        for (int form = 1; form <= 16; form *= 2) printf("%d %d %d %d %d\\n", k, n, m, form, wide_cfg(m, n, k, form));
}
""")
    taken = {tuple(r[:4]): r[4] >= 0 for r in rows}
    plain, norm, pair, norm_pair, fp8 = 1, 2, 4, 8, 16
    for n in (1056, 2048):
        for m in (9, 12, 16):
            for form in (plain, fp8):
                assert not taken[6144, n, m, form] and not taken[2048, n, m, form]
                assert taken[1024, n, m, form] and taken[3072, n, m, form] and taken[6144, n, 17, form]
            assert not taken[2048, n, m, norm] and not taken[2048, n, m, pair]
            assert taken[2048, n, m, norm_pair] and taken[6144, n, m, pair] and taken[2048, n, 17, norm]
    assert all(taken[k, 2080, m, plain] for k in (2048, 6144) for m in (9, 16))


def test_wide_rule_takes_every_k_that_a_built_run_holds(tmp_path):
    """No list of K: each multiple of 64 in the range takes tiles whose waves hold it in the shortest built runs, each multiple of
    128 the half strips; the ends of the range."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include "wide_rule.h"
using namespace qtts;
int main() {
  for (int k = 1; k <= 8192; ++k) {
    const int t = wide_cfg(27, 2048, k, kWidePlain);
    const HalfCfg h = half_cfg(8, 2048, k);
    printf("%d %d %d %d\\n", k, t < 0 ? 0 : kWideTiles[t].waves, t < 0 ? 0 : kWideTiles[t].cpw, h.waves * h.upw);
  }
}
""")
    for k, waves, cpw, units in rows:
        assert (waves > 0) == (k % 64 == 0 and 512 < k <= 6144), k
        if waves:
            assert waves <= k // 64 <= waves * cpw and (k // 64 > 3 * 16 or waves * cpw <= 48), k
        assert (units > 0) == (k % 128 == 0 and 512 < k <= 6144), k
        assert not units or k // 128 <= units, k


def test_half_strips_take_one_round_of_workgroups(tmp_path):
    """Two half strips times the 8-row parts, at most 256: the last row of each line of strips, and the first past it."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include "wide_rule.h"
using namespace qtts;
int main() {
  const int ns[] = {1, 16, 17, 64, 200, 512, 1000, 1024, 2048, 2049};
  for (int n : ns)
    for (int m = 1; m <= 1100; ++m) printf("%d %d %d\\n", n, m, half_cfg(m, n, 2048).waves);
}
""")
    last = {}
    for n, m, waves in rows:
        if waves:
            assert m >= 5, (n, m)
            last[n] = m
    assert last == {1: 1024, 16: 1024, 17: 512, 64: 256, 200: 72, 512: 32, 1000: 16, 1024: 16, 2048: 8}


def test_decode_kernel_keeps_few_strips_that_half_strips_cannot_split(tmp_path):
    """9-16 rows on up to 64 strips with K an odd multiple of 64 (no half strips): the decode kernel from where it measured faster,
    K > 3072, or K > 1280 with the norm inside; whole units of 128 and 17 rows go on as before."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include <initializer_list>
#include "wide_rule.h"
using namespace qtts;
int main() {
  const int ks[] = {1088, 1344, 1984, 2048, 3008, 3136, 3200, 4032, 6080}, ns[] = {224, 1024}, ms[] = {9, 16, 17};
  for (int k : ks)
    for (int n : ns)
      for (int m : ms)
        for (int form : {kWidePlain, kWideFp8, kWideNorm, kWidePair})
          printf("%d %d %d %d %d\\n", k, n, m, form, wide_cfg(m, n, k, form) >= 0 || (form != kWideNorm && form != kWidePair && half_cfg(m, n, k).waves));
}
""")
    plain, norm, pair, fp8 = 1, 2, 4, 16
    assert len(rows) == 9 * 2 * 3 * 4
    for k, n, m, form, taken in rows:
        odd = k % 128 != 0 and m <= 16
        if form in (plain, fp8):
            want = not (odd and k > 3072)
        elif form == norm:
            want = k <= 2048 and not (odd and k > 1280)
        else:
            want = not (3072 < k <= 4096 and m <= 16)
        assert taken == want, (k, n, m, form)


def test_wide_grids_fill_one_round_of_each_die(tmp_path):
    """Workgroups go to the eight dies in turn, 32 compute units each: no die gets a second round of a grid that the rule counts
    as one, with the columns padded to eights in each row block or not."""
    rows = _run(tmp_path, """
#include <stdio.h>
#include <initializer_list>
#include "wide_rule.h"
using namespace qtts;
int main() {
  int worst = 0, calls = 0, padded = 0;
  for (int k : {768, 1024, 1536, 2048, 3072, 6144})
    for (int n = 32; n <= 20000; n += 32)
      for (int m = 5; m <= 128; ++m)
        for (int form = 1; form <= 16; form *= 2) {
          const int t = wide_cfg(m, n, k, form);
          if (t < 0) continue;
          const int cols = ((n + 15) / 16 + kWideTiles[t].nb - 1) / kWideTiles[t].nb, blocks = (m + 16 * kWideTiles[t].mb - 1) / (16 * kWideTiles[t].mb);
          const int x = wide_grid_x(cols, blocks);
          int die[8] = {0};
          for (int b = 0; b < blocks; ++b)
            for (int c = 0; c < cols; ++c) ++die[(b * x + c) % 8];
          for (int d = 0; d < 8; ++d) worst = die[d] > worst ? die[d] : worst;
          ++calls;
          padded += x % 8 == 0;
          if (x < cols) worst = 1000;
        }
  printf("%d %d %d\\n", worst, calls, padded);
}
""")
    worst, calls, padded = rows[0]
    assert worst == 32 and calls > 10000 and padded > 0.9 * calls
