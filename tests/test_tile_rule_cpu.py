"""The rule for the width of the BF16x3 half-transform's column tiles
(csrc/f2jk_tiles.h), compiled for the host: a width that the kernel has, within
the cap, and never more column tiles (each a pass over B) than the even widths
2 to 10 with the fewest columns would give."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include <cstdio>
#include <initializer_list>
#include "f2jk_tiles.h"
int main() {
    for (int rows : {128, 256})
        for (int cap : {2, 4, 5, 6, 8, 10})
            for (int need = 1; need <= 300; ++need)
                std::printf("%d %d %d %d\n", rows, cap, need, f2jk::bf16_tile_units(need, cap, rows));
}
"""


def _fewest_columns(need, cap, widths):
    best = None
    for w in widths:
        if w <= cap and (best is None or -(-need // w) * w < best[0]):
            best = (-(-need // w) * w, w)
    return best[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_no_width_adds_a_pass_over_b(tmp_path):
    src, exe = tmp_path / "rule.cc", str(tmp_path / "rule")
    src.write_text(MAIN)
    build = subprocess.run(["g++", "-std=c++17", f"-I{ROOT}/forte2_amd/csrc", str(src), "-o", exe],
                           capture_output=True, text=True, timeout=120)
    assert build.returncode == 0, build.stderr
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120).stdout
    seen = 0
    for rows, cap, need, w in (map(int, line.split()) for line in out.splitlines()):
        seen += 1
        assert 1 <= w <= cap
        if rows == 128:
            assert w == _fewest_columns(need, cap, (10, 8, 6, 5, 4, 2))
        else:
            assert w in (1, 2, 3, 4, 5, 6, 7, 8, 10)
            for widths in ((10, 8, 6, 4, 2), (10, 8, 6, 5, 4, 2)):
                assert -(-need // w) <= -(-need // _fewest_columns(need, cap, widths)), (cap, need, w)
    assert seen == 2 * 6 * 300
