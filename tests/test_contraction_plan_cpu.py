"""The P splits of the FP64 contraction's tiles (csrc/f2jk_tiles.h, compiled for
the host): no kind of tile is left with more than about twice the steps of
another, whatever the remainder of nbf, and the totals add up."""

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
    for (int slots : {1, 64, 256, 512})
        for (int width : {8, 24, 80, 240})
            for (int N = 1; N <= 1600; N += N < 300 ? 1 : 13)
                for (int Pc : {1, 7, 400, 2000}) {
                    const f2jk::DTiles m = f2jk::dtile_plan(N, Pc, width, slots);
                    std::printf("%d %d %d  %d %d %d %d  %d %d %d %d  %d %d %d\n", slots, N, Pc, m.cnt[0], m.cnt[1], m.cnt[2],
                                m.cnt[3], m.ns[0], m.ns[1], m.ns[2], m.ns[3], m.G, m.total, m.nt);
                }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_steps_of_the_tiles_are_balanced(tmp_path):
    src, exe = tmp_path / "plan.cc", str(tmp_path / "plan")
    src.write_text(MAIN)
    build = subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT}/forte2_amd/csrc", str(src), "-o", exe],
                           capture_output=True, text=True, timeout=120)
    assert build.returncode == 0, build.stderr
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120).stdout
    seen = 0
    for slots, N, Pc, *v in (tuple(map(int, line.split())) for line in out.splitlines()):
        cnt, ns, (G, total, nt) = v[:4], v[4:8], v[8:]
        present = [n for c, n in zip(cnt, ns) if c]
        assert nt == -(-N // 128) and sum(cnt) == nt * (nt + 1) // 2
        assert all(1 <= n <= Pc for n in present) and G == max(present)
        assert total == sum(c * n for c, n in zip(cnt, ns))
        if min(present) >= 8:
            # costs between 9 and 16, each rounded down to whole splits
            seen += 1
            assert max(present) <= 16 / 9 * (min(present) + 1), (slots, N, Pc, cnt, ns)
    assert seen > 1000
