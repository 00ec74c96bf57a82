"""The traffic table of bench.py is tied to every source of the J/K library."""

import glob
import os

import bench


def test_every_jk_source_is_hashed():
    have = {os.path.relpath(p, bench.ROOT) for p in glob.glob(os.path.join(bench.ROOT, "forte2_amd", "csrc", "f2jk*"))}
    assert have == set(bench.KERNEL_SOURCES)
