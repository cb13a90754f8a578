"""Every ray of a traversal launch is traced once, whatever the grid: also by
grids of fewer blocks than there are work counters."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("split") / "work_split_check.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fPIC", "-shared", "-o", out,
                    os.path.join(HERE, "native", "work_split_check.cpp")], check=True)
    L = ctypes.CDLL(out)
    L.work_split_check.argtypes = [ctypes.c_uint32] * 4
    return L.work_split_check


@pytest.mark.parametrize("blocks", [1, 2, 3, 8, 31, 63, 64, 65, 100, 1024, 4096])
def test_every_slot_is_dealt_once(check, blocks):
    waves = 2 * blocks
    for n in [0, 1, 2, 63, 64, 65] + [k * waves + d for k in (1, 15, 16, 17, 64, 128, 256, 400) for d in (-1, 0, 1)]:
        if n > 2_000_000:
            continue
        for own in {waves, 1, max(1, waves // 3)}:  # both queries of a bounce share the grid
            assert check(n, blocks, 2, own) == 0, (n, blocks, own)
