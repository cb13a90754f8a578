"""Sizes that the renderer's allocations and launches share with the render
service's reservations (csrc/render_sizes.h)."""
import ctypes
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def sizes(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("sizes") / "render_sizes_check.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-o", out,
                    os.path.join(HERE, "native", "render_sizes_check.cpp")], check=True)
    L = ctypes.CDLL(out)
    L.guide_train_blocks.restype = ctypes.c_uint32
    L.guide_train_blocks.argtypes = [ctypes.c_uint32]
    return L


def test_training_sums_depend_on_the_rows_alone(sizes):
    """A training step's blocks are the order of its gradient's sums: one per
    64 rows, at most 512, and nothing of the device in the launch."""
    for rows, blocks in ((1, 1), (64, 1), (65, 2), (32_767, 512), (32_768, 512), (32_769, 512), (1 << 18, 512),
                         (512 * 64 - 64, 511), (0xffffffff, 512)):
        assert sizes.guide_train_blocks(rows) == blocks
    src = open(os.path.join(HERE, "..", "drawlab_amd", "csrc", "hip", "guide.hip")).read()
    train = re.search(r"\ndl_status guide_train\(.*?\n}\n", src, re.S).group(0)
    assert "k_train<<<blocks," in train and "num_cus" not in train
