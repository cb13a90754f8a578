"""What a build leaves with its context for the next one gives way to any other
allocation of the context that needs the room, but not while a build uses it."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("dmalloc") / "dmalloc_check.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", os.path.join(ROCM, "include"),
                    "-fPIC", "-shared", "-Wl,-Bsymbolic", "-o", out,
                    os.path.join(HERE, "native", "dmalloc_check.cpp")], check=True)
    L = ctypes.CDLL(out)
    L.dmalloc_check.argtypes = [ctypes.c_size_t, ctypes.c_int]
    return L.dmalloc_check


@pytest.mark.parametrize("nbytes,building,got,kept", [
    (200, 0, True, True),     # fits beside them
    (201, 0, True, False),    # fits without them
    (1000, 0, True, False),
    (1001, 0, False, False),  # larger than the device
    (201, 1, False, True),    # in use
    (200, 1, True, True),
])
def test_kept_build_memory_gives_way(check, nbytes, building, got, kept):
    assert check(nbytes, building) == (1 if got else 0) + (2 if kept else 0)
