"""The index arithmetic of the kernels' grid-stride walks (csrc/qmcx_walk.hpp) at ranges that end near INT_MAX,
compiled for the host."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "miniqmc_amd", "csrc")
INT_MAX = 2**31 - 1


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    src = d / "walk.cpp"
    src.write_text('#include "qmcx_walk.hpp"\n'
                   'extern "C" int next(int u, int step, int end) { return qmcx::walk_next(u, step, end); }\n'
                   'extern "C" int div_up(int a, int b) { return qmcx::ceil_div(a, b); }\n')
    so = d / "walk.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-I" + CSRC, str(src), "-o", str(so)])
    return C.CDLL(str(so))


@pytest.mark.parametrize("end", [1, 5, 1000, 262144, 262145, INT_MAX - 7, INT_MAX - 262144, INT_MAX])
@pytest.mark.parametrize("step", [1, 1024, 262144])
def test_walk(lib, end, step):
    for start in {0, 1, end // 2, max(end - step - 1, 0), max(end - step, 0), max(end - 1, 0)}:
        if start >= end:
            continue
        u, visited = start, 0
        while u < end and visited < 4:   # the last steps of the range, or a few of a long one
            n = lib.next(u, step, end)
            assert n == min(u + step, end)
            u, visited = n, visited + 1


@pytest.mark.parametrize("a", [0, 1, 23, 24, 25, INT_MAX - 7, INT_MAX])
@pytest.mark.parametrize("b", [1, 2, 4, 6, 24])
def test_ceil_div(lib, a, b):
    assert lib.div_up(a, b) == -(-a // b)
