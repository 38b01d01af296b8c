"""Which workgroup of a linear takes which tile (csrc/tile_logic.h), on the CPU: every tile is taken once."""
import ctypes as C
import os
import subprocess
import tempfile

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib():
    so = os.path.join(tempfile.mkdtemp(prefix="lbm_tiles_host_"), "tiles_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-o", so, os.path.join(HERE, "native", "tiles_host.cpp")])
    got = C.CDLL(so)
    got.lbm_tiles_host.restype = got.lbm_divide_host.restype = C.c_longlong
    return got


@pytest.mark.parametrize("panel_shift", [2, 3])
def test_every_tile_is_taken_once(lib, panel_shift):
    for m_tiles in (1, 2, 3, 7, 9, 31, 32, 33, 257):
        for n_tiles in (1, 3, 4, 5, 8, 11, 12, 15, 16, 48, 64, 65):
            hits = np.zeros(m_tiles * n_tiles, dtype=np.int32)
            assert lib.lbm_tiles_host(m_tiles, n_tiles, panel_shift, hits.ctypes.data_as(C.c_void_p)) == 0
            assert (hits == 1).all(), (m_tiles, n_tiles)


@pytest.mark.parametrize("d", [1, 2, 3, 5, 7, 8, 12, 63, 64, 100, 1023, 65535, 65536, 65537, 2 ** 31 - 1])
def test_division_by_a_launch_constant(lib, d):
    assert lib.lbm_divide_host(C.c_longlong(0), C.c_longlong(9973), d) == -1
    assert lib.lbm_divide_host(C.c_longlong(2 ** 31 - 1 - 70000), C.c_longlong(1), d) == -1
