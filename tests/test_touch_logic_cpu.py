"""The lines that a launch asks for ahead (csrc/touch_logic.h), on the CPU: every line of every range is read once and
nothing outside the ranges, by workgroups of their own and by wavefronts beside the computing ones."""
import ctypes as C
import os
import subprocess
import tempfile

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib():
    so = os.path.join(tempfile.mkdtemp(prefix="lbm_touch_host_"), "touch_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-Wno-unknown-pragmas", "-o", so,
                           os.path.join(HERE, "native", "touch_host.cpp")])
    got = C.CDLL(so)
    got.lbm_touch_host.restype = C.c_longlong
    return got


@pytest.mark.parametrize("lines", [(0, 0, 0, 0), (1, 0, 0, 0), (8, 9, 15, 1), (16384, 65536, 65536, 49152)])
@pytest.mark.parametrize("launch", [(48, 208, 448, None), (1, 255, 448, None), (224, 32, 448, None), (384, 128, 512, None), (127, 0, 448, 384),
                                    (128, 0, 704, 640), (1, 0, 448, 384)])
def test_every_line_is_read_once(lib, lines, launch):
    grid_x, wgs, threads, wave_first = launch
    grid_y = 1 + -(-wgs // grid_x)
    at = [(r + 1) << 40 for r in range(4)]
    reads = [np.zeros(max(n, 1), dtype=np.int32) for n in lines]
    outside = lib.lbm_touch_host((C.c_uint * 4)(*lines), (C.c_longlong * 4)(*at), wgs, grid_x, grid_y, threads,
                                 -1 if wave_first is None else wave_first, (C.POINTER(C.c_int) * 4)(*[r.ctypes.data_as(C.POINTER(C.c_int)) for r in reads]))
    assert outside == 0
    for n, r in zip(lines, reads):
        assert (r[:n] == 1).all()
