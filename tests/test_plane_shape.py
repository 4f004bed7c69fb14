"""Row buffers of the plane kernels on the CPU: plane_shape.hpp compiled with the
host compiler and asked for every grid, launch shape, precision and divisor."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "chemrust-scf_amd", "csrc")
LDS = 160 * 1024
# second radix of each grid's line and its row scratch in 8-byte slots
GRIDS = {8: (4, 12), 12: (4, 20), 16: (4, 20), 18: (9, 27), 24: (6, 70), 32: (8, 40), 36: (9, 41),
         48: (12, 108), 64: (8, 72), 72: (9, 88), 96: (12, 140), 108: (9, 137), 128: (16, 144),
         144: (12, 204)}


@pytest.fixture(scope="module")
def row_buffers(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    src = d / "shape.cpp"
    src.write_text('#include "plane_shape.hpp"\nextern "C" int f(size_t l, size_t c, size_t r, '
                   'size_t t, size_t z, int n, int na, int g, int d) {\n'
                   '  return chs::plane_row_buffers(l, c, r, t, z, n, na, g, d);\n}\n')
    so = d / "shape.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(so)],
                   check=True)
    f = ctypes.CDLL(str(so)).f
    f.argtypes = [ctypes.c_size_t] * 5 + [ctypes.c_int] * 4
    return f


def shapes():
    for n, (n2, slots) in GRIDS.items():
        for csz in (8, 16):
            for threads in (256, 512, 1024):
                for div in (1, 2, 4, 8):
                    for n_act in sorted({1, n // 4, n // 2 - 1, n}):
                        for extra in (0, 8 * n2 * (16 + 1)):
                            yield n, n2, slots, csz, threads, div, n_act, extra


def test_row_buffers_stay_on_the_plane(row_buffers):
    some = 0
    for n, n2, slots, csz, threads, div, n_act, extra in shapes():
        for rs in (n // 2 + 1, n):
            cmp_bytes, row, tab = n * rs * csz, 8 * slots, 4 * n + extra
            groups = threads // 64 * (64 // n2)
            nrb = row_buffers(LDS, cmp_bytes, row, tab, csz, n, n_act, groups, div)
            at = (n, csz, threads, div, n_act, extra, rs, nrb)
            if cmp_bytes + row + tab > LDS:
                assert nrb == 0, at
                continue
            assert 1 <= nrb <= min(n, groups), at  # group g loads row g's V_eff
            assert cmp_bytes + nrb * row + tab <= LDS, at
            some += 1
            if csz == 16:  # every group that the divisor and the LDS leave
                assert nrb == min(n, max(1, min(groups, (LDS - cmp_bytes - tab) // row) // div)), at
    assert some > 1000


def test_plane_that_does_not_fit(row_buffers):
    assert row_buffers(LDS, LDS - 100, 101, 0, 8, 64, 30, 28, 1) == 0
    assert row_buffers(LDS, LDS - 100, 100, 0, 8, 64, 30, 28, 1) == 1
