"""Kernel choices that name no kernel (from CHS_GEMM_CHOICE or a line of the
tuning cache) run the vector kernel: every output is written."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("choice", [9, 15, 0x3c])
@pytest.mark.parametrize("dt,tol", [(np.complex64, 3e-6), (np.complex128, 1e-13)])
def test_unknown_kernel_choice(monkeypatch, choice, dt, tol):
    monkeypatch.setenv("CHS_GEMM_CHOICE", str(choice))
    c = chs.Context(0)
    rng = np.random.default_rng(choice)
    m, n, k = 300, 260, 700
    rand = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(dt)
    A, B, C0 = rand(m, k), rand(n, k), rand(n, m)  # column-major A (k x m), B (k x n), C
    a, b, cc = (chs.Gpu.from_host(c, x) for x in (A, B, C0))
    if dt == np.complex128:
        chs.zgemm(c, "C", "N", m, n, k, 1.0, a, k, b, k, 0.0, cc, m)
    else:
        P = chs.C.POINTER(chs.C.c_float)
        one, zero = np.array([1, 0], np.float32), np.zeros(2, np.float32)
        c.check(chs.lib().chs_cgemm(c.h, b"C", b"N", m, n, k, one.ctypes.data_as(P), a.ptr, k,
                                    b.ptr, k, zero.ctypes.data_as(P), cc.ptr, m))
    ref = B.astype(complex) @ A.astype(complex).conj().T
    # the tolerances of the other kernel choices
    assert np.abs(cc.sync_to_host() - ref).max() < tol * np.abs(ref).max()
    c.close()
