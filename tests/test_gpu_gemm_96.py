"""complex64 GEMM tiles of 96 rows (96 x 64 and 96 x 32) at the edges of their
tiles, K stages and slices, against float64 numpy; the choice falls back to a
64 x 64 tile for the operand forms these tiles do not have."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("choice", [7, 8, 0x37, 0x38])
@pytest.mark.parametrize("opa,opb,m,n,k", [("N", "N", 96, 64, 16), ("N", "N", 97, 65, 17),
                                           ("C", "N", 95, 33, 15), ("C", "N", 193, 31, 1300),
                                           ("N", "N", 1, 160, 33), ("C", "N", 200, 97, 4099),
                                           ("N", "C", 100, 40, 70), ("T", "N", 100, 40, 70)])
def test_96_row_tiles(monkeypatch, choice, opa, opb, m, n, k):
    monkeypatch.setenv("CHS_GEMM_CHOICE", str(choice))
    c = chs.Context(0)
    rng = np.random.default_rng(choice + m)
    rand = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    op = lambda x, o: x if o == "N" else x.T if o == "T" else x.conj().T
    A, B = rand(*((m, k) if opa == "N" else (k, m))), rand(*((k, n) if opb == "N" else (n, k)))
    C0 = rand(m, n)
    f = lambda x: chs.Gpu.from_host(c, np.ascontiguousarray(x.T))  # column-major
    a, b, cc = f(A), f(B), f(C0)
    P = chs.C.POINTER(chs.C.c_float)
    al, be = np.array([0.7, -0.2], np.float32), np.array([0.3, 0.1], np.float32)
    c.check(chs.lib().chs_cgemm(c.h, opa.encode(), opb.encode(), m, n, k, al.ctypes.data_as(P),
                                a.ptr, A.shape[0], b.ptr, B.shape[0], be.ctypes.data_as(P), cc.ptr,
                                m))
    got = cc.sync_to_host().T
    ref = (0.7 - 0.2j) * op(A.astype(complex), opa) @ op(B.astype(complex), opb) \
        + (0.3 + 0.1j) * C0.astype(complex)
    # the tolerance of the other complex64 kernels
    assert np.abs(got - ref).max() / np.abs(ref).max() < 3e-6
    c.close()
