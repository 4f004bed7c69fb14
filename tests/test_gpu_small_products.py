"""The small-product GEMM kernel (32 x 32 tiles, K split over wavefronts) at the
edges of its tiles, K chunks and slices, and the filter's coefficient step that
uses it, with and without an S matrix, against plain numpy."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


def cgemm(c, dt, opa, m, n, k, a, lda, b, ldb, be, cc, ldc):
    if dt == np.complex128:
        chs.zgemm(c, opa, "N", m, n, k, 1.0, a, lda, b, ldb, be, cc, ldc)
        return
    fp = lambda v: np.array([v, 0.0], np.float32)
    one, bet = fp(1.0), fp(be)
    P = chs.C.POINTER(chs.C.c_float)
    c.check(chs.lib().chs_cgemm(c.h, opa.encode(), b"N", m, n, k, one.ctypes.data_as(P), a.ptr, lda,
                                b.ptr, ldb, bet.ctypes.data_as(P), cc.ptr, ldc))


@pytest.mark.parametrize("opa", ["N", "C"])
@pytest.mark.parametrize("m,n,k", [(1, 2, 1), (31, 33, 7), (32, 32, 8), (33, 31, 9), (64, 20, 31),
                                   (40, 17, 128), (32, 20, 2945), (65, 70, 1027)])
def test_small_kernel_edges(monkeypatch, opa, m, n, k):
    monkeypatch.setenv("CHS_GEMM_CHOICE", "6")
    c = chs.Context(0)
    rng = np.random.default_rng(m * 1000 + k)
    rand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    ldb, ldc = k + 3, m + 5
    A = rand(k, m) if opa == "N" else rand(m, k)  # column-major op(A), its leading axis last
    B, C0 = rand(n, ldb), rand(n, ldc)
    opA = A.T if opa == "N" else A.conj()
    for dt, eps in ((np.complex128, 2.0 ** -53), (np.complex64, 2.0 ** -24)):
        a, b, c0 = A.astype(dt), B.astype(dt), C0.astype(dt)
        cc = chs.Gpu.from_host(c, c0)
        cgemm(c, dt, opa, m, n, k, chs.Gpu.from_host(c, a), m if opa == "N" else k,
              chs.Gpu.from_host(c, b), ldb, 0.5, cc, ldc)
        got = cc.sync_to_host()
        ref = (opA.astype(dt).astype(complex) @ b[:, :k].T.astype(complex)).T \
            + 0.5 * c0[:, :m].astype(complex)
        # three real products of K terms, each sum rounded as it grows
        bound = 16 * eps * (np.sqrt(k) + 8) * np.sqrt(k + 1)
        assert np.abs(got[:, :m] - ref).max() < bound * 4
        assert np.array_equal(got[:, m:], c0[:, m:])  # rows past m untouched
    c.close()


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("q0", [0.0, 0.25])
def test_filter_coefficient_step(ctx, q0, dt):
    n, h, n_b, P, deg = 24, 5, 7, 37, 6
    r = np.arange(-h, h + 1)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= h * h]
    kin = 0.3 * (mil * mil).sum(1)
    rng = np.random.default_rng(11)
    rand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    v = 0.3 * rng.standard_normal((n, n, n))
    beta = rand(P, len(kin)) * 0.7 / np.sqrt(len(kin))
    d, q = rng.uniform(0.5, 2.0, P), np.full(P, q0)
    psi = rand(n_b, len(kin)).astype(dt)
    ham = chs.Hamiltonian(ctx, n, mil, kin, v)
    ham.bind_projectors(beta, d, q)
    b4 = np.array([14.0, 2.0, 8.0, 6.0])
    got = chs.chebyshev_filter(ctx, chs.Gpu.from_host(ctx, psi), deg, b4).sync_to_host()
    ix, iy, iz = (mil % n).T

    def op(x):
        g = np.zeros((n_b, n, n, n), complex)
        g[:, iz, iy, ix] = x
        g = np.fft.fftn(np.fft.ifftn(g, axes=(1, 2, 3)) * v, axes=(1, 2, 3))
        y = kin * x + g[:, iz, iy, ix] + ((x @ beta.conj().T) * d) @ beta
        if q0:
            M = np.linalg.inv(np.diag(1.0 / q) + beta.conj() @ beta.T)
            y = y - ((y @ beta.conj().T) @ M.T) @ beta
        return (y - b4[2] * x) / b4[3]

    a = psi.astype(complex)
    b = op(a)
    for _ in range(deg - 1):
        a, b = b, 2.0 * op(b) - a
    # the filter's tolerances against the oracle
    assert np.abs(got - b).max() / np.abs(b).max() < (1e-10 if dt == np.complex128 else 2e-5)
    del ham
