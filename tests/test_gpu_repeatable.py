"""FP64 products and Rayleigh-Ritz do not depend on the tuner's timings: a
tuning context, one without tuning and one per kernel choice give the same sums
for a shape, and the eigenvectors keep their signs."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


def product(monkeypatch, opa, m, n, k, a, b, **env):
    for name in ("CHS_GEMM_TUNE", "CHS_GEMM_CHOICE"):
        monkeypatch.delenv(name, raising=False)
    for name, v in env.items():
        monkeypatch.setenv(name, v)
    c = chs.Context(0)
    out = chs.Gpu.from_host(c, np.zeros((n, m), complex))
    chs.zgemm(c, opa, "N", m, n, k, 1.0, chs.Gpu.from_host(c, a), a.shape[1],
              chs.Gpu.from_host(c, b), k, 0.0, out, m)
    got = out.sync_to_host()
    c.close()
    return got


# K slices: many and short, the bound on their length, one
@pytest.mark.parametrize("opa,m,n,k,ti", [("C", 512, 512, 20001, 1), ("C", 160, 97, 4099, 0),
                                          ("C", 449, 449, 1023, 0), ("N", 700, 33, 65, 0)])
def test_zgemm_sums_follow_the_shape(monkeypatch, opa, m, n, k, ti):
    rng = np.random.default_rng(k)
    rand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    a, b = rand(*((m, k) if opa == "C" else (k, m))), rand(n, k)
    tuned = product(monkeypatch, opa, m, n, k, a, b)
    assert np.array_equal(tuned, product(monkeypatch, opa, m, n, k, a, b, CHS_GEMM_TUNE="0"))
    for v in (1, 3):  # the 64 x 64 kernels at the same split
        got = product(monkeypatch, opa, m, n, k, a, b, CHS_GEMM_CHOICE=str(v + 16 * ti))
        assert np.array_equal(tuned, got)
    ref = (a.conj() if opa == "C" else a.T) @ b.T
    # three real products of K terms, each sum rounded as it grows
    assert np.abs(tuned - ref.T).max() < 64 * 2.0 ** -53 * (np.sqrt(k) + 8) * np.sqrt(k)


def test_eigenvector_signs_follow_the_input(monkeypatch):
    n, h, n_b = 64, 14, 400  # 28 upper tiles, 18 or more slices of K = 11,513
    r = np.arange(-h, h + 1)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= h * h]
    kin = 0.05 * (mil * mil).sum(1)
    rng = np.random.default_rng(3)
    psi = rng.standard_normal((n_b, len(kin))) + 1j * rng.standard_normal((n_b, len(kin)))
    v = 0.3 * rng.standard_normal((n, n, n))
    out = []
    for tune in ("1", "0"):
        monkeypatch.setenv("CHS_GEMM_TUNE", tune)
        c = chs.Context(0)
        H = chs.Hamiltonian(c, n, mil, kin, v)
        y = chs.Gpu.from_host(c, psi)
        eps, _ = chs.rayleigh_ritz(c, y)
        out.append((eps, y.sync_to_host()))
        del H
        c.close()
    assert np.array_equal(out[0][0], out[1][0])
    # the back-transformation's products are tuned among kernels that add in
    # another order: a few eps, where a changed sign would show as 2
    assert np.abs(out[0][1] - out[1][1]).max() < 1e-10 * np.abs(out[0][1]).max()
