"""Filter and Lanczos bound with ultrasoft projectors whose augmentation charges
are small, large or of very different size within one binding, against plain
numpy (S^{-1} through (1 + Q B)^{-1}, which no Q makes ill-conditioned)."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu

N, P = 24, 37
Q = {"0.1": np.full(P, 0.1), "1e-3": np.full(P, 1e-3), "1e-6": np.full(P, 1e-6),
     "1e-12": np.full(P, 1e-12), "mixed": np.logspace(-1, -12, P),
     "wide": np.logspace(3, -12, P)}


@pytest.fixture(params=list(Q))
def system(request, ctx):
    r = np.arange(-5, 6)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= 25]
    kin = 0.3 * (mil * mil).sum(1)
    rng = np.random.default_rng(11)
    rand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    v = 0.3 * rng.standard_normal((N, N, N))
    beta = rand(P, len(kin)) * 0.7 / np.sqrt(len(kin))
    d, q = rng.uniform(0.5, 2.0, P), Q[request.param]
    psi = rand(7, len(kin))
    ham = chs.Hamiltonian(ctx, N, mil, kin, v)
    ham.bind_projectors(beta, d, q)
    ix, iy, iz = (mil % N).T
    B = beta.conj() @ beta.T
    M = np.linalg.solve(np.eye(P) + q[:, None] * B, np.diag(q))

    def sinv_h(x):
        g = np.zeros((len(x), N, N, N), complex)
        g[:, iz, iy, ix] = x
        g = np.fft.fftn(np.fft.ifftn(g, axes=(1, 2, 3)) * v, axes=(1, 2, 3))
        y = kin * x + g[:, iz, iy, ix] + ((x @ beta.conj().T) * d) @ beta
        return y - ((y @ beta.conj().T) @ M.T) @ beta

    yield ctx, psi, sinv_h, beta, q
    del ham


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
def test_filter(system, dt):
    ctx, psi, sinv_h, _, _ = system
    b4 = np.array([14.0, 2.0, 8.0, 6.0])
    x = psi.astype(dt)
    got = chs.chebyshev_filter(ctx, chs.Gpu.from_host(ctx, x), 8, b4).sync_to_host()
    step = lambda y: (sinv_h(y) - b4[2] * y) / b4[3]
    a = x.astype(complex)
    b = step(a)
    for _ in range(7):
        a, b = b, 2.0 * step(b) - a
    # FP64: 8 steps of transforms and 500-term products, each a few eps of the
    # iterate; complex64: the filter's tolerance against the oracle
    tol = 1e-12 if dt == np.complex128 else 2e-5
    assert np.abs(got - b).max() / np.abs(b).max() < tol


def test_lanczos(system):
    ctx, psi, sinv_h, beta, q = system
    n, k, seed = psi.shape[1], 10, 4
    s, u = seed, []
    for _ in range(4 * n):
        s = (s * 25214903917 + 11) & 0xFFFFFFFFFFFF
        u.append(s / 2.0 ** 48)
    u = np.array(u).reshape(-1, 2)
    z = np.sqrt(-2.0 * np.log(1.0 - u[:, 0])) * np.cos(2.0 * np.pi * u[:, 1])
    S = lambda x: x + ((x @ beta.conj().T) * q) @ beta
    dot = lambda x, y: float((x.conj() * y).sum().real)
    v, vp, bp = (z[::2] + 1j * z[1::2])[None], 0.0, 0.0
    v = v / np.sqrt(dot(v, S(v)))
    al, be = [], []
    for _ in range(k):
        y = sinv_h(v)
        al.append(dot(S(v), y))
        f = y - al[-1] * v - bp * vp
        be.append(np.sqrt(dot(f, S(f))))
        vp, bp, v = v, be[-1], f / be[-1]
    w = np.linalg.eigvalsh(np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1))
    up, lo = chs.lanczos_bound(ctx, k, seed)
    # ten steps of FP64 vectors; rounding grows by a small factor a step
    assert abs(up - (w[-1] + be[-1])) < 1e-10 * abs(up)
    assert abs(lo - w[0]) < 1e-10 * abs(up)
