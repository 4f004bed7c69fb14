"""Lanczos bound on both sides of the length from which its vector steps run in
many workgroups, with ultrasoft projectors, against plain numpy."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [14, 15])  # 11,513 and 14,147 plane waves
def test_lanczos_bound_sizes(ctx, h):
    N, P, k, seed = 64, 5, 6, 4
    r = np.arange(-h, h + 1)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= h * h]
    n = len(mil)
    assert (n <= 12288) == (h == 14)
    kin = 0.05 * (mil * mil).sum(1)
    rng = np.random.default_rng(h)
    v0 = 0.3 * rng.standard_normal((N, N, N))
    beta = (rng.standard_normal((P, n)) + 1j * rng.standard_normal((P, n))) * 0.7 / np.sqrt(n)
    d, q = rng.uniform(0.5, 2.0, P), rng.uniform(0.1, 0.4, P)
    ham = chs.Hamiltonian(ctx, N, mil, kin, v0)
    ham.bind_projectors(beta, d, q)
    ix, iy, iz = (mil % N).T
    M = np.linalg.solve(np.eye(P) + q[:, None] * (beta.conj() @ beta.T), np.diag(q))
    proj = lambda x, c: ((x @ beta.conj().T) * c) @ beta

    def sinv_h(x):
        g = np.zeros((N, N, N), complex)
        g[iz, iy, ix] = x
        y = kin * x + np.fft.fftn(np.fft.ifftn(g) * v0)[iz, iy, ix] + proj(x, d)
        return y - ((y @ beta.conj().T) @ M.T) @ beta

    s, u = seed, []
    for _ in range(4 * n):
        s = (s * 25214903917 + 11) & 0xFFFFFFFFFFFF
        u.append(s / 2.0 ** 48)
    u = np.array(u).reshape(-1, 2)
    z = np.sqrt(-2.0 * np.log(1.0 - u[:, 0])) * np.cos(2.0 * np.pi * u[:, 1])
    dot = lambda x, y: float((x.conj() * (y + proj(y, q))).sum().real)
    v, vp, bp, al, be = z[::2] + 1j * z[1::2], 0.0, 0.0, [], []
    v = v / np.sqrt(dot(v, v))
    for _ in range(k):
        y = sinv_h(v)
        al.append(dot(v, y))
        f = y - al[-1] * v - bp * vp
        be.append(np.sqrt(dot(f, f)))
        vp, bp, v = v, be[-1], f / be[-1]
    w = np.linalg.eigvalsh(np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1))
    up, lo = chs.lanczos_bound(ctx, k, seed)
    # six steps of FP64 vectors; rounding grows by a small factor a step
    assert abs(up - (w[-1] + be[-1])) < 1e-10 * abs(up)
    assert abs(lo - w[0]) < 1e-10 * abs(up)
    del ham
