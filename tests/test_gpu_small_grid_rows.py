"""Plane kernel on grids with fewer rows than a large workgroup has lane
groups (16 to 36 points): after the tuner has run every launch shape, H|psi> must
be that of a plain numpy transform. (That no shape reads V_eff past its end is
checked on the CPU, in test_plane_shape.py.)"""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 24, 32, 36])
def test_hpsi_c64_after_tuning_on_small_grids(ctx, n):
    h = n // 4 - 1  # a sphere that fits half the grid
    r = np.arange(-h, h + 1)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= h * h]
    kin = 0.02 * (mil * mil).sum(1)
    rng = np.random.default_rng(n)
    v = rng.standard_normal((n, n, n))
    n_b = 5
    psi = (rng.standard_normal((n_b, len(kin))) + 1j * rng.standard_normal((n_b, len(kin))))
    psi = psi.astype(np.complex64)
    H = chs.Hamiltonian(ctx, n, mil, kin, v)
    chs.autotune_hpsi(ctx, n_b, chs.C64)
    got = chs.apply_full_hamiltonian(ctx, chs.Gpu.from_host(ctx, psi)).sync_to_host()
    ix, iy, iz = (mil % n).T
    g = np.zeros((n_b, n, n, n), complex)
    g[:, iz, iy, ix] = psi
    g = np.fft.fftn(np.fft.ifftn(g, axes=(1, 2, 3)) * v, axes=(1, 2, 3))
    ref = kin * psi + g[:, iz, iy, ix]
    # single-precision transforms of length n^3: a few eps log2(n^3)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 2e-5
    del H
