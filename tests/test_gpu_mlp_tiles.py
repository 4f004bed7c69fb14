"""Training pass of the preconditioner network at the edges of its 16-sample
tiles and 4-wavefront workgroups: band lengths around a tile,
more bands than wavefronts, masked bands; against the FP64 oracle."""
import numpy as np
import pytest

import chs
import mlp as OM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,lb", [(2, 15), (3, 16), (5, 17), (9, 33), (1100, 16)])
def test_loss_grad_tile_edges(ctx, nb, lb):
    rng = np.random.default_rng(100 * nb + lb)
    n = nb * lb
    eb = np.repeat(rng.uniform(0.4, 2.0, nb), lb)
    feat = np.stack([rng.uniform(0.0, 12.0, n), np.log(eb), np.full(n, -0.3), np.full(n, 0.5)],
                    1).astype(np.float32)
    r = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    e = (-0.7 * r + 0.3 * (rng.standard_normal(n) + 1j * rng.standard_normal(n)))
    e = e.astype(np.complex64)
    w = np.ones(n, np.float32)
    if nb > 2:
        w[lb:2 * lb] = 0.0  # a band without a reference partner
    net = chs.Mlp(ctx)
    th = net.params
    th = (th + 0.1 * rng.standard_normal(th.size)).astype(np.float32)  # every layer takes part
    net.params = th
    pairs = {"feat": chs.Gpu.from_host(ctx, feat), "r": chs.Gpu.from_host(ctx, r),
             "e": chs.Gpu.from_host(ctx, e), "w": chs.Gpu.from_host(ctx, w), "n": n, "cap": n,
             "band_len": lb}
    loss, grad = net.loss_grad(pairs)
    ref_loss, ref = OM.loss_grad(th, feat.astype(np.float64), r.astype(np.complex128),
                                 e.astype(np.complex128), w, lb)
    # FP32 products of 64 terms through three layers and their transposes, and
    # the loss coefficient g2 s c - a, whose terms cancel to about a tenth
    assert abs(loss - ref_loss) < 2e-6 * max(1.0, abs(ref_loss))
    assert np.abs(grad - ref).max() < 1e-4 * np.abs(ref).max() + 1e-9
    net.close()
