"""Training pass of the preconditioner network with saturated units: silu of a
pre-activation of +-1e3 to +-1e35 is the value itself or zero, as in the FP64
oracle, and a NaN feature of a used sample reaches the loss."""
import numpy as np
import pytest

import chs
import mlp as OM

pytestmark = pytest.mark.gpu


def system(ctx):
    nb, lb = 3, 20
    n = nb * lb
    rng = np.random.default_rng(5)
    eb = np.repeat(rng.uniform(0.4, 2.0, nb), lb)
    feat = np.stack([rng.uniform(0.0, 12.0, n), np.log(eb), np.full(n, -0.3), np.full(n, 0.5)],
                    1).astype(np.float32)
    r = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    e = (-0.7 * r + 0.3 * (rng.standard_normal(n) + 1j * rng.standard_normal(n)))
    e, w = e.astype(np.complex64), np.ones(n, np.float32)
    net = chs.Mlp(ctx)
    th = (net.params + 0.1 * rng.standard_normal(net.params.size)).astype(np.float32)
    return net, th, feat, r, e, w, lb


def on_device(ctx, feat, r, e, w, lb):
    up = lambda x: chs.Gpu.from_host(ctx, x)
    return {"feat": up(feat), "r": up(r), "e": up(e), "w": up(w), "n": len(w), "cap": len(w),
            "band_len": lb}


# layer 1's biases start at 256, layer 2's weights at 320
@pytest.mark.parametrize("z", [-1e3, -1e5, -1e35, 1e3, 1e5])
def test_saturated_unit(ctx, z):
    net, th, feat, r, e, w, lb = system(ctx)
    th[256 + 3] = z
    if z > 0:  # the unit passes z on: keep what the next layer makes of it small
        th[320 + 3:320 + 64 * 64:64] = 0.3 / z * np.sign(th[320 + 3:320 + 64 * 64:64])
    net.params = th
    loss, grad = net.loss_grad(on_device(ctx, feat, r, e, w, lb))
    with np.errstate(over="ignore"):
        ref_loss, ref = OM.loss_grad(th, feat.astype(np.float64), r.astype(np.complex128),
                                     e.astype(np.complex128), w, lb)
    # the tolerances of the unsaturated network, and its gradient's scale apart
    # from the weights that take the large unit's value
    big = np.zeros(th.size, bool)
    big[320 + 3:320 + 64 * 64:64] = z > 0
    assert abs(loss - ref_loss) < 2e-6 * max(1.0, abs(ref_loss))
    for part in (big, ~big):
        if part.any():
            assert np.abs(grad - ref)[part].max() < 1e-4 * np.abs(ref)[part].max() + 1e-9
    net.close()


def test_nan_feature_reaches_the_loss(ctx):
    net, th, feat, r, e, w, lb = system(ctx)
    net.params = th
    feat[25, 2] = np.nan
    loss, grad = net.loss_grad(on_device(ctx, feat, r, e, w, lb))
    assert not np.isfinite(loss) or not np.isfinite(grad).all()
    net.close()
