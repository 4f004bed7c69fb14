"""Growth guard of the filters with projectors bound, where it runs one step
behind the recurrence: the step it names and its norms, against numpy.

One plane wave that nothing couples to lies X = 20 half widths above the window;
its share of the block starts at `a` and grows about 40-fold a step, so `a` sets
the step at which the block's norm first grows more than tenfold."""
import numpy as np
import pytest

import chs

pytestmark = pytest.mark.gpu

N, P, N_B = 16, 9, 5
B4 = np.array([14.0, 2.0, 8.0, 6.0])
OUT = 0  # the outlying plane wave


def parts(seed, q0):
    r = np.arange(-3, 4)
    mil = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    mil = mil[(mil * mil).sum(1) <= 9 - seed]
    kin = 3.0 + 0.5 * (mil * mil).sum(1)
    kin[OUT] = B4[2] + 20.0 * B4[3]
    rng = np.random.default_rng(seed)
    rand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    beta = rand(P, len(kin)) * 0.5 / np.sqrt(len(kin))
    beta[:, OUT] = 0.0
    psi = rand(N_B, len(kin))
    psi /= np.linalg.norm(psi)
    return mil, kin, beta, rng.uniform(0.2, 0.6, P), np.full(P, q0), psi


def operator(kin, beta, d, q):
    """S^{-1} H with V_eff = 0."""
    M = np.linalg.solve(np.eye(P) + q[:, None] * (beta.conj() @ beta.T), np.diag(q))

    def op(x):
        y = kin * x + ((x @ beta.conj().T) * d) @ beta
        return y - ((y @ beta.conj().T) @ M.T) @ beta
    return op


def expected(norms, first):
    """First step whose norm is over ten times the step's before, from first + 1."""
    for k in range(first + 1, len(norms)):
        if norms[k] > 10.0 * norms[k - 1]:
            return k, norms[k - 1], norms[k]
    return None


def plain_norms(op, x, degree):
    a, b = x, (op(x) - B4[2] * x) / B4[3]
    out = [np.linalg.norm(a), np.linalg.norm(b)]
    for _ in range(degree - 1):
        a, b = b, 2.0 * (op(b) - B4[2] * b) / B4[3] - a
        out.append(np.linalg.norm(b))
    return out


def check(call, want, tol):
    if want is None:
        call()
        return
    with pytest.raises(chs.ChebyshevDiverged) as e:
        call()
    d = e.value.diag
    assert d.iteration == want[0]
    assert abs(d.norm_previous - want[1]) < tol * want[1]
    assert abs(d.norm_current - want[2]) < tol * want[2]
    assert abs(d.growth_factor - want[2] / want[1]) < 2 * tol * want[2] / want[1]


# the share, the step it makes the guard name, the degree: that step the last
# one, one in the middle, none reached
CASES = [(1.0, 2, 2), (1.0, 2, 5), (3e-4, 3, 3), (3e-4, 3, 4), (1e-5, 4, 4), (1e-5, 4, 6),
         (1.0, None, 1), (3e-4, None, 2)]


@pytest.mark.parametrize("q0", [0.0, 0.25])
@pytest.mark.parametrize("dt,tol", [(np.complex128, 1e-11), (np.complex64, 1e-4)])
@pytest.mark.parametrize("a,step,degree", CASES)
def test_plain_filter(ctx, a, step, degree, dt, tol, q0):
    mil, kin, beta, d, q, psi = parts(0, q0)
    psi[:, OUT] = a / np.sqrt(N_B)
    want = expected(plain_norms(operator(kin, beta, d, q), psi, degree), 1)
    assert (want and want[0]) == step
    ham = chs.Hamiltonian(ctx, N, mil, kin, np.zeros((N, N, N)))
    ham.bind_projectors(beta, d, q)
    x = chs.Gpu.from_host(ctx, psi.astype(dt))
    check(lambda: chs.chebyshev_filter(ctx, x, degree, B4), want, tol)
    del ham


@pytest.mark.parametrize("prec,tol", [("C128", 1e-9), ("C64", 1e-4)])
@pytest.mark.parametrize("q0", [0.0, 0.25])
@pytest.mark.parametrize("a,step,degree", [(1.0, 3, 3), (1.0, 3, 5), (1e-4, 4, 4), (1e-4, 4, 6),
                                           (1.0, None, 2), (1e-4, None, 3)])
def test_residual_filter(ctx, a, step, degree, q0, prec, tol):
    mil, kin, beta, d, q, psi = parts(0, q0)
    psi[:, OUT] = a / np.sqrt(N_B)
    eps = np.linspace(4.0, 6.0, N_B)
    op = operator(kin, beta, d, q)
    w = op(psi) - eps[:, None] * psi
    t0, t1 = np.ones(N_B), (eps - B4[2]) / B4[3]
    r0, r1 = np.zeros_like(psi), w / B4[3]
    norms = [0.0, np.linalg.norm(r1)]
    for _ in range(degree - 1):
        r0, r1 = r1, 2.0 * (op(r1) - B4[2] * r1) / B4[3] - r0 + (2.0 / B4[3]) * t1[:, None] * w
        t0, t1 = t1, 2.0 * (eps - B4[2]) / B4[3] * t1 - t0
        norms.append(np.linalg.norm(r1))
    want = expected(norms, 2)
    assert (want and want[0]) == step
    ham = chs.Hamiltonian(ctx, N, mil, kin, np.zeros((N, N, N)))
    ham.bind_projectors(beta, d, q)
    x = chs.Gpu.from_host(ctx, psi)
    check(lambda: chs.chebyshev_filter_residual(ctx, x, eps, degree, B4, getattr(chs, prec)), want,
          tol)
    del ham


@pytest.mark.parametrize("dt,tol", [(np.complex128, 1e-11), (np.complex64, 1e-4)])
def test_kpoint_filter(ctx, dt, tol):
    """Three k-points, the second diverging at step 3, on the eager call and on
    graph replays."""
    ks = [parts(s, 0.25) for s in range(3)]
    dev = lambda x: chs.Gpu.from_host(ctx, x)
    d, q = ks[0][3], ks[0][4]
    kset = chs.KSet(ctx, N, [dev(k[0]) for k in ks], [dev(k[1]) for k in ks],
                    dev(np.zeros((N, N, N))), [dev(k[2]) for k in ks], dev(d), dev(q))
    for i, k in enumerate(ks):
        k[5][:, OUT] = (3e-4 if i == 1 else 0.0) / np.sqrt(N_B)
    want = expected(plain_norms(operator(ks[1][1], ks[1][2], d, q), ks[1][5], 5), 1)
    assert want[0] == 3
    blocks = [dev(k[5].astype(dt)) for k in ks]
    for _ in range(3):
        for b, k in zip(blocks, ks):
            src = dev(k[5].astype(dt))
            ctx.check(chs.lib().chs_d2d(ctx.h, b.ptr, src.ptr, src.nbytes))
        with pytest.raises(chs.ChebyshevDiverged, match="k-point 1"):
            check_diag(kset, blocks, want, tol)
    del kset


def check_diag(kset, blocks, want, tol):
    try:
        kset.filter(blocks, 5, np.tile(B4, (3, 1)))
    except chs.ChebyshevDiverged as e:
        assert e.diag.iteration == want[0]
        assert abs(e.diag.norm_previous - want[1]) < tol * want[1]
        assert abs(e.diag.norm_current - want[2]) < tol * want[2]
        raise
