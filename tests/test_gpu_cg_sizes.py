"""The conductance solve at the edges of its kernels' work split: one row, one
block, more rows than one pass of the grid; solves that end before, at and
after batches of iterations are queued ahead.  Chains of rods between the
electrodes whose lengths and places are exact in binary, so the closed form is
exact; a residual of 1e-12 bounds the error by the condition number of a chain
of n, at most 4 n^2."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu

LEN, A, GAP, LAM = 0.875, 1.0 / 64.0, 0.1, 0.02


def _chains(count, n):
    side = int(np.ceil(np.sqrt(count)))
    edge = max(2.0, 0.25 * side)
    y, z = np.divmod(np.arange(count), side)
    r = np.zeros((count, n, 8), np.float32)
    r[:, :, 0] = np.arange(n) + 0.5
    r[:, :, 1] = (0.25 * y + 0.125)[:, None]
    r[:, :, 2] = (0.25 * z + 0.125)[:, None]
    r[:, :, 3] = 1.0
    r[:, :, 6] = LEN
    r[:, :, 7] = A
    p = nf.normalize(nf.default_params(box=(float(max(n, 2)), edge, edge), n_rods=count * n, len=LEN, radius=A,
                                       contact_gap=GAP, elec_axis=0, tunnel_lambda=LAM, precision=nf.NF_PREC_FP64))
    return p, r.reshape(-1, 8)


def _resistances(p, n):
    g = lambda gap: p.tunnel_g0 * np.exp(-gap / LAM)
    inner, end = 1.0 - LEN - 2 * A, 0.5 - LEN / 2 - A
    return np.array([1 / g(end)] + [1 / g(inner)] * (n - 1) + [1 / g(end)])


@pytest.mark.parametrize("count,n", [(1, 2), (1, 200), (3, 5), (51, 5), (70, 129), (90000, 3)])
def test_chains(count, n):
    p, rods = _chains(count, n)
    res = _resistances(p, n)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        pk.contacts(GAP)
        pk.network()
        for _ in range(2):
            ci, v = pk.conductance(tol=1e-12, max_iter=1000, potentials=True)
            tol = 4 * n * n * 1e-12
            assert ci["converged"] == 1 and ci["unknowns"] == count * n and ci["residual"] <= 1e-12
            assert ci["conductance"] == pytest.approx(count / res.sum(), rel=max(tol, 1e-11))
            assert ci["current_sink"] == pytest.approx(count / res.sum(), rel=max(tol, 1e-11))
            want = 1.0 - np.cumsum(res)[:-1] / res.sum()
            np.testing.assert_allclose(v.reshape(count, n), np.broadcast_to(want, (count, n)), atol=max(tol, 1e-11))


@pytest.mark.parametrize("max_iter", [1, 16, 17, 128, 143, 150])
def test_iterations_end_at_the_limit(max_iter):
    p, rods = _chains(2, 200)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        pk.contacts(GAP)
        pk.network()
        ci, _ = pk.conductance(tol=1e-14, max_iter=max_iter, potentials=True)
        assert ci["iterations"] == max_iter and ci["converged"] == 0
        full, v = pk.conductance(tol=1e-12, max_iter=5000, potentials=True)
        assert full["converged"] == 1 and full["iterations"] % 16 == 0
