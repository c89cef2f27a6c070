"""Sizes and electrodes of components counted by waves and blocks: one component
of everything, pairs only, two that alternate by id, sizes around a block."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu

LEN, A, GAP, LAM = 0.875, 1.0 / 64.0, 0.1, 0.02


def _rows(count, n, order):
    """count chains of n rods along x; order: rods of one chain together, or taken in turn."""
    side = int(np.ceil(np.sqrt(count)))
    y, z = np.divmod(np.arange(count), side)
    r = np.zeros((count, n, 8), np.float32)
    r[:, :, 0] = np.arange(n) + 0.5
    r[:, :, 1] = (0.25 * y + 0.125)[:, None]
    r[:, :, 2] = (0.25 * z + 0.125)[:, None]
    r[:, :, 3] = 1.0
    r[:, :, 6] = LEN
    r[:, :, 7] = A
    if order == "in turn":
        r = r.transpose(1, 0, 2)
    r = np.ascontiguousarray(r.reshape(-1, 8))
    if order == "mixed":
        r = r[np.random.default_rng(1).permutation(len(r))]
    return r, max(2.0, 0.25 * side)


@pytest.mark.parametrize("order", ["together", "in turn", "mixed"])
@pytest.mark.parametrize("count,n,span", [(1, 1, 4), (1, 1100, 0), (2, 700, 0), (513, 2, 0), (3, 341, 0), (600, 2, 4),
                                          (40000, 2, 0), (2, 20000, 0)])
def test_components(count, n, span, order):
    if count * n > 2000 and order == "mixed":
        order = "together"
    rods, edge = _rows(count, n, order)
    length = float(max(n + span, 2))
    p = nf.normalize(nf.default_params(box=(length, edge, edge), n_rods=len(rods), len=LEN, radius=A, contact_gap=GAP,
                                       elec_axis=0, tunnel_lambda=LAM, precision=nf.NF_PREC_FP64))
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        c = pk.contacts(GAP)
        info, net = pk.network()
        labels = net["labels"]
        ids, sizes = np.unique(labels, return_counts=True)
        assert info["n_components"] == len(ids) == count and info["largest"] == sizes.max() == n
        assert info["percolating"] == (count if span == 0 else 0)
        assert info["n_edges"] == count * (n - 1)
        assert info["n_source"] == count and info["n_sink"] == (count if span == 0 else 0)
        ci, v = pk.conductance(potentials=True, max_iter=16)
        assert ci["unknowns"] == (count * n if span == 0 else 0)
