"""Contacts from crossing lists against the oracle and the cell-pair engine:
rods across faces, inexact and far-off directions, lists that are too short,
wide gaps, the smallest packings."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu


def _rods(n, box, length, seed, radius=0.005, spread=None):
    g = np.random.default_rng(seed)
    u = g.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    r = np.zeros((n, 8), np.float32)
    r[:, :3] = g.uniform(0, 1, (n, 3)) * np.asarray(box) * 0.999999
    r[:, 3:6] = u
    r[:, 6] = length if np.isscalar(length) else g.uniform(*length, n)
    r[:, 7] = radius if np.isscalar(radius) else g.uniform(*radius, n)
    return r


def _scaled(r, f, seed):
    g = np.random.default_rng(seed)
    r = r.copy()
    r[:, 3:6] *= g.uniform(1 - f, 1 + f, (len(r), 1)).astype(np.float32)
    return r


B = (3.0, 3.0, 3.0)
CASES = {
    "one rod": (B, _rods(1, B, 1.0, 1), 0.01),
    "two rods": (B, _rods(2, B, 2.5, 2), 0.4),
    "uniform": (B, _rods(1500, B, 1.0, 3), 0.002),
    "a rod spans the box": ((1.05, 1.3, 1.1), _rods(80, (1.05, 1.3, 1.1), 2.0, 4), 0.004),
    "mixed lengths and radii": (B, _rods(1500, B, (0.05, 2.5), 5, radius=(0.001, 0.03)), 0.003),
    "directions off by 4e-4": (B, _scaled(_rods(1500, B, 1.0, 6), 4e-4, 6), 0.002),
    "directions off by 5%: another way": (B, _scaled(_rods(1500, B, 1.0, 7), 0.05, 7), 0.002),
    "gap as wide as the rods: another way": (B, _rods(200, B, 0.5, 8), 0.5),
    "longer than the box: another way": ((1.2, 1.2, 1.2), _rods(60, (1.2, 1.2, 1.2), 3.0, 9), 0.004),
    "all in one corner: lists too short": (B, _rods(1500, (0.3, 0.3, 0.3), 1.0, 10), 0.001),
}


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("name", list(CASES))
def test_same_contacts_as_the_oracle(name, prec):
    box, rods, gap = CASES[name]
    p = nf.normalize(nf.default_params(box=box, n_rods=len(rods), len=float(rods[:, 6].max()), radius=0.005,
                                       contact_gap=gap, precision=prec))
    o = oracle.contacts(p, rods, gap, threads=4)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        for _ in range(2):
            c = pk.contacts(gap)
            g64 = pk.contact_gap64(c.n)
            np.testing.assert_array_equal(c.I, o["I"])
            np.testing.assert_array_equal(c.col, o["J"])
            np.testing.assert_array_equal(c.image, o["image"])
            np.testing.assert_array_equal(g64.view(np.uint64), o["gap64"].view(np.uint64))


@pytest.mark.parametrize("n,law", [(50000, "const"), (70000, "const"), (150000, "lognormal")])
def test_same_contacts_as_every_pair(n, law):
    """Generated packings on both sides of the size rule, and the network's
    walk after either cell list."""
    kw = dict(len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.3, len_min=0.3, len_max=3.0) if law == "lognormal" else {}
    edge = (n / 70.0) ** (1.0 / 3.0)
    p = nf.normalize(nf.default_params(box=(edge,) * 3, n_rods=n, len=1.0, radius=0.005, seed=17, contact_gap=0.002, **kw))
    got = []
    for engine in (nf.NF_ENGINE_FOOTPRINT, nf.NF_ENGINE_CELLS):
        with nf.Packing(p, {nf.NF_OPT_CONTACT_ENGINE: engine}) as pk:
            pk.generate()
            c = pk.contacts(p.contact_gap)
            assert pk.contact_engine()["engine"] == engine
            info, arr = pk.node_network()
            info.pop("device_ms")
            pk.network()
            got.append((c, pk.contact_gap64(c.n), pk.contact_area(c.n), info, arr))
    (a, ga, sa, ia, na), (b, gb, sb, ib, nb) = got
    for x, y in ((a.row_ptr, b.row_ptr), (a.col, b.col), (a.image, b.image), (ga.view(np.uint64), gb.view(np.uint64)),
                 (sa.view(np.uint64), sb.view(np.uint64))):
        np.testing.assert_array_equal(x, y)
    assert ia == ib
    for k in na:
        np.testing.assert_array_equal(na[k], nb[k])
