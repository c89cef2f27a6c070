"""Contacts on both sides of the sizes and crowding from which they are found
over crossing lists: the same list by the default way, by home cells and by cell
pairs, of generated rods and of given ones unlike the parameters."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu

WAYS = ({}, {nf.NF_OPT_FOOTPRINT_FINE: 200}, {nf.NF_OPT_CONTACT_ENGINE: nf.NF_ENGINE_CELLS})
LOGN = dict(len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.3, len_min=0.3, len_max=3.0)


def _edge(n, crowd):
    return (n * 0.5 * np.pi * 0.01 * 1.04 / crowd) ** (1.0 / 3.0)


def _compare(p, rods, gap):
    got = []
    for options in WAYS:
        with nf.Packing(p, options) as pk:
            if rods is None:
                pk.generate()
            else:
                pk.set_rods(rods)
            c = pk.contacts(gap)
            got.append((c.row_ptr, c.col, c.image, pk.contact_gap64(c.n).view(np.uint64)))
    assert len(got[0][1]) > 100
    for other in got[1:]:
        for a, b in zip(got[0], other):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("n,crowd,law", [
    (30000, 1.0, "const"), (30001, 1.0, "const"), (60000, 0.7, "const"), (60000, 0.8, "const"), (100000, 2.4, "const"),
    (160000, 2.2, "const"), (160000, 2.4, "const"),
    (100000, 2.8, "const"), (210000, 0.4, "const"), (210000, 0.6, "const"), (100000, 0.9, "const"), (100000, 1.1, "const"),
    (60000, 0.3, "logn"), (61000, 0.3, "logn"), (100000, 0.44, "logn"), (140000, 0.5, "logn"),
    (160000, 0.5, "logn"), (160000, 1.0, "logn")])
def test_generated_rods(n, crowd, law, prec):
    _compare(nf.normalize(nf.default_params(box=(_edge(n, crowd),) * 3, n_rods=n, len=1.0, radius=0.005, seed=17,
                                            contact_gap=0.002, precision=prec, max_rounds=30,
                                            **(LOGN if law == "logn" else {}))), None, 0.002)


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("length", [0.1, 3.0, (0.05, 2.0)])
@pytest.mark.parametrize("law", ["const", "logn"])
def test_given_rods_unlike_the_parameters(law, length, prec):
    g = np.random.default_rng(5)
    n, box = 70000, (9.0, 8.0, 10.0)
    rods = np.zeros((n, 8), np.float32)
    rods[:, :3] = g.uniform(0, 1, (n, 3)) * np.asarray(box) * 0.999999
    u = g.normal(size=(n, 3))
    rods[:, 3:6] = u / np.linalg.norm(u, axis=1, keepdims=True)
    rods[:, 6] = length if np.isscalar(length) else g.uniform(*length, n)
    rods[:, 7] = 0.004
    p = nf.normalize(nf.default_params(box=box, n_rods=n, len=1.0, radius=0.005, contact_gap=0.001, precision=prec,
                                       **(LOGN if law == "logn" else {})))
    _compare(p, rods, 0.001)


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("n,crowd,peak,law", [(60000, 0.9, 8.0, "const"), (61000, 0.9, 8.0, "const"),
                                              (100000, 2.1, 8.0, "const"), (200000, 0.5, 20.0, "logn"),
                                              (60000, 0.9, 3.0, "const")])
def test_agglomerates(n, crowd, peak, law, prec):
    b = _edge(n, crowd)
    _compare(nf.normalize(nf.default_params(box=(b,) * 3, n_rods=n, len=1.0, radius=0.005, seed=19, contact_gap=0.002,
                                            precision=prec, max_rounds=30, den_law=nf.NF_DEN_AGGLOM, n_agg=16,
                                            agg_peak=peak, agg_sigma=b / 20, **(LOGN if law == "logn" else {}))),
             None, 0.002)
