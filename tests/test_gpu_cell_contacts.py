"""Contacts by cell pairs: the same list as by footprints at the sizes where a
chunk's words of probes end, and no longer than the work takes where rods are
few: a pass over 200,000 spread-out rods against the floor of an almost empty
one, which is the waves' last additions to the counters."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu

CELLS = {nf.NF_OPT_CONTACT_ENGINE: nf.NF_ENGINE_CELLS}


def _params(n, crowd, **kw):
    edge = max((n * 0.5 * np.pi * 0.01 / crowd) ** (1.0 / 3.0), 2.1)
    return nf.normalize(nf.default_params(box=(edge,) * 3, n_rods=n, len=1.0, radius=0.005, seed=5, contact_gap=0.004, **kw))


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("per_cell", [1, 31, 32, 33, 63, 64, 65, 97, 130])
def test_chunks_of_probes(per_cell, prec):
    """27 cells of one reach that hold about so many rods each."""
    g = np.random.default_rng(per_cell)
    n, box = 27 * per_cell, 3.1
    rods = np.zeros((n, 8), np.float32)
    cell = np.stack(np.unravel_index(np.arange(27), (3, 3, 3)), 1)
    rods[:, :3] = (np.repeat(cell, per_cell, 0) + g.uniform(0.01, 0.99, (n, 3))) * (box / 3.0)
    u = g.normal(size=(n, 3))
    rods[:, 3:6] = u / np.linalg.norm(u, axis=1, keepdims=True)
    rods[:, 6], rods[:, 7] = 1.0, 0.005
    p = nf.normalize(nf.default_params(box=(box,) * 3, n_rods=n, len=1.0, radius=0.005, contact_gap=0.004, precision=prec))
    got = []
    for options in (CELLS, {nf.NF_OPT_FOOTPRINT_FINE: 200}):
        with nf.Packing(p, options) as pk:
            pk.set_rods(rods)
            c = pk.contacts(0.004)
            got.append((c.row_ptr, c.col, c.image, pk.contact_gap64(c.n).view(np.uint64)))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    assert per_cell < 30 or len(got[0][1]) > 0


def test_few_rods_take_little_time():
    ms = {}
    for n in (2000, 200000):
        with nf.Packing(_params(n, 0.1), CELLS) as pk:
            pk.generate()
            pk.contacts(0.002)
            t = []
            for _ in range(10):
                pk.contacts(0.002)
                t.append(pk.contact_stats()["kernel_ms"]["pairs"])
            ms[n] = sorted(t)[5]
    assert ms[200000] < 1.6 * ms[2000], ms
