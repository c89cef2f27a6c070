"""The generation passes over crossing lists: packings at the edges of what the
lists hold, against the oracle or against the cell-pair engine, which tests
every pair within reach under NF_OPT_TEST_ALL_PAIRS."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu

EXACT = {nf.NF_OPT_TEST_ALL_PAIRS: 1}
LOGN = dict(len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.3)


def _params(**kw):
    base = dict(radius=0.005, seed=31, max_rounds=12)
    base.update(kw)
    return nf.normalize(nf.default_params(**base))


def _same(p, options=None):
    """The default run and the exhaustive one: same packing, same counters."""
    with nf.Packing(p, EXACT) as pk:
        so = pk.generate()[0]
        ro = pk.rods()
    with nf.Packing(p, options) as pk:
        st = pk.generate()[0]
        rods = pk.rods()
        again = pk.generate()[0]
        rods2 = pk.rods()
    for s, r in ((st, rods), (again, rods2)):
        for k in ("n_accepted", "rounds", "status", "candidates", "proposals", "rejected_old", "rejected_new"):
            assert getattr(s, k) == getattr(so, k), k
        np.testing.assert_array_equal(r.view(np.uint32), ro.view(np.uint32))
    return st, again


SMALL = {
    "a rod spans the box": dict(box=(1.02, 1.02, 1.02), n_rods=120, len=2.0),
    "longer than the box: no lists": dict(box=(0.95, 0.95, 0.95), n_rods=60, len=2.0),
    "one fine cell across": dict(box=(1.2, 6.0, 3.0), n_rods=300, len=1.0),
    "one rod": dict(box=(2.0, 2.0, 2.0), n_rods=1, len=1.0),
    "many cells per rod": dict(box=(4.0, 4.0, 4.0), n_rods=2500, len=3.5, radius=0.002),
    "axis-parallel": dict(box=(3.0, 3.0, 3.0), n_rods=800, len=1.0, ort_law=nf.NF_ORT_VMF, kappa=1e7, axis=(0, 1, 0)),
    "mixed lengths past jamming": dict(box=(2.6, 2.6, 2.6), n_rods=1500, len=0.8, len_min=0.1, len_max=2.4, **LOGN),
    "wide rods": dict(box=(3.0, 3.0, 3.0), n_rods=300, len=0.5, radius=0.08),
}


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("name", list(SMALL))
def test_same_packing_as_the_oracle(name, prec):
    p = _params(precision=prec, **SMALL[name])
    ro, so, _ = oracle.generate(p, threads=4)
    with nf.Packing(p) as pk:
        st = pk.generate()[0]
        rods = pk.rods()
    assert (st.n_accepted, st.rounds) == (so["n_accepted"], so["rounds"])
    assert (st.rejected_old, st.rejected_new) == (so["rejected_old"], so["rejected_new"])
    np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))


# lanes per probe (8, 4, 2, 1) follow the round's proposals; constant lengths
# past the size rule take the cell-pair engine and its line filter
LARGE = {
    "20,000 rods": dict(box=(5, 5, 5), n_rods=20000, len=1.0),
    "90,000 rods": dict(box=(9, 9, 9), n_rods=90000, len=1.0),
    "250,000 rods": dict(box=(14, 14, 14), n_rods=250000, len=1.0),
    "600,000 mixed rods": dict(box=(24, 24, 24), n_rods=600000, len=1.0, len_min=0.3, len_max=3.0, **LOGN),
    "350,000 rods on cells": dict(box=(20, 20, 20), n_rods=350000, len=1.0),
    "120,000 dilute rods on cells": dict(box=(18, 18, 18), n_rods=120000, len=1.0),
}


@pytest.mark.parametrize("name", list(LARGE))
def test_same_packing_as_every_pair(name):
    _same(_params(max_rounds=1000, **LARGE[name]))


@pytest.mark.parametrize("scale", [20, 300])
def test_lists_that_overflow_grow(scale):
    """Lists (and cell slots) far shorter than planned overflow; the packing is
    generated again with twice the room and stays the same."""
    st, again = _same(_params(box=(3.0, 3.0, 3.0), n_rods=2500, len=1.0), {nf.NF_OPT_SLOT_SCALE: scale})
    assert st.slot_growths > 0 and again.slot_growths == 0


def test_batch_with_and_without_lists():
    ps = [_params(stream=i, **kw) for i, kw in enumerate(
        [SMALL["a rod spans the box"], SMALL["longer than the box: no lists"], SMALL["one rod"],
         SMALL["mixed lengths past jamming"], LARGE["20,000 rods"]])]
    with nf.Packing(ps, EXACT) as pk:
        so = pk.generate()
        ro = [pk.rods(i) for i in range(len(ps))]
    with nf.Packing(ps) as pk:
        st = pk.generate()
        for i in range(len(ps)):
            assert (st[i].n_accepted, st[i].rounds) == (so[i].n_accepted, so[i].rounds)
            assert (st[i].rejected_old, st[i].rejected_new) == (so[i].rejected_old, so[i].rejected_new)
            np.testing.assert_array_equal(pk.rods(i).view(np.uint32), ro[i].view(np.uint32))


def test_options_and_graph_keep_the_packing():
    """Switching the pair-test option between generations of one handle, and
    the captured round."""
    p = _params(box=(3.0, 3.0, 3.0), n_rods=2500, len=1.0)
    with nf.Packing(p) as pk:
        pk.generate()
        r0 = pk.rods()
        pk.set_option(nf.NF_OPT_TEST_ALL_PAIRS, 1)
        pk.generate()
        np.testing.assert_array_equal(pk.rods().view(np.uint32), r0.view(np.uint32))
        pk.set_option(nf.NF_OPT_TEST_ALL_PAIRS, 0)
        pk.set_option(nf.NF_OPT_GRAPH, 1)
        for _ in range(3):
            pk.generate()
            np.testing.assert_array_equal(pk.rods().view(np.uint32), r0.view(np.uint32))


def test_state_file_names_the_planned_grid(tmp_path):
    """The passes of a large packing of one length run on wider cells; the
    state file still names the grid of the default cell edge."""
    p = _params(**LARGE["350,000 rods on cells"])
    with nf.Packing(p) as pk:
        pk.generate()
        pk.save_state(str(tmp_path / "s.bin"))
    hd = nf.read_state_header(str(tmp_path / "s.bin"))
    reach = p.len * 1.000001 + 2.0 * p.radius
    assert hd["ext"] == (int(p.box[0] / (0.85 * reach)),) * 3
    assert hd["n_rods"] == 350000
