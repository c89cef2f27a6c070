"""The cell-pair engine with its line filter (NF_OPT_CROSSING_LISTS off): the
packings of the line filter's and the work list's tests, which have crossing
lists by default, against the oracle; larger ones against the lists and against
every pair within reach."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle
from tests.test_gpu_line_filter import PACKINGS
from tests.test_gpu_work_list import GRIDS

pytestmark = pytest.mark.gpu

CELLS = {nf.NF_OPT_CROSSING_LISTS: 0}
SPLIT = {nf.NF_OPT_CROSSING_LISTS: 0, nf.NF_OPT_PART_SHIFT: 3, nf.NF_OPT_SPLIT_MIN: 8}
COUNTERS = ("n_accepted", "rounds", "status", "candidates", "proposals", "rejected_old", "rejected_new")
PRECISIONS = [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK]


def _run(p, options):
    with nf.Packing(p, options) as pk:
        st = pk.generate()[0]
        return st, pk.rods()


def _same_as_oracle(p, options):
    ro, so, _ = oracle.generate(p, threads=4)
    st, rods = _run(p, options)
    for k in ("n_accepted", "rounds", "proposals", "rejected_old", "rejected_new"):
        assert getattr(st, k) == so[k], k
    np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))
    return st


@pytest.mark.parametrize("prec", PRECISIONS)
@pytest.mark.parametrize("options", [CELLS, SPLIT], ids=["by cost", "own split"])
@pytest.mark.parametrize("name", list(PACKINGS))
def test_line_filter(name, options, prec):
    st = _same_as_oracle(nf.normalize(nf.default_params(seed=21, precision=prec, max_rounds=10, **PACKINGS[name])), options)
    assert st.rejected_old + st.rejected_new > 0


@pytest.mark.parametrize("prec", PRECISIONS)
@pytest.mark.parametrize("options", [CELLS, SPLIT], ids=["by cost", "own split"])
@pytest.mark.parametrize("name", list(GRIDS))
def test_work_list(name, options, prec):
    box, n, length, cell = GRIDS[name]
    _same_as_oracle(nf.normalize(nf.default_params(box=(box,) * 3, n_rods=n, len=length, radius=0.005, seed=5,
                                                   cell_size=cell, precision=prec, max_rounds=12)), options)


LOGN = dict(len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.5, len_min=0.2, len_max=3.0)
# crowded, so that proposals are cut and dense cells dealt over several items
LARGE = {
    "40,000 rods past jamming": dict(box=(4.6,) * 3, n_rods=40000, len=1.0, max_rounds=14),
    "40,000 mixed rods": dict(box=(7.0,) * 3, n_rods=40000, len=1.0, max_rounds=30, **LOGN),
    "60,000 aligned rods": dict(box=(6.0,) * 3, n_rods=60000, len=1.0, max_rounds=30, ort_law=nf.NF_ORT_VMF, kappa=1e4,
                                axis=(1, 1, 0)),
    "30,000 in agglomerates": dict(box=(7.0,) * 3, n_rods=30000, len=1.0, max_rounds=30, den_law=nf.NF_DEN_AGGLOM, n_agg=4,
                                   agg_sigma=0.8, agg_peak=4.0, **LOGN),
}


@pytest.mark.parametrize("prec", PRECISIONS)
@pytest.mark.parametrize("name", list(LARGE))
def test_same_packing_as_lists_and_every_pair(name, prec):
    p = nf.normalize(nf.default_params(radius=0.005, seed=31, precision=prec, **LARGE[name]))
    st, rods = _run(p, CELLS)
    assert st.rejected_old > 0 and st.rejected_new > 0
    for options in (None, {nf.NF_OPT_TEST_ALL_PAIRS: 1}):
        so, ro = _run(p, options)
        for k in COUNTERS:
            assert getattr(st, k) == getattr(so, k), k
        np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))


def test_batch_and_switching():
    """Uneven instances on the cell pairs, and one handle switched between its
    engines, eager and from the captured round."""
    ps = [nf.normalize(nf.default_params(box=(b,) * 3, n_rods=n, len=1.0, radius=0.005, seed=9, stream=i, max_rounds=r, **kw))
          for i, (b, n, r, kw) in enumerate([(2.5, 1500, 8, {}), (3.0, 40, 8, LOGN), (1.6, 1500, 6, {}), (4.0, 900, 8, LOGN)])]
    want = [oracle.generate(p, threads=4)[0] for p in ps]
    with nf.Packing(ps) as pk:
        for lists, graph in ((0, 0), (1, 0), (0, 1), (1, 1), (0, 1)):
            pk.set_option(nf.NF_OPT_GRAPH, graph)
            pk.set_option(nf.NF_OPT_CROSSING_LISTS, lists)
            for _ in range(2):
                pk.generate()
                for i, ro in enumerate(want):
                    np.testing.assert_array_equal(pk.rods(i).view(np.uint32), ro.view(np.uint32))
