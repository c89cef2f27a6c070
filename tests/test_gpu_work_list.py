"""The work list of the generation passes: packings whose cells are dealt over
many items, hold more than one chunk of probes, or mostly none, against the
oracle bit for bit."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu

GRIDS = {
    # box, rods, rod length, cell edge
    "one cell, rods reach their images": (1.3, 250, 1.0, 5.0),
    "eight cells, several chunks each": (2.4, 1500, 1.0, 1.1),
    "one rod per cell and empty cells": (4.0, 1200, 0.8, 0.25),
    "a single rod": (2.0, 1, 1.0, 0.0),
}


@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("options", [{}, {nf.NF_OPT_TEST_ALL_PAIRS: 1},
                                     {nf.NF_OPT_PART_SHIFT: 3, nf.NF_OPT_SPLIT_MIN: 8}])
def test_packing_does_not_depend_on_the_split(grid, prec, options):
    box, n, length, cell = GRIDS[grid]
    p = nf.normalize(nf.default_params(box=(box,) * 3, n_rods=n, len=length, radius=0.005, seed=5, cell_size=cell,
                                       precision=prec, max_rounds=12))
    ro, so, _ = oracle.generate(p, threads=4)
    with nf.Packing(p, options=options) as pk:
        st = pk.generate()[0]
        rods = pk.rods()
    assert (st.n_accepted, st.rounds, st.proposals) == (so["n_accepted"], so["rounds"], so["proposals"])
    np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))
    if nf.NF_OPT_TEST_ALL_PAIRS in options:
        assert st.pair_tests == so["pair_tests"]


def test_batch_of_uneven_packings():
    """Instances that end at different rounds, one of them past jamming."""
    ps = [nf.normalize(nf.default_params(box=(b,) * 3, n_rods=n, len=1.0, radius=0.005, seed=9, stream=i, max_rounds=r))
          for i, (b, n, r) in enumerate([(2.5, 1500, 8), (3.0, 40, 8), (1.6, 1500, 6), (4.0, 900, 8)])]
    with nf.Packing(ps) as pk:
        st = pk.generate()
        got = [pk.rods(i) for i in range(len(ps))]
    for p, s, rods in zip(ps, st, got):
        ro, so, _ = oracle.generate(p, threads=4)
        assert (s.n_accepted, s.rounds) == (so["n_accepted"], so["rounds"])
        np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))
