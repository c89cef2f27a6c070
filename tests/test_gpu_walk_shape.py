"""The waves-per-CU options reach the passes over crossing lists: same packing
whatever they say, and a launch of one wave per CU takes its time."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("old,new", [(1, 1), (3, 16), (16, 5), (0, 2)])
def test_packing_does_not_depend_on_the_waves(old, new, prec):
    p = nf.normalize(nf.default_params(box=(2.4,) * 3, n_rods=1500, len=1.0, radius=0.005, seed=5, precision=prec,
                                       max_rounds=12))
    ro, so, _ = oracle.generate(p, threads=4)
    with nf.Packing(p, {nf.NF_OPT_WAVES_OLD: old, nf.NF_OPT_WAVES_NEW: new}) as pk:
        st = pk.generate()[0]
        rods = pk.rods()
    for k in ("n_accepted", "rounds", "proposals", "rejected_old", "rejected_new"):
        assert getattr(st, k) == so[k], k
    np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))


@pytest.mark.parametrize("option,stage", [(nf.NF_OPT_WAVES_OLD, "reject_old"), (nf.NF_OPT_WAVES_NEW, "reject_new")])
def test_waves_have_effect(option, stage):
    """One wave per CU hides none of the fetches' latency: several times slower
    than sixteen, of which half is asked."""
    p = nf.normalize(nf.default_params(box=(16.0,) * 3, n_rods=200000, len=1.0, radius=0.005, seed=5))
    ms = {}
    for waves in (16, 1):
        with nf.Packing(p, {nf.NF_OPT_PROFILE: 1, option: waves}) as pk:
            ms[waves] = min(pk.generate()[0].to_dict()["kern_ms"][stage] for _ in range(4))
    assert ms[1] > 1.5 * ms[16], ms
