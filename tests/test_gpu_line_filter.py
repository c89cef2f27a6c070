"""The line filter in front of the generation's pair tests drops no pair that
cuts: packings of nearly parallel, thick, very thin, long and mixed rods, in
small and large boxes, against the oracle bit for bit."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu

VMF = dict(ort_law=nf.NF_ORT_VMF, axis=(1, 2, 3))
PACKINGS = {
    "nearly parallel": dict(box=(2, 2, 2), n_rods=900, len=1.0, radius=0.01, kappa=1e6, **VMF),
    "aligned": dict(box=(2, 2, 2), n_rods=900, len=1.0, radius=0.01, kappa=50.0, **VMF),
    "thick": dict(box=(3, 3, 3), n_rods=300, len=1.0, radius=0.12),
    "short as wide": dict(box=(3, 3, 3), n_rods=600, len=0.05, radius=0.1),
    "very thin in a large box": dict(box=(60, 60, 60), n_rods=2500, len=16.0, radius=0.0005),
    "soft core and separation": dict(box=(2, 2, 2), n_rods=700, len=0.8, radius=0.01, soft_frac=0.6, sep=0.004),
    "mixed lengths": dict(box=(3, 3, 3), n_rods=1500, len=0.6, len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.8, len_min=0.02,
                          len_max=2.5, radius=0.006),
    "images": dict(box=(1.1, 1.4, 2.2), n_rods=150, len=1.0, radius=0.008),
}


@pytest.mark.parametrize("prec", [nf.NF_PREC_FP64, nf.NF_PREC_FP32_RECHECK])
@pytest.mark.parametrize("name", list(PACKINGS))
def test_same_packing_as_the_oracle(name, prec):
    p = nf.normalize(nf.default_params(seed=21, precision=prec, max_rounds=10, **PACKINGS[name]))
    ro, so, _ = oracle.generate(p, threads=4)
    with nf.Packing(p) as pk:
        st = pk.generate()[0]
        rods = pk.rods()
    assert (st.n_accepted, st.rounds) == (so["n_accepted"], so["rounds"])
    assert (st.rejected_old, st.rejected_new) == (so["rejected_old"], so["rejected_new"])
    assert st.rejected_old + st.rejected_new > 0
    np.testing.assert_array_equal(rods.view(np.uint32), ro.view(np.uint32))
