"""A conductance solve whose numbers break down ends without a solution: a rod
between others whose couplings all underflow has no diagonal."""
import math

import numpy as np
import pytest

import nanofiller_amd as nf
from tests.test_cpu_network import _rod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lam,solvable", [(0.02, True), (1e-4, False)])
def test_couplings_that_underflow(lam, solvable):
    rods = np.stack([_rod((0.45, 0.5, 0.5), (1, 0, 0), 0.9, 0.01), _rod((1.5, 0.5, 0.5), (1, 0, 0), 0.9, 0.01),
                     _rod((2.55, 0.5, 0.5), (1, 0, 0), 0.9, 0.01)])
    p = nf.normalize(nf.default_params(box=(3.0, 1.0, 1.0), n_rods=3, len=0.9, radius=0.01, contact_gap=0.2, elec_axis=0,
                                       tunnel_lambda=lam, precision=nf.NF_PREC_FP64))
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        pk.contacts(p.contact_gap)
        info, _ = pk.network()
        assert info["percolating"] == 1
        ci, v = pk.conductance(tol=1e-10, max_iter=1000, potentials=True)
    assert ci["unknowns"] == 3
    if solvable:
        assert ci["converged"] == 1 and ci["residual"] <= 1e-10 and 0.0 < ci["conductance"] < 1.0
        assert np.all((v > 0.0) & (v < 1.0))
    else:
        assert ci["converged"] == 0 and math.isnan(ci["residual"])
