"""Centre distances far below the rods' spacing, where the cells are widened for
more rods each: spread out, in clumps (cells for the rods as they lie, empty ones
left out), on both sides of the rule, against the oracle bit for bit."""
import time

import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu


def _centres(n, box, part, seed):
    """A part of the rods in a corner of a twentieth of the box, the others anywhere."""
    g = np.random.default_rng(seed)
    x = g.uniform(0, 1, (n, 3)) * np.asarray(box) * 0.999999
    k = int(n * part)
    x[:k] *= 0.05
    return x


CASES = {  # box, rods, part in the corner, bins, width
    "spread out": ((2.4, 2.4, 2.4), 4000, 0.0, 1, 0.05),
    "below the rule": ((2.4, 2.4, 2.4), 4000, 0.0, 8, 0.015),
    "at the rule": ((2.4, 2.4, 2.4), 1000, 0.0, 10, 0.0094),
    "few rods, many cells": ((9.0, 9.0, 9.0), 40, 0.5, 4, 0.02),
    "two rods": ((9.0, 9.0, 9.0), 2, 1.0, 4, 0.05),
    "flat": ((12.0, 0.4, 12.0), 3000, 0.0, 3, 0.02),
    "half in a corner": ((6.0, 6.0, 6.0), 3000, 0.5, 16, 0.005),
    "all in a corner": ((6.0, 6.0, 6.0), 2000, 1.0, 16, 0.005),
    "all in a corner, many bins": ((8.0, 8.0, 8.0), 2000, 1.0, 1000, 0.0002),
}


def _packing(box, xyz):
    rods = np.zeros((len(xyz), 8), np.float32)
    rods[:, :3] = xyz
    rods[:, 5] = 1.0
    rods[:, 6] = 0.3
    rods[:, 7] = 0.001
    return nf.normalize(nf.default_params(box=box, n_rods=len(rods), len=0.3, radius=0.001)), rods


@pytest.mark.parametrize("name", list(CASES))
def test_same_as_the_oracle(name):
    box, n, part, bins, width = CASES[name]
    p, rods = _packing(box, _centres(n, box, part, 11))
    o = oracle.centre_distance(p, rods, bins, width)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        for _ in range(2):
            g = pk.centre_distance(bins, width)
            np.testing.assert_array_equal(g["counts"], o["counts"])
            assert (g["pairs"], g["sum_d_q24"], g["sum_d2_q16"]) == (o["pairs"], o["sum_d_q24"], o["sum_d2_q16"])


def test_what_was_refused_still_is():
    p, rods = _packing((20.0, 20.0, 20.0), _centres(100, (20, 20, 20), 0.0, 1))
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        with pytest.raises(nf.NFError):
            pk.centre_distance(1, 0.04)


@pytest.mark.parametrize("part", [0.0, 1.0])
def test_small_distances_cost_no_more_than_large_ones(part):
    """A few hundred pairs out of 100,000 rods: less work than the millions
    within a tenth of the box, and no longer."""
    box = (15.0,) * 3
    p, rods = _packing(box, _centres(100000, box, part, 3))
    near, far = (0.05, 1.5) if part == 0.0 else (0.05, 0.2)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        t = {}
        for w in (near, far):
            pk.centre_distance(1, w)
            ts = []
            for _ in range(5):
                t0 = time.perf_counter()
                pk.centre_distance(1, w)
                ts.append(time.perf_counter() - t0)
            t[w] = min(ts)
    assert t[near] < t[far] + 2e-4, t
