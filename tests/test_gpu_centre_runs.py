"""Centre distances over runs of cells against the oracle, bit for bit: places
on a lattice (distances on bin edges, coinciding centres), distances beyond the
box, one bin and the most bins, the smallest packings, an uneven one."""
import numpy as np
import pytest

import nanofiller_amd as nf
import oracle

pytestmark = pytest.mark.gpu


def _lattice(n, box, step, seed):
    g = np.random.default_rng(seed)
    return np.stack([g.integers(0, int(b / step), n) * step for b in box], 1)


def _uniform(n, box, seed, f=1.0):
    return np.random.default_rng(seed).uniform(0, 1, (n, 3)) * np.asarray(box) * f * 0.999999


CASES = {  # box, centres, bins, width
    "no rods near": ((4.0, 4.0, 4.0), np.array([[0.1, 0.1, 0.1], [2.0, 2.0, 2.0]]), 8, 0.01),
    "one rod": ((1.0, 1.0, 1.0), np.array([[0.1, 0.9, 0.5]]), 16, 0.25),
    "two rods, many images": ((1.0, 1.5, 2.0), np.array([[0.1, 0.9, 0.5], [0.9, 0.1, 1.9]]), 64, 0.125),
    "lattice, distances on edges": ((2.0, 3.0, 2.0), _lattice(900, (2, 3, 2), 0.125, 1), 8, 0.125),
    "half steps": ((2.0, 2.0, 2.0), _lattice(500, (2, 2, 2), 2.0**-10, 2), 1024, 2.0**-10),
    "one bin": ((3.0, 3.0, 3.0), _uniform(2000, (3, 3, 3), 3), 1, 0.37),
    "beyond the box": ((1.0, 1.0, 1.0), _uniform(300, (1, 1, 1), 4), 30, 0.1),
    "flat box": ((8.0, 0.5, 4.0), _uniform(1500, (8, 0.5, 4), 5), 50, 0.01),
    "a wide box": ((5000.0, 5000.0, 5000.0), _uniform(4000, (5000, 5000, 5000), 6), 100, 9.0),
    "most in a corner": ((6.0, 6.0, 6.0), np.concatenate([_uniform(1500, (6, 6, 6), 7, 0.08),
                                                          _uniform(500, (6, 6, 6), 8)]), 20, 0.05),
    "a row of cells around the box": ((1.0, 9.0, 9.0), _uniform(3000, (1, 9, 9), 9), 12, 0.1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_same_as_the_oracle(name):
    box, xyz, bins, width = CASES[name]
    rods = np.zeros((len(xyz), 8), np.float32)
    rods[:, :3] = xyz
    rods[:, 5] = 1.0
    rods[:, 6] = max(box) / 50
    rods[:, 7] = 0.001
    p = nf.normalize(nf.default_params(box=box, n_rods=len(rods), len=max(box) / 50, radius=0.001))
    o = oracle.centre_distance(p, rods, bins, width)
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        for _ in range(2):
            g = pk.centre_distance(bins, width)
            np.testing.assert_array_equal(g["counts"], o["counts"])
            assert (g["pairs"], g["sum_d_q24"], g["sum_d2_q16"]) == (o["pairs"], o["sum_d_q24"], o["sum_d2_q16"])
