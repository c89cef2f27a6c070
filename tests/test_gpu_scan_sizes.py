"""Row offsets (a prefix sum over the rods' contact counts) at the edges of the
scan: one workgroup, the first tiled size, whole and ragged tiles, the most
tiles whose sums each block adds up itself, and one more."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu

TILE = 2048


@pytest.mark.parametrize("n", [2, 16382, 16384, 16386, 9 * TILE - 2, 9 * TILE, 9 * TILE + 2, 300000,
                               2048 * TILE, 2048 * TILE + 2])
def test_row_offsets(n):
    sites = n // 2
    side = int(np.ceil(sites ** (1.0 / 3.0)))
    g = np.arange(sites)
    xyz = np.stack([g % side, (g // side) % side, g // (side * side)], 1) * 0.125 + 0.0625
    rods = np.zeros((n, 8), np.float32)
    rods[0::2, :3] = xyz
    rods[1::2, :3] = xyz
    rods[1::2, 0] += 0.015625
    rods[:, 5] = 1.0
    rods[:, 6] = 0.03125
    rods[:, 7] = 0.00390625
    edge = max(0.125 * side, 0.25)
    p = nf.normalize(nf.default_params(box=(edge,) * 3, n_rods=n, len=max(0.03125, edge / 128), radius=0.00390625))
    with nf.Packing(p) as pk:
        pk.set_rods(rods)
        c = pk.contacts(0.01)  # 1/64 apart, 1/128 between the surfaces: each pair and nothing else
    assert c.n == sites
    np.testing.assert_array_equal(c.row_ptr, ((np.arange(n + 1) + 1) // 2).astype(np.uint32))
    np.testing.assert_array_equal(c.col, 2 * np.arange(sites) + 1)
