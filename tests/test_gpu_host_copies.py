"""Rods to the device and back, bit for bit, at the sizes where the way of the
copy changes: what the small pinned block holds, one chunk, all chunks of the
large one, chunks that take a slot again, copies shared by threads."""
import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 100, 8191, 8192, 8193, 30000, 262143, 262144, 262145, 700001])
def test_round_trip(n):
    g = np.random.default_rng(n)
    box = (3.0, 4.0, 5.0)
    rods = np.empty((n, 8), np.float32)
    rods[:, :3] = g.uniform(0, 1, (n, 3)) * np.asarray(box) * 0.99999
    rods[:, 3:6] = g.normal(size=(n, 3))
    rods[:, 6] = g.uniform(1e-3, 2.0, n)
    rods[:, 7] = g.uniform(1e-4, 0.1, n)
    p = nf.normalize(nf.default_params(box=box, n_rods=max(n, 1), len=0.05, radius=0.001))
    with nf.Packing(p) as pk:
        for r in (rods, rods[::-1].copy(), rods[: n // 2]):
            pk.set_rods(r)
            for _ in range(2):
                np.testing.assert_array_equal(pk.rods().view(np.uint32), r.view(np.uint32))
        if n:
            bad = rods.copy()
            bad[n - 1, 0] = box[0]
            with pytest.raises(nf.NFError):
                pk.set_rods(bad)
            np.testing.assert_array_equal(pk.rods().view(np.uint32), rods[: n // 2].view(np.uint32))


@pytest.mark.parametrize("n,gap", [(1500, 0.002), (20000, 0.02), (60000, 0.08)])
def test_arrays_of_several_sizes_arrive_whole(n, gap):
    edge = (n / 300.0) ** (1.0 / 3.0)
    p = nf.normalize(nf.default_params(box=(edge,) * 3, n_rods=n, len=0.4, radius=0.005, seed=3, contact_gap=gap,
                                       tunnel_lambda=0.01))
    with nf.Packing(p) as pk:
        pk.generate()
        c = pk.contacts(gap)
        assert c.row_ptr[0] == 0 and c.row_ptr[-1] == c.n and np.all(np.diff(c.row_ptr.astype(np.int64)) >= 0)
        rows = np.repeat(np.arange(n), np.diff(c.row_ptr.astype(np.int64)))
        assert np.all(c.col > rows) and c.col.max() < n and np.all(c.gap <= gap)
        g64 = pk.contact_gap64(c.n)
        np.testing.assert_array_equal(g64.astype(np.float32), c.gap)
        info, net = pk.network()
        assert net["row_ptr"][-1] == info["nnz"] and net["col"].max() == n + 1
        sums = np.add.reduceat(net["val"], net["row_ptr"][:-1].astype(np.int64))[:n]
        diag = net["val"][net["col"] == np.repeat(np.arange(n + 2), np.diff(net["row_ptr"].astype(np.int64)))][:n]
        np.testing.assert_allclose(sums, 0.0, atol=1e-12 * np.abs(diag).max())


def test_two_threads_read_one_packing():
    from concurrent.futures import ThreadPoolExecutor

    p = nf.normalize(nf.default_params(box=(4.0, 4.0, 4.0), n_rods=30000, len=0.2, radius=0.003, seed=11,
                                       contact_gap=0.004))
    with nf.Packing(p) as pk:
        pk.generate()
        rods = pk.rods()
        c = pk.contacts(0.004)
        gaps = pk.contact_gap64(c.n)
        with ThreadPoolExecutor(2) as ex:
            jobs = [(ex.submit(pk.rods), ex.submit(pk.contact_gap64, c.n)) for _ in range(20)]
            for a, b in jobs:
                np.testing.assert_array_equal(a.result().view(np.uint32), rods.view(np.uint32))
                np.testing.assert_array_equal(b.result().view(np.uint64), gaps.view(np.uint64))
