"""Short results to the host: whole at the sizes where the way of the copy
changes, and one short array as quick as the runtime's own copy of it."""
import ctypes as C
import time

import numpy as np
import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu


def _v(a):
    return None if a is None else a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 16383, 16384, 16385, 65536, 196607, 196608, 196609])
def test_arrays_arrive_whole(n):
    edge = max((n / 100.0) ** (1.0 / 3.0), 1.0)
    p = nf.normalize(nf.default_params(box=(edge,) * 3, n_rods=n, len=0.4, radius=0.005, seed=3, contact_gap=0.02,
                                       tunnel_lambda=0.01))
    L = nf.lib()
    with nf.Packing(p) as pk:
        pk.generate()
        pk.contacts(0.02)
        info, net = pk.network()
        m = info["nnz"]
        for _ in range(2):
            labels, col, val = np.full(n, 7, np.uint32), np.full(m, 7, np.uint32), np.full(m, 7.0)
            for args in ((labels, None, None, None), (None, None, col, None), (None, None, None, val)):
                assert L.nf_get_network(pk._h, *[_v(a) for a in args], C.c_uint64(m)) == nf.NF_OK
            for a, k in ((labels, "labels"), (col, "col"), (val, "val")):
                np.testing.assert_array_equal(a, net[k])
            a, b = np.full(n, 7, np.uint32), np.full(m, 7, np.uint32)
            assert L.nf_get_network(pk._h, _v(a), None, _v(b), None, C.c_uint64(m)) == nf.NF_OK
            np.testing.assert_array_equal(a, net["labels"])
            np.testing.assert_array_equal(b, net["col"])


def test_results_queued_behind_kernels():
    """Reduction and statistics read a few words in the middle of their work."""
    p = nf.normalize(nf.default_params(box=(3.0,) * 3, n_rods=3000, len=1.0, radius=0.005, seed=7, contact_gap=0.01))
    with nf.Packing(p) as pk:
        pk.generate()
        rods = pk.rods()
        first = None
        for _ in range(5):
            pk.set_rods(rods)
            pk.contacts(0.01)
            got = (pk.histograms(bins=8)["centre"].tolist(), pk.centre_distance(4, 0.1)["counts"].tolist(),
                   pk.reduce(2)[1].tolist())
            first = first or got
            assert got == first


def test_a_short_read_takes_no_longer_than_a_copy():
    p = nf.normalize(nf.default_params(box=(3.0,) * 3, n_rods=40000, len=0.1, radius=0.002, seed=7, contact_gap=0.002))
    hip = C.CDLL("libamdhip64.so.7")
    L = nf.lib()
    d = C.c_void_p()
    assert hip.hipMalloc(C.byref(d), C.c_size_t(1 << 20)) == 0

    def median(f):
        ts = []
        for _ in range(300):
            t0 = time.perf_counter()
            f()
            ts.append(time.perf_counter() - t0)
        return sorted(ts)[150] * 1e6

    with nf.Packing(p) as pk:
        pk.generate()
        pk.contacts(0.002)
        pk.network()
        for n in (100, 40000):
            out = np.zeros(40000, np.uint32)
            if n == 100:
                b = np.zeros(pk.contacts(0.0005).n)
                assert 0 < len(b) <= 2000
                read = lambda: L.nf_get_contact_gap64(pk._h, _v(b), C.c_uint64(len(b)))  # noqa: E731
                size = 8 * len(b)
            else:
                pk.network()
                read = lambda: L.nf_get_network(pk._h, _v(out), None, None, None, C.c_uint64(0))  # noqa: E731
                size = 4 * n
            own = median(read)
            raw = median(lambda: hip.hipMemcpy(_v(out), d, C.c_size_t(size), 2))
            assert own < 1.5 * raw, (size, own, raw)
    hip.hipFree(d)
