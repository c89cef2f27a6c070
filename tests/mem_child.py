"""Runs one scenario of test_gpu_memory_limits.py with the allocators of
tests/native/mem_limit.cpp in front of the HIP runtime's, which have to be in
place before the library is loaded: in a process of its own."""
import ctypes as C
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(HERE))
M = C.CDLL(os.path.join(HERE, "native", "libnf_mem_limit.so"), mode=C.RTLD_GLOBAL)
M.nfm_live.restype = M.nfm_peak.restype = C.c_size_t
M.nfm_limit.argtypes = [C.c_size_t]
NO_LIMIT = C.c_size_t(-1).value
SLAB = 256 << 20  # the largest that blocks are cut from

import numpy as np  # noqa: E402

import nanofiller_amd as nf  # noqa: E402


def params(n, box, **kw):
    kw = dict(dict(len=1.0, radius=0.005, seed=3, contact_gap=0.004, max_rounds=40), **kw)
    return nf.normalize(nf.default_params(box=(box,) * 3, n_rods=n, **kw))


def flat(*arrays):
    return b"".join(np.ascontiguousarray(a).tobytes() for a in arrays)


def contacts(pk, gap=0.004):
    c = pk.contacts(gap)
    return flat(c.row_ptr, c.col, c.gap, c.image, pk.contact_gap64(c.n), pk.contact_area(c.n))


def everything(pk):
    out = [flat(pk.rods()) if pk.generate() else b"", contacts(pk)]
    h = pk.histograms(bins=16)
    out.append(flat(h["centre"], h["polar"], h["mutual"]))
    out.append(flat(pk.centre_distance(16, 0.02)["counts"]))
    net = pk.network()[1]
    out.append(flat(net["labels"], net["row_ptr"], net["col"], net["val"]))
    # (rounded differently from run to run: the order of the unknowns is not fixed)
    info, v = pk.conductance(tol=1e-12, max_iter=50000, potentials=True)
    assert info["converged"] == 1 and info["unknowns"] > 100
    out.append(flat(pk.reduce(2)[1]))
    return out, info["conductance"], v


def no_pinned_memory():
    p = params(3000, 2.5, tunnel_lambda=0.002)
    want = everything_of(p)
    M.nfm_pinned(0)
    got = everything_of(p)
    M.nfm_pinned(1)
    for k, (a, b) in enumerate(zip(got[0], want[0])):
        assert a == b, k
    assert abs(got[1] - want[1]) <= 1e-8 * want[1]
    np.testing.assert_allclose(got[2], want[2], rtol=0, atol=1e-8)


def everything_of(p):
    with nf.Packing(p) as pk:
        return everything(pk)


def create_at_the_limit():
    """A handle for which the crossing lists do not fit generates all the same."""
    p = params(20000, 5.0)
    with nf.Packing(p) as pk:
        pk.generate()
        want = flat(pk.rods())
        full = M.nfm_peak()
    for less in (1, full // 16, full // 8, full // 4):
        M.nfm_limit(full - less)
        with nf.Packing(p) as pk:
            M.nfm_limit(NO_LIMIT)
            pk.generate()
            assert flat(pk.rods()) == want, less


def contacts_at_the_limit():
    """A call that runs out of memory says so, one that has enough is right,
    and neither leaves anything behind for the next."""
    p = params(20000, 4.0)
    with nf.Packing(p) as pk:
        pk.generate()
        rods = pk.rods()
        base = M.nfm_live()
        want = contacts(pk)
        full = M.nfm_peak() - base
    fits = 0
    for part in range(16, -1, -1):
        with nf.Packing(p) as pk:
            pk.set_rods(rods)
            M.nfm_limit(M.nfm_live() + full * part // 16)
            try:
                assert contacts(pk) == want, part
                fits += 1
            except nf.NFError as e:
                assert e.code == nf.NF_E_NOMEM, (part, e)
            M.nfm_limit(NO_LIMIT)
            assert contacts(pk) == want, part
            pk.generate()
            assert flat(pk.rods()) == flat(rods), part
    assert 0 < fits


def another_instance():
    """What the calls on one instance held is there for the next one's; a slab
    that the handle's own blocks share stays."""
    ps = [params(2000000, 34.0, contact_gap=0.03), params(3000000, 40.0, stream=1)]
    with nf.Packing(ps) as pk:
        pk.generate()
        pk.select(1)
        want = contacts(pk)
        alone = M.nfm_peak()
    assert M.nfm_live() == 0
    with nf.Packing(ps) as pk:
        pk.generate()
        own = M.nfm_live()
        pk.contacts(0.03)
        pk.network()
        held = M.nfm_live() - own
        assert held > 3 * SLAB, held
        pk.select(1)
        M.nfm_limit(alone + SLAB)
        assert contacts(pk) == want
        M.nfm_limit(NO_LIMIT)
    assert M.nfm_live() == 0


def lists_make_room():
    """Crossing lists of the generation give way to a call that needs their
    memory; the next generation makes the same packing."""
    p = params(400000, 16.0, len_law=nf.NF_LEN_LOGNORMAL, len_sigma=0.3, len_min=0.3, len_max=3.0)
    engine = {nf.NF_OPT_CONTACT_ENGINE: nf.NF_ENGINE_CELLS}
    with nf.Packing(p, engine) as pk:
        pk.generate()
        rods = flat(pk.rods())
        want = contacts(pk)
    with nf.Packing(p, engine) as pk:
        pk.generate()
        M.nfm_limit(M.nfm_live() + (2 << 20))
        assert contacts(pk) == want
        pk.generate()
        assert flat(pk.rods()) == rods
        assert contacts(pk) == want
        M.nfm_limit(NO_LIMIT)
        pk.generate()
        assert flat(pk.rods()) == rods


def small_handles():
    """A small packing's handle takes a few allocations, not one per array, and
    gives them back."""
    M.nfm_calls.restype = C.c_long
    p = params(2000, 3.0)
    for _ in range(3):
        before = M.nfm_calls()
        with nf.Packing(p) as pk:
            assert M.nfm_calls() - before <= 10, M.nfm_calls() - before
            pk.generate()
            contacts(pk)
            pk.network()
            after = M.nfm_calls()
            for _ in range(3):
                pk.generate()
                contacts(pk)
                pk.network()
            assert M.nfm_calls() == after
        assert M.nfm_live() == 0


if __name__ == "__main__":
    print("[scenario]", sys.argv[1], flush=True)
    globals()[sys.argv[1]]()
    print("ok", flush=True)
