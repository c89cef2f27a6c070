"""A staging slot that holds no rod never passes the cell-pair engine's filter,
whatever its memory holds; a slot with the probe's own rod always does."""
import ctypes as C
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libnf_line.so")

BITS = {"NaN": 0x7FC00000, "negative NaN": 0xFFFFFFFF, "infinity": 0x7F800000, "minus infinity": 0xFF800000,
        "largest": 0x7F7FFFFF, "minus largest": 0xFF7FFFFF, "denormal": 0x00000001, "zero": 0, "one": 0x3F800000}


def _apart(probe, slot, valid):
    if not os.path.exists(LIB):
        pytest.skip("line harness not built (run __graft_entry__.build())")
    L = C.CDLL(LIB)
    L.nfh_slot_apart.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_float, C.c_float, C.c_float, C.c_void_p]
    out = np.zeros(2, np.float32)
    L.nfh_slot_apart(probe.ctypes.data, slot.ctypes.data, valid, 0.01, 2e-7, 3.0, out.ctypes.data)
    return out


@pytest.mark.parametrize("name", list(BITS))
def test_empty_slots_stay_out(name):
    g = np.random.default_rng(1)
    for k in range(200):
        u = g.normal(size=3)
        probe = np.r_[g.uniform(-0.5, 0.5, 3), u / np.linalg.norm(u), 1.0, 0.005].astype(np.float32)
        slot = probe.copy()
        slot[g.uniform(size=8) < (1.0 if k == 0 else 0.5)] = np.uint32(BITS[name]).view(np.float32)
        # the engine reads the sign bit alone
        assert not np.any(np.signbit(_apart(probe, slot, 0))), (name, slot)


def test_a_rod_meets_itself():
    probe = np.array([0.3, -0.2, 0.1, 0.6, 0.0, 0.8, 1.0, 0.005], np.float32)
    assert np.all(np.signbit(_apart(probe, probe.copy(), 1)))
