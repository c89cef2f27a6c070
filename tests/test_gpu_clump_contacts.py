"""Rods in a clump, whose crossing lists are too short: the list pass is tried
once per set of rods and gap, and the contacts are right by whatever way."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import sys
sys.path.insert(0, {root!r})
import numpy as np
import nanofiller_amd as nf
import oracle

def say(what):
    sys.stderr.flush()
    print("[step]", what, file=sys.stderr, flush=True)

def rods(n, box, part, seed):
    g = np.random.default_rng(seed)
    r = np.zeros((n, 8), np.float32)
    r[:, :3] = g.uniform(0, 1, (n, 3)) * box * part
    u = g.normal(size=(n, 3))
    r[:, 3:6] = u / np.linalg.norm(u, axis=1, keepdims=True)
    r[:, 6], r[:, 7] = 0.5, 0.002
    return r

def check(pk, p, r, gap):
    o = oracle.contacts(p, r, gap, threads=4)
    c = pk.contacts(gap)
    np.testing.assert_array_equal(c.col, o["J"])
    np.testing.assert_array_equal(c.image, o["image"])
    np.testing.assert_array_equal(pk.contact_gap64(c.n).view(np.uint64), o["gap64"].view(np.uint64))

p = nf.normalize(nf.default_params(box=(4.0,) * 3, n_rods=2000, len=0.5, radius=0.002, contact_gap=0.001))
clump, even = rods(2000, 4.0, 0.15, 1), rods(2000, 4.0, 1.0, 2)
with nf.Packing(p) as pk:
    pk.set_rods(clump)
    for k, gap in (("first", 0.001), ("again", 0.001), ("wider", 0.002), ("narrower", 0.0005), ("wide again", 0.001)):
        say(k)
        check(pk, p, clump, gap)
    pk.set_rods(even)
    say("even")
    check(pk, p, even, 0.001)
    pk.set_rods(clump)
    say("clump")
    check(pk, p, clump, 0.001)
    pk.generate()
    say("generated")
    check(pk, p, pk.rods(), 0.001)
say("end")
"""


def test_lists_that_were_too_short_are_not_tried_again():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CHILD.format(root=root)], capture_output=True, text=True, timeout=100,
                       env={**os.environ, "NF_TRACE": "1"})
    assert r.returncode == 0, r.stdout + r.stderr
    tried, now = {}, None
    for line in r.stderr.splitlines():
        if line.startswith("[step]"):
            now = line[7:]
            tried[now] = 0
        elif "crossing-list pass launched" in line:
            tried[now] += 1
    assert tried == {"first": 1, "again": 0, "wider": 0, "narrower": 1, "wide again": 0, "even": 1, "clump": 1,
                     "generated": 1, "end": 0}, tried
