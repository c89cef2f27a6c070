"""Milestone dumps of a generation that runs out of room: a round whose lists
of survivors were too short is drawn again, so nothing of it may be saved."""
import os

import pytest

import nanofiller_amd as nf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [5, 20, 300])
def test_same_dumps_as_without_overflow(tmp_path, scale):
    p = nf.normalize(nf.default_params(box=(3.0, 3.0, 3.0), n_rods=2500, len=1.0, radius=0.01, seed=31, max_rounds=12))
    got = {}
    for name, options in (("planned", None), ("short", {nf.NF_OPT_SLOT_SCALE: scale})):
        d = tmp_path / name
        d.mkdir()
        with nf.Packing(p, options) as pk:
            pk.set_milestones([0.02, 0.5, 1.0, 1.5, 2.0, 2.5, 2.9], str(d))
            st = pk.generate()[0]
        if options:
            assert st.slot_growths > 0
        got[name] = {f: (d / f).read_bytes() for f in sorted(os.listdir(d))}
    assert got["planned"]
    assert list(got["short"]) == list(got["planned"])
    for f in got["planned"]:
        assert got["short"][f] == got["planned"][f], f
