"""A run without salinity leaves `rays` and `pras` unused, whatever they hold:
zeros there make 1/Rrho infinite or undefined, and none of it may reach the
buoyancy of the base columns.

The run with the unused values against the same run with the defaults: the
arithmetic is the same, so the fields are the same to the last bit.
"""
import numpy as np
import pytest

import pyafid
from helpers import load_state, random_state

pytestmark = pytest.mark.gpu

FIELDS = ("vx", "vy", "vz", "temp", "pr", "rux", "ruy", "ruz", "rutemp")
UNUSED = [dict(pras=0.0), dict(rays=0.0), dict(rays=0.0, pras=0.0), dict(pras=0.0, active_s=1)]


def _fields(cfg, st):
    g = pyafid.Solver(cfg)
    load_state(g, st, upload=True)
    for _ in range(2):
        g.time_marcher(1e-3)
    out = {f: g.download(f) for f in FIELDS}
    g.close()
    return out


# nxm 40 and 130: two columns per wavefront and one; 520: above the register kernel's rows
@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("nxm", [40, 130, 520])
@pytest.mark.parametrize("gaxis", [1, 2, 3])
@pytest.mark.parametrize("unused", UNUSED, ids=lambda d: "_".join(f"{k}{v:g}" for k, v in d.items()))
def test_unused_salinity_parameters(unused, gaxis, nxm, form):
    cfg = dict(nxm=nxm, nym=6, nzm=4, istr3=8, rayt=1e6, prat=0.7, gaxis=gaxis, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    st = random_state(cfg, 5)
    ref, got = _fields(cfg, st), _fields(dict(cfg, **unused), st)
    for f in FIELDS:
        assert np.isfinite(ref[f]).all() and np.array_equal(got[f], ref[f]), f
