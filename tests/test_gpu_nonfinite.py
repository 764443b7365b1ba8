"""A transfer leaves finite what its stencils do not read: with one infinite
value in the source (as a run that blows up has it), the points of the result
that are not finite are those of the FP64 oracle's, near the walls, across the
periodic ends, and for pairs of lines whose sources differ and do not.
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state
from test_gpu_phase import pf_state

pytestmark = pytest.mark.gpu

SIZES = [((20, 12, 18), (40, 24, 36)), ((20, 12, 18), (30, 18, 27)), ((24, 12, 16), (60, 18, 40)), ((70, 8, 9), (140, 13, 18))]
CALLS = [("sal", "interp_vel_mgrd", ("vx", "vy", "vz"), ("vxr", "vyr", "vzr")), ("sal", "interp_sal_multigrid", ("sal",), ("salc",)),
         ("phi", "interp_temp_multigrid", ("temp",), ("tempr",)), ("phi", "interp_phi_multigrid", ("phi",), ("phic",))]


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,call,source,result", CALLS, ids=lambda v: v if isinstance(v, str) else "")
@pytest.mark.parametrize("base,fine", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_infinities_stay_where_they_are_read(base, fine, kind, call, source, result, form):
    cfg = dict(nxm=base[0], nym=base[1], nzm=base[2], istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1,
               nxmr=fine[0], nymr=fine[1], nzmr=fine[2])
    cfg.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else dict(phasefield=1, pf_eps=0.1))
    for at in ((5, 4, 3), (0, 0, 0), (-1, -1, -2), (7, 5, 2), (4, 3, 9), (3, 6, 12)):
        st = random_state(cfg, 4) if kind == "sal" else pf_state(cfg, 4)
        for f in source:
            st[f][at] = np.inf
        o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
        load_state(o, st, upload=False)
        load_state(g, st, upload=True)
        for s in (o, g):
            s.call(call)
        for f in result:
            assert np.array_equal(np.isfinite(g.download(f)), np.isfinite(o.field(f))), (f, at)
        o.close()
        g.close()
