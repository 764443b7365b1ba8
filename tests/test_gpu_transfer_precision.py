"""What the transfers of the mixed form (FP32 refined fields) round.

vyr / vzr: the sum along the line runs in FP64, so a mean flow does not lose a
little at every refined step.  A mean of 350 (|values| < 512 with the overshoot
of the stencils at the walls) with noise of 1e-3: the start of a line is common
to it, so its error, taken from that of the line's first point, holds the FP32
storage of the two points, half a unit of 2^-15 each, and that of n gradients
of 1e-3 (16 roundings each at most).
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state

pytestmark = pytest.mark.gpu

# walks cut between wavefronts and (1152 wavefronts) whole ones; ratios 2 and others
LINES = [((24, 144, 6), (48, 288, 12)), ((24, 6, 144), (48, 12, 288)), ((40, 96, 96), (70, 144, 162)), ((130, 32, 54), (260, 64, 108)),
         ((384, 24, 192), (768, 48, 384)), ((384, 192, 24), (768, 384, 48))]


@pytest.mark.parametrize("base,fine", LINES, ids=lambda s: "x".join(map(str, s)))
def test_sums_along_a_mean_flow(base, fine):
    cfg = dict(nxm=base[0], nym=base[1], nzm=base[2], istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1,
               nxmr=fine[0], nymr=fine[1], nzmr=fine[2], salinity=1, rays=-2e6, pras=4.0)
    st = random_state(cfg, 13)
    for f in ("vy", "vz"):
        st[f] = 350.0 + 2e-3 * st[f]
    o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED))
    load_state(o, st, upload=False)
    load_state(g, st, upload=True)
    for s in (o, g):
        s.call("interp_vel_mgrd")
    for f, axis in (("vyr", 1), ("vzr", 0)):
        n = fine[1] if f == "vyr" else fine[2]
        err = (g.download(f) - o.field(f))[..., :fine[0]]
        drift = np.abs(err - err.take([0], axis=axis)).max()
        tol = 2.0 ** -15 + n * 1e-3 * 16 * 2.0 ** -24
        assert drift <= tol, (f, drift, tol)
    o.close()
    g.close()
