"""What the transfers of the mixed form (FP32 refined fields) round.

vyr / vzr: the sum along the line runs in FP64, so a mean flow does not lose a
little at every refined step.  A mean of 350 (|values| < 512 with the overshoot
of the stencils at the walls) with noise of 1e-3: the start of a line is common
to it, so its error, taken from that of the line's first point, holds the FP32
storage of the two points, half a unit of 2^-15 each, and that of n gradients
of 1e-3 (16 roundings each at most).

Refined -> coarse: weights and sums in FP64, so that of values that FP32 holds
phic (FP64) carries the 32 roundings of the FP64 form and salc (FP32) one more
of its own.  (At x ratio 2 phi takes another kernel, FP32 throughout.)
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state
from test_gpu_phase import pf_state

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


# refined x ratios of phi other than 2 and grids of S that do and do not bracket, odd sizes, pairs of lines and single ones
DOWN = [((96, 48, 54), (168, 96, 108)), ((96, 48, 54), (240, 72, 80)), ((24, 12, 6), (30, 18, 15)), ((20, 6, 9), (61, 13, 20)),
        ((200, 4, 6), (256, 8, 12)), ((300, 4, 4), (330, 12, 12)), ((33, 9, 8), (99, 27, 24))]


@pytest.mark.parametrize("base,fine", DOWN, ids=lambda s: "x".join(map(str, s)))
def test_to_coarse_rounds_once(base, fine):
    for kind, call, src, name in (("sal", "interp_sal_multigrid", "sal", "salc"), ("phi", "interp_phi_multigrid", "phi", "phic")):
        cfg = dict(nxm=base[0], nym=base[1], nzm=base[2], istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1,
                   nxmr=fine[0], nymr=fine[1], nzmr=fine[2])
        cfg.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else dict(phasefield=1, pf_eps=0.1))
        st = random_state(cfg, 17) if kind == "sal" else pf_state(cfg, 17)
        st[src] = st[src].astype(np.float32).astype(np.float64)
        o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED))
        load_state(o, st, upload=False)
        load_state(g, st, upload=True)
        for s in (o, g):
            s.call(call)
        n = base[0]
        a, b = g.download(name)[..., :n], o.field(name)[..., :n]
        tol = 32 * 2.0 ** -53 + (2.0 ** -24 if kind == "sal" else 0.0)
        assert np.abs(a - b).max() <= tol * np.abs(b).max(), name
        o.close()
        g.close()
