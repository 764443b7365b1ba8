"""The coarse -> refined transfers (vxr, vyr, vzr, tempr) at the edges of their
layout: rows per lane (4 or 2 in FP32, 2 in FP64), wavefronts per row, odd
lines, walks of fewer and more than the 64 steps whose stencils a wavefront
holds, walks cut between wavefronts and whole ones, refinement ratios 2, other
ones above one, one, and below one; base rows longer than refined ones; whole
arrays, so that the unused index after an upload and the wall faces count.

Against the FP64 oracle.  A value is a sum of n <= max(nxmr, nymr, nzmr) terms,
each a gradient (a difference of values up to 0.5, so of the size of the
result's steps) through three stencils (absolute weights up to 1.3 each):
n + 16 roundings of at most 8 units of the result's max norm.
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state, relerr, uniform
from test_gpu_phase import PF, pf_state

pytestmark = pytest.mark.gpu

# (base), (refined)
SIZES = [((s, 4, 6), (2 * s, 8, 12)) for s in (3, 31, 32, 33, 63, 64, 65, 95, 96, 127, 128, 129, 255, 256, 257, 384, 512)]
SIZES += [((20, 6, 9), (61, 13, 20)), ((24, 12, 6), (30, 18, 15)), ((16, 6, 8), (40, 18, 8)), ((8, 2, 144), (16, 4, 288)), ((8, 144, 2), (16, 289, 4)),
          ((256, 2, 288), (512, 4, 576)), ((256, 288, 2), (512, 576, 4)), ((384, 4, 128), (769, 8, 256))]
# ratios that set-up takes in the mixed form only
FLAT = [((16, 8, 9), (32, 8, 8)), ((80, 8, 12), (84, 16, 24)), ((90, 8, 12), (70, 20, 30)), ((130, 6, 6), (120, 12, 12))]
CASES = [(b, f, p) for b, f in SIZES for p in ("fp64", "mixed")] + [(b, f, "mixed") for b, f in FLAT]


@pytest.mark.parametrize("base,fine,form", CASES, ids=lambda s: s if isinstance(s, str) else "x".join(map(str, s)))
def test_transfers_match_the_oracle(base, fine, form):
    n = max(fine)
    tol = 8 * (n + 16) * 2.0 ** (-53 if form == "fp64" else -24)
    for kind, call, names in (("sal", "interp_vel_mgrd", ("vxr", "vyr", "vzr")), ("phi", "interp_temp_multigrid", ("tempr",))):
        cfg = dict(nxm=base[0], nym=base[1], nzm=base[2], istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1,
                   nxmr=fine[0], nymr=fine[1], nzmr=fine[2])
        cfg.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else
                   dict(phasefield=1, pf_a=PF["pf_a"], pf_s=PF["pf_s"], pf_tm=PF["pf_tm"], pf_eps=0.1))
        st = random_state(cfg, 7) if kind == "sal" else pf_state(cfg, 7)
        for f in names:
            st[f] = np.ones((fine[2], fine[1], fine[0] + 1))
        o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
        load_state(o, st, upload=False)
        load_state(g, st, upload=True)
        o.call(call)
        g.call(call)
        for f in names:
            e = relerr(g.download(f), o.field(f))
            assert e <= tol, (f, e, tol)
        o.close()
        g.close()


def test_upload_between_graph_replays():
    """An upload of vyr after the capture: the next replay clears its unused index again."""
    cfg = dict(nxm=16, nym=6, nzm=6, istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1, nxmr=32, nymr=12, nzmr=12, salinity=1, rays=-2e6, pras=4.0)
    st = random_state(cfg, 3)
    got = []
    for graph in (False, True):
        g = pyafid.Solver(cfg)
        load_state(g, st, upload=True)
        for _ in range(3):
            g.upload("vyr", np.ones((12, 12, 33)))
            g.time_marcher_graph(1e-3, 2) if graph else [g.time_marcher(1e-3) for _ in range(2)]
            got.append(g.download("vyr"))
        g.close()
    for a, b in zip(got[:3], got[3:]):
        assert np.array_equal(a, b) and not np.any(b[..., 32])


# refined -> coarse: wavefronts per row, rows that the coarse ones outnumber,
# pairs of lines and single ones, ranges of z, grids that bracket and that do not
DOWN = [((s, 4, 6), (2 * s, 8, 12), {}) for s in (2, 3, 4, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 255, 256, 257, 384, 512)]
DOWN += [((8, 2, 288), (16, 4, 576), {}), ((16, 9, 2), (32, 18, 4), {}), ((32, 64, 48), (64, 128, 96), {}), ((128, 192, 4), (256, 384, 8), {}),
         ((20, 6, 9), (61, 13, 20), {}), ((24, 12, 6), (30, 18, 15), {}), ((24, 6, 6), (40, 12, 12), dict(istr3r=0)),
         ((60, 3, 4), (120, 6, 8), dict(sfixs=0)), ((60, 3, 4), (120, 6, 8), dict(sfixn=0))]
DOWN_FLAT = [((200, 4, 6), (256, 8, 12), {}), ((300, 4, 4), (330, 12, 12), dict(sfixs=0, sfixn=0))]      # mixed form only
DOWN = [d + (p,) for d in DOWN for p in ("fp64", "mixed")] + [d + ("mixed",) for d in DOWN_FLAT]


@pytest.mark.parametrize("base,fine,more,form", DOWN, ids=lambda s: s if isinstance(s, str) else "_".join(s) if isinstance(s, dict) else "x".join(map(str, s)))
def test_to_coarse_matches_the_oracle(base, fine, more, form):
    """Three stencils of 4 terms (absolute weights up to 1.3 each) of values
    rounded once: 32 units of the result's max norm."""
    tol = 32 * 2.0 ** (-53 if form == "fp64" else -24)
    for kind, call, name in (("sal", "interp_sal_multigrid", "salc"), ("phi", "interp_phi_multigrid", "phic"), ("phi", "add_latent_heat", "hro")):
        if form == "mixed" and call == "add_latent_heat":
            continue                                            # per-routine physics is FP64
        cfg = dict(nxm=base[0], nym=base[1], nzm=base[2], istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1,
                   nxmr=fine[0], nymr=fine[1], nzmr=fine[2])
        cfg.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else
                   dict(phasefield=1, pf_a=PF["pf_a"], pf_s=PF["pf_s"], pf_tm=PF["pf_tm"], pf_eps=0.1))
        cfg.update(more)
        st = random_state(cfg, 9) if kind == "sal" else pf_state(cfg, 9)
        if kind == "sal":
            st["salbp"] = uniform(91, (fine[2], fine[1], 1))
            st["saltp"] = uniform(92, (fine[2], fine[1], 1)) - 1.0
        if call == "add_latent_heat":
            st["rhsr"] = uniform(93, (fine[2], fine[1], fine[0] + 1)) - 0.5
            st["hro"] = uniform(94, (base[2], base[1], base[0] + 1))
            st["hro"][..., -1] = 0.0
        else:
            st[name] = np.ones((base[2], base[1], base[0] + 1))
        o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
        load_state(o, st, upload=False)
        load_state(g, st, upload=True)
        for s in (o, g):
            s.set_substep(1e-3, 1)
            s.call(call)
        n = base[0] if name == "hro" else base[0] + 1           # (hro(nx) is unused)
        e = relerr(g.download(name)[..., :n], o.field(name)[..., :n])
        assert e <= tol, (call, e, tol)
        o.close()
        g.close()
