"""The refined column kernel (S and phi) at the edges of its layout: rows per
lane (4 in FP32, 2 in FP64), per group and groups per column, the smallest
and the largest column, odd y and z, more columns than the workgroups take in
one walk, fixed and zero-flux walls.  Two whole steps against the FP64 oracle:
1e-10 of each array's max norm in FP64 (as the other step tests); in the mixed
form the relative L2 difference of the field itself is at most 1e-5 (its
history is not compared there: it is a divided difference of vxr, whose FP32
storage alone moves it by up to 2e-5 where 766 cells cluster at the walls).
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state, relerr
from test_gpu_phase import PF, pf_state

pytestmark = pytest.mark.gpu

SIZES = [(6, 3, 2), (60, 4, 3), (62, 2, 2), (64, 6, 2), (66, 3, 4), (126, 4, 2), (128, 2, 3), (130, 4, 4), (190, 2, 3), (192, 3, 2),
         (194, 4, 2), (254, 2, 2), (256, 3, 4), (258, 2, 3), (382, 2, 3), (384, 2, 2), (386, 3, 2), (510, 2, 2), (512, 2, 3),
         (514, 2, 2), (766, 2, 3), (768, 2, 2), (770, 2, 3), (1022, 2, 2), (1024, 2, 2), (61, 4, 3), (10, 36, 32), (140, 24, 48)]


def _cfg(kind, size, **kw):
    n, ny, nz = size
    c = dict(nxm=max(2, (n + 1) // 2), nym=ny, nzm=nz, istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1, nxmr=n, nymr=2 * ny, nzmr=2 * nz)
    c.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else
             dict(phasefield=1, pf_a=PF["pf_a"], pf_s=PF["pf_s"], pf_tm=PF["pf_tm"], pf_eps=0.1))
    c.update(kw)
    return c


CASES = [_cfg(k, s) for k in ("sal", "phi") for s in SIZES]
CASES += [_cfg("sal", (70, 4, 6), sfixs=a, sfixn=b) for a, b in ((0, 1), (1, 0), (0, 0))]


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg", CASES, ids=lambda c: f"{'sal' if c.get('salinity') else 'phi'}_{c['nxmr']}x{c['nymr']}x{c['nzmr']}_{c.get('sfixs', 1)}{c.get('sfixn', 1)}")
def test_steps_match_the_oracle(cfg, form):
    sal = bool(cfg.get("salinity"))
    st = random_state(cfg, 31) if sal else pf_state(cfg, 31)
    objs = [pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))]
    for q, o in enumerate(objs):
        load_state(o, st, upload=q == 1)
        if sal:
            o.call("interp_vel_mgrd")
            o.call("interp_sal_multigrid")
        for _ in range(2):
            o.time_marcher(1e-3)
    n = cfg["nxmr"]
    for f in (("sal", "rusal") if sal else ("phi", "ruphi", "rhsr"))[:None if form == "fp64" else 1]:
        a, b = objs[1].download(f)[..., :n], objs[0].field(f)[..., :n]
        if form == "fp64":
            assert relerr(a, b) <= 1e-10, f
        else:
            assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), f
    for o in objs:
        o.close()
