"""The register form of the base column kernel (up to 512 wall-normal cells)
at the edges of its layout: rows per lane and group (64, 128, 192, 256, 384,
512 cells and their neighbours), odd and single y / z, more columns than the
workgroups take in one walk, every wall condition and buoyancy axis, active
salinity and moisture.  Whole steps against the FP64 oracle: 1e-10 of each
field's max norm in FP64 (as the other step tests); in the mixed form the
FP32 explicit terms bound the relative L2 difference by 1e-5.
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state, relerr

pytestmark = pytest.mark.gpu

FIELDS = ("vx", "vy", "vz", "temp", "pr", "rux", "ruy", "ruz", "rutemp")
CASES = [dict(nxm=n, nym=ny, nzm=nz, istr3=8, rayt=1e6, prat=0.7) for n, ny, nz in
         ((2, 4, 3), (31, 6, 4), (63, 3, 4), (64, 9, 4), (65, 6, 3), (127, 4, 2), (128, 18, 2), (129, 6, 4), (191, 3, 3),
          (192, 12, 2), (193, 4, 3), (255, 2, 4), (256, 6, 2), (257, 4, 2), (383, 4, 3), (384, 9, 2), (385, 4, 2), (511, 3, 2),
          (512, 2, 3), (40, 1, 16), (70, 1, 27), (16, 72, 64), (66, 54, 48), (130, 48, 96))]
CASES += [dict(nxm=72, nym=6, nzm=8, istr3=4, str3=1.3, rayt=1e5, prat=1.0, **kw) for kw in
          (dict(gaxis=2), dict(gaxis=3, inslws=0), dict(inslwn=0, tfixn=0, dpdy=0.3), dict(tfixs=0, xplusu=0.4, xminusu=-0.3),
           dict(moist=1), dict(nsst=1))]
CASES += [dict(nxm=66, nym=6, nzm=8, multires=1, nxmr=132, nymr=12, nzmr=16, salinity=1, istr3=8, istr3r=8, rayt=1e6,
               rays=-2e6, pras=4.0, active_s=1, gaxis=g) for g in (1, 2, 3)]


def _id(c):
    extra = "_".join(f"{k}{v}" for k, v in c.items() if k in ("gaxis", "inslws", "inslwn", "tfixs", "tfixn", "moist", "nsst"))
    return f"{c['nxm']}x{c['nym']}x{c['nzm']}_{extra}"


def _state(cfg):
    st = random_state(cfg, 21)
    if cfg.get("moist"):
        st["humid"] = np.abs(st["temp"]) * 0.3
        st["ruhumid"] = st["rutemp"] * 0.1
    return st


def _steps(obj, cfg, st, upload):
    load_state(obj, st, upload=upload)
    if cfg.get("salinity"):
        obj.call("interp_vel_mgrd")
        obj.call("interp_sal_multigrid")
    if cfg.get("moist"):
        obj.call("set_humidity_bcs")
        obj.call("update_saturation")
    for _ in range(2):
        obj.time_marcher(1e-3)


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg", CASES, ids=_id)
def test_steps_match_the_oracle(cfg, form):
    st = _state(cfg)
    o = pyoracle.Oracle(cfg)
    _steps(o, cfg, st, False)
    g = pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
    _steps(g, cfg, st, True)
    for f in FIELDS:
        a, b = g.download(f), o.field(f)
        n = cfg["nxm"]
        a, b = (a, b) if f in ("vx", "rux") else (a[..., :n], b[..., :n])
        if f == "pr":
            a, b = a - a.mean(), b - b.mean()
        if form == "fp64":
            assert relerr(a, b) <= 1e-10, f
        else:
            assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), f
    g.close()
    o.close()
