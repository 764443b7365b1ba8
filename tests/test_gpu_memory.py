"""Device memory of a two-grid context: the refined fields and the second buffer
of S or phi, and no scratch of the transfers beside them (at ratio 2 that would
be a quarter of a refined field; a sixteenth is left for tables)."""
import numpy as np
import pytest

import pyafid
from helpers import load_state, random_state
from test_gpu_column_reg import CASES, FIELDS, _id, _state, _steps
from test_gpu_phase import pf_state

pytestmark = pytest.mark.gpu


# refined arrays: S, its explicit terms, three velocities (FP64: two more for the per-routine calls) and the second buffer of S;
# phi, its explicit terms, T, d phi (FP64: one more) and the second buffer of phi.  base: FP64 and FP32 arrays of the base grid
# that the single-grid context does not have (phic, the latent heat; salc)
@pytest.mark.parametrize("kind,form,refined,base", [("sal", "fp64", 8, (0, 0)), ("sal", "mixed", 6, (0, 1)), ("phi", "fp64", 6, (1, 0)), ("phi", "mixed", 5, (2, 0))])
def test_two_grid_context(kind, form, refined, base):
    one = dict(nxm=96, nym=96, nzm=128, istr3=8, rayt=1e6, prat=1.0, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    two = dict(one, multires=1, nxmr=192, nymr=192, nzmr=256, istr3r=8)
    two.update(dict(salinity=1, rays=-2e6, pras=4.0) if kind == "sal" else dict(phasefield=1, pf_eps=0.1))
    size = []
    for cfg in (one, two):
        g = pyafid.Solver(cfg)
        size.append(g.device_bytes())
        g.close()
    field = (4 if form == "mixed" else 8) * 256 * 192 * (-(-193 // 16) * 16)
    nb = 128 * 96 * (-(-97 // 16) * 16)
    assert size[1] - size[0] <= refined * field + (8 * base[0] + 4 * base[1]) * nb + field // 16


@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_transfers_leave_the_scalar_alone(form):
    """A transfer between two steps (as a host that looks at vxr makes) changes nothing in the steps."""
    cfg = dict(nxm=20, nym=12, nzm=16, istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1, nxmr=40, nymr=24, nzmr=32, salinity=1,
               rays=-2e6, pras=4.0, active_s=1, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    st, got = random_state(cfg, 41), []
    for more in (False, True):
        g = pyafid.Solver(cfg)
        load_state(g, st, upload=True)
        for _ in range(3):
            if more:
                g.call("interp_vel_mgrd")
                g.call("interp_sal_multigrid")
                g.call("interp_vel_mgrd")
            else:
                g.call("interp_vel_mgrd")
                g.call("interp_sal_multigrid")
            g.time_marcher(1e-3)
        got.append({f: g.download(f) for f in ("vx", "vy", "vz", "temp", "sal", "rusal", "vxr", "salc")})
        g.close()
    for f in got[0]:
        assert np.array_equal(got[0][f], got[1][f]), f


@pytest.mark.parametrize("form,fields", [("fp64", 16), ("mixed", 10)])
def test_ensemble_rows(form, fields):
    """The rows of an ensemble member are whole 64 bytes, no more: 71 values take 72, 80 take 80, so that
    eight values a row and field lie between the two runs (16 or more fields in FP64, the 10 of the state
    and its second buffers at least in the mixed form)."""
    size = []
    for nxm in (70, 79):
        cfg = dict(nxm=nxm, nym=1, nzm=256, istr3=8, rayt=1e6, prat=1.0, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
        e = pyafid.Ensemble([cfg], [dict(dt=1e-3)])
        size.append(e.device_bytes())
        e.close()
    assert size[1] - size[0] >= fields * 8 * 256 * 8


TIGHT = {"one grid": dict(nxm=70, nym=18, nzm=24, istr3=8, rayt=1e6, prat=1.0),
         "salinity": dict(nxm=70, nym=18, nzm=24, istr3=8, rayt=1e6, prat=1.0, multires=1, nxmr=134, nymr=36, nzmr=48, istr3r=8,
                          salinity=1, rays=-2e6, pras=4.0, active_s=1),
         "phase field": dict(nxm=70, nym=18, nzm=24, istr3=8, rayt=1e6, prat=1.0, multires=1, nxmr=134, nymr=36, nzmr=48,
                             istr3r=8, phasefield=1, pf_eps=0.05, pf_r0=0.2),
         "ratio 2": dict(nxm=67, nym=18, nzm=24, istr3=8, rayt=1e6, prat=1.0, multires=1, nxmr=134, nymr=36, nzmr=48,
                         istr3r=8, phasefield=1, pf_eps=0.05, pf_r0=0.2)}


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("case", sorted(TIGHT))
def test_tight_rows(case, form, monkeypatch):
    """71 and 135 values: 80 and 144 padded to 128 bytes, 72 and 136 to 64, which set-up takes where the
    first do not fit (AFID_TIGHT_ROWS=1: at once).  The steps are the same."""
    cfg = dict(TIGHT[case], precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    names = ["vx", "vy", "vz", "temp", "pr"]
    names += ["sal", "vxr", "vyr", "salc"] if "salinity" in cfg else ["phi", "tempr", "phic"] if "phasefield" in cfg else []
    size, got = [], []
    for tight in ("0", "1"):
        monkeypatch.setenv("AFID_TIGHT_ROWS", tight)
        g = pyafid.Solver(cfg)
        size.append(g.device_bytes())
        g.upload("tempbp", np.ones((cfg["nzm"], cfg["nym"], 1)))
        g.create_initial_conditions(3, 0.05)
        for _ in range(2):
            g.time_marcher(1e-4)
        got.append({f: g.download(f) for f in names})
        g.close()
    assert size[1] < 0.98 * size[0]
    for f in names:
        assert np.array_equal(got[0][f], got[1][f]), f


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg", CASES, ids=_id)
def test_tight_rows_of_base_columns(cfg, form, monkeypatch):
    st, got = _state(cfg), []
    for tight in ("0", "1"):
        monkeypatch.setenv("AFID_TIGHT_ROWS", tight)
        g = pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
        _steps(g, cfg, st, True)
        got.append({f: g.download(f) for f in FIELDS})
        g.close()
    for f in FIELDS:
        assert np.array_equal(got[0][f], got[1][f]), f


# rows that 64 bytes hold with and without room to spare
@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("nxm,nxmr", [(3, 7), (5, 9), (15, 31), (32, 63), (33, 66), (63, 127), (64, 128), (100, 199), (127, 255), (130, 263), (380, 767)])
@pytest.mark.parametrize("kind", ["sal", "phi"])
def test_tight_rows_of_refined_fields(kind, nxm, nxmr, form, monkeypatch):
    cfg = dict(nxm=nxm, nym=4, nzm=6, istr3=8, istr3r=8, rayt=1e6, prat=1.0, multires=1, nxmr=nxmr, nymr=8, nzmr=12,
               precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    cfg.update(dict(salinity=1, rays=-2e6, pras=4.0, active_s=1) if kind == "sal" else dict(phasefield=1, pf_eps=0.1))
    st = random_state(cfg, 51) if kind == "sal" else pf_state(cfg, 51)
    names = ["vx", "temp", "sal", "rusal", "vxr", "vyr", "vzr", "salc"] if kind == "sal" else ["vx", "temp", "phi", "ruphi", "tempr", "phic"]
    got = []
    for tight in ("0", "1"):
        monkeypatch.setenv("AFID_TIGHT_ROWS", tight)
        g = pyafid.Solver(cfg)
        load_state(g, st, upload=True)
        for _ in range(2):
            g.time_marcher(1e-4)
        got.append({f: g.download(f) for f in names})
        g.close()
    for f in names:
        assert np.array_equal(got[0][f], got[1][f]), f
