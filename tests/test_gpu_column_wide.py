"""The register form of the base column kernel for fields of 4 GiB and more
(64-bit plane bases) and for smaller ones (32-bit offsets into whole fields):
the same arithmetic, so the same bits, on every layout of the kernel
(AFID_COLUMN_WIDE=1 selects the first on a small grid); and a grid whose fields
are really that large.
"""
import numpy as np
import pytest

import pyafid
from helpers import load_state, random_state, relerr
from test_gpu_column_reg import CASES, FIELDS, _id, _state, _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg", CASES, ids=_id)
def test_wide_form_is_the_same(cfg, form, monkeypatch):
    st, got = _state(cfg), []
    for wide in ("0", "1"):
        monkeypatch.setenv("AFID_COLUMN_WIDE", wide)
        g = pyafid.Solver(dict(cfg, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64))
        _steps(g, cfg, st, True)
        got.append({f: g.download(f) for f in FIELDS})
        g.close()
    for f in FIELDS:
        assert np.array_equal(got[0][f], got[1][f]), f


def test_fields_above_4_gib():
    """128 periods of a 500 x 144 x 64 run in z (4.8 GB a field): each period
    is that run, up to the round-off of the longer transform (1e-10 of each
    field's max norm, as the other step tests)."""
    n, reps = (500, 144, 64), 128
    cfg = dict(nxm=n[0], nym=n[1], nzm=n[2], istr3=8, rayt=1e6, prat=0.7, zlen=1.0)
    st = random_state(cfg, 31)
    st = {f: st[f] for f in ("vz", "temp", "tempbp")}
    small = pyafid.Solver(cfg)
    load_state(small, st, upload=True)
    small.time_marcher(1e-3)
    big = pyafid.Solver(dict(cfg, nzm=n[2] * reps, zlen=float(reps)))
    for f, a in st.items():
        print("upload", f, flush=True)
        big.upload(f, np.tile(a, (reps, 1, 1)))
    big.time_marcher(1e-3)
    for f in ("vx", "vy", "vz", "temp"):
        print("compare", f, flush=True)
        a, b = small.download(f), big.download(f)
        for t in (0, 1, 64, 113, 114, reps - 1):
            assert relerr(b[t * n[2]:(t + 1) * n[2], :, :n[0]], a[..., :n[0]]) <= 1e-10, (f, t)
        del b
    small.close()
    big.close()
