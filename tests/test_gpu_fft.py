"""The transforms of the pressure solve for every number of stages and every
radix (16, 12, 9, 8, 6, 4, 3, 2), one line to sixteen a workgroup, rows that
end inside a workgroup's lines, odd rows (half a pair of real lines), lines
that one stage transforms and lines whose workgroup needs 1024 threads.

FP64: the pressure correction from a given divergence against the oracle,
1e-11 of its max norm (round-off of transforms and tridiagonal solves, as the
whole-step tests).  Mixed form: one step, relative L2 difference of the
velocity from the oracle's at most 1e-5.
"""
import numpy as np
import pytest

import pyafid
import pyoracle
from helpers import load_state, random_state, relerr, uniform

pytestmark = pytest.mark.gpu

LINES = [1, 2, 3, 4, 6, 8, 9, 12, 16, 18, 24, 27, 32, 36, 48, 54, 64, 72, 81, 96, 108, 128, 144, 162, 192, 216, 243, 256, 288, 324, 384, 432,
         486, 512, 576, 648, 768, 864, 972, 1024, 1152, 1296, 1458, 1536, 2048, 2187, 3456, 4096]      # (the oracle ends at 4096)
SIZES = [(5 + (3 * q) % 17, n, 3) for q, n in enumerate(LINES)] + [(5 + (5 * q) % 19, 4, n) for q, n in enumerate(LINES)]


def _cfg(size):
    nx, ny, nz = size
    return dict(nxm=nx, nym=ny, nzm=nz, istr3=8, rayt=1e5, prat=1.0, ylen=max(0.5, ny / 16.0), zlen=max(0.5, nz / 16.0))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_pressure_solve(size):
    cfg = _cfg(size)
    nx, ny, nz = size
    d = uniform(71, (nz, ny, nx + 1)) - 0.5
    d[..., nx] = 0.0
    o, g = pyoracle.Oracle(cfg), pyafid.Solver(cfg)
    o.field("dph")[...] = d
    g.upload("dph", d)
    for s in (o, g):
        s.set_substep(1e-3, 1)
        s.call("solve_pressure_correction")
    assert relerr(g.download("dph")[..., :nx], o.field("dph")[..., :nx]) <= 1e-11
    o.close()
    g.close()


@pytest.mark.parametrize("size", [s for s in SIZES if s[1] > 1 and s[2] > 1 and max(s) <= 1152 or max(s) == 2187], ids=lambda s: "x".join(map(str, s)))
def test_mixed_step(size):
    cfg = _cfg(size)
    st = random_state(cfg, 17)
    o, g = pyoracle.Oracle(cfg), pyafid.Solver(dict(cfg, precision=pyafid.MIXED))
    load_state(o, st, upload=False)
    load_state(g, st, upload=True)
    for s in (o, g):
        s.time_marcher(1e-3)
    for f in ("vx", "vy", "vz"):
        a, b = g.download(f), o.field(f)
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), f
    o.close()
    g.close()
