"""Periodic sizes that the transforms do not take are refused at set-up, those
whose factors would not fit a transform plan among them (3^15 has 15)."""
import pytest

import pyafid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("size,why", [(3 ** 15, "must factor into 2 and 3"), (10, "must factor into 2 and 3")])
@pytest.mark.parametrize("axis", ["nym", "nzm"])
def test_refused_sizes(axis, size, why, form):
    cfg = dict(nxm=2, nym=1, nzm=1, istr3=8, rayt=1e5, prat=1.0, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    with pytest.raises(pyafid.AfidError, match=why):
        pyafid.Solver(dict(cfg, **{axis: size}))
