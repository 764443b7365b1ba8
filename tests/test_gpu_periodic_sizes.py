"""Periodic sizes that the transforms do not take are refused at set-up, those
whose factors would not fit a transform plan among them (3^15 has 15), and a
refusal, of a size or for memory, leaves nothing behind for the next set-up."""
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


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes", [dict(nym=2 ** 14), dict(nzm=2 ** 14), dict(nxm=1000, nym=8192, nzm=8192)],
                         ids=lambda d: "_".join(f"{k}{v}" for k, v in d.items()))
def test_next_set_up_after_a_refusal(sizes, form):
    """16384 is beyond one workgroup's transform; a field of 541 GB beyond the card."""
    cfg = dict(nxm=6, nym=4, nzm=4, istr3=8, rayt=1e5, prat=1.0, precision=pyafid.MIXED if form == "mixed" else pyafid.FP64)
    with pytest.raises(pyafid.AfidError):
        pyafid.Solver(dict(cfg, **sizes))
    g = pyafid.Solver(cfg)
    g.time_marcher(1e-3)
    g.close()
