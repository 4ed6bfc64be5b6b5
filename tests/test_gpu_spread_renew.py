"""Spreading after atoms moved far without a list rebuild: the bins' room is
renewed, and the calls that follow spread as fast as with a fresh list."""
import numpy as np
import pytest

from thrid_amd import abi, systems

pytestmark = pytest.mark.gpu


def _spread(prec, sysd, build_at, pos):
    """Device time of the spreading per call at pos, and the last forces, with
    the list of the positions build_at."""
    from thrid_amd.pgk import ForceContext
    mts = abi.Mts(0, 0, 0, 0, 0, abi.MTS_LONG, 0)
    c = ForceContext(dict(sysd, pos=build_at), prec)
    c.mklist(sysd["rcut_book"])
    c.calforce(abi.MTS_LONG, mts)
    c.set_positions(pos)
    for _ in range(5):
        c.calforce(abi.MTS_LONG, mts)
    c.profile(1)
    for _ in range(20):
        f = c.calforce(abi.MTS_LONG, mts)["force"]
    ms, calls = c.profile(0)
    c.close()
    return ms[2] / calls[2], f   # stage 2: spreading


# squeezed to an eighth of the volume, nearly every atom is in a bin without
# room for it: three times the time as long as the starts stay.  Forces as in
# test_gpu_spread_bins: FP64 sums in another order, exact integers in mixed
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 0.0)])
def test_starts_are_renewed(prec, tol):
    s = systems.mixture_box(24000, "water", seed=3)
    pos = 0.5 * s["pos"]
    fresh, f0 = _spread(prec, s, pos, pos)
    moved, f1 = _spread(prec, s, s["pos"], pos)
    assert np.max(np.abs(f1 - f0)) <= tol * np.max(np.abs(f0))
    assert moved < 2.0 * fresh
