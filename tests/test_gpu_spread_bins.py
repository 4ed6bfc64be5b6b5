"""The spreading bins between list builds: atoms that leave their bin's room
(a configuration squeezed after the list was built) are spread all the same."""
import numpy as np
import pytest

from thrid_amd import abi, systems

pytestmark = pytest.mark.gpu


def _reciprocal(prec, sysd, pos, build_at):
    """The reciprocal part alone at pos, with the list (and the bins' room) of
    the positions build_at, or without a list."""
    from thrid_amd.pgk import ForceContext
    c = ForceContext(dict(sysd, pos=pos if build_at is None else build_at), prec)
    mts = abi.Mts(0, 0, 0, 0, 0, abi.MTS_LONG, 0)
    if build_at is not None:
        c.mklist(sysd["rcut_book"])
        c.calforce(abi.MTS_LONG, mts)
        c.set_positions(pos)
    out = [c.calforce(abi.MTS_LONG, mts) for _ in range(2)]
    c.close()
    return out


# squeeze 1: the same positions; 0.5, 0.15: 8 and 300 times the bins' slots in
# an eighth and a three-hundredth of the box; grids with 4- and 8-point tiles.
# Sums of up to 648 charges on a grid point in another order (FP64 rounding);
# exact integers in the mixed form
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 0.0)])
@pytest.mark.parametrize("nfft", [(24, 24, 24), (72, 72, 72)])
@pytest.mark.parametrize("squeeze", [1.0, 0.5, 0.15])
def test_spread_after_motion(prec, tol, nfft, squeeze):
    s = systems.water_box(nfft=nfft)
    pos = s["pos"] * squeeze
    fresh = _reciprocal(prec, s, pos, None)
    moved = _reciprocal(prec, s, pos, s["pos"])
    for a in moved:
        d = np.max(np.abs(a["force"] - fresh[0]["force"]))
        assert d <= tol * np.max(np.abs(fresh[0]["force"]))
    assert np.max(np.abs(fresh[1]["force"] - fresh[0]["force"])) <= \
        tol * np.max(np.abs(fresh[0]["force"]))
