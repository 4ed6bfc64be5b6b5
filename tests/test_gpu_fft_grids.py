"""SPME grids whose lines the batched FFT passes cut unevenly: odd lengths,
planes that end inside a block's rows, lines with the longest tables."""
import numpy as np
import pytest

from thrid_amd import abi
from helpers import water648, rms_rel, ene

pytestmark = pytest.mark.gpu

GRIDS = [(25, 27, 45), (36, 25, 50), (24, 45, 108), (27, 50, 288), (20, 20, 1024), (50, 32, 75)]


# FP64: rounding of two transforms of ~1e5 points; mixed: the FP32 form's
# accuracy against the oracle's FP64 (1e-4 is the form's own limit)
@pytest.mark.parametrize("prec,tol,etol", [("fp64", 1e-10, 1e-10), ("mixed", 1e-4, 1e-4)])
@pytest.mark.parametrize("grid", GRIDS)
def test_grid_matches_oracle(oracle_mod, prec, tol, etol, grid):
    from thrid_amd.pgk import ForceContext
    s = dict(water648(), nfft=np.array(grid, np.int32))
    o = oracle_mod.Oracle(s)
    o.mklist(s["rcut_book"], 0)
    ref = o.calforce(abi.MTS_LONG)
    c = ForceContext(s, prec)
    c.mklist(s["rcut_book"])
    got = c.calforce(abi.MTS_LONG)
    c.close()
    assert rms_rel(got["force"], ref["force"]) < tol
    assert abs(ene(got, "pot_ewk") - ene(ref, "pot_ewk")) < etol * abs(ene(ref, "pot_ewk"))
    k = abi.TENS_NAMES.index("pot_virit_coul")
    scale = np.max(np.abs(ref["virt"][k]))
    assert np.max(np.abs(got["virt"][k] - ref["virt"][k])) < 10 * etol * scale
