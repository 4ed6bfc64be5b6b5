"""The volume mode's flux form: region sets at the edges of its two region
passes (one, two, one wave's width and past it, the most, regions that overlap
or leave gaps) against the two-step calforce_hf + calheatf."""
import numpy as np
import pytest

from thrid_amd import abi, md
from helpers import small_slab

pytestmark = pytest.mark.gpu


def _regions(kind, lz):
    if kind.startswith("tiled"):
        z = np.linspace(0.0, lz, int(kind[5:]) + 1)
        return z[:-1], z[1:]
    if kind == "one":
        return np.array([0.3 * lz]), np.array([0.7 * lz])
    if kind == "inner":      # equal bins that leave both ends out
        z = np.linspace(0.4 * lz, 0.6 * lz, 9)
        return z[:-1], z[1:]
    return np.array([0.1, 0.3, 0.32, 0.8]) * lz, np.array([0.5, 0.45, 0.33, 1.0]) * lz


# the two-step form keeps its mixed per-atom arrays in 2^-32 fixed point: its
# regions' sums carry up to a few thousand roundings of 1.2e-10 per term
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 1e-7), ("fp32", 1e-11)])
@pytest.mark.parametrize("kind", ["one", "tiled2", "tiled63", "tiled64", "inner", "gaps"])
def test_volume_flux_matches_two_step(prec, tol, kind):
    from thrid_amd.pgk import ForceContext
    s = small_slab()
    lz = float(s["box"][2])
    z1, z2 = _regions(kind, lz)
    water = s["atype"] <= 2
    com = np.stack([np.bincount(s["molid"] - 1, s["mass"] * s["pos"][:, d], s["nmol"])
                    for d in range(3)], 1) / np.bincount(s["molid"] - 1, s["mass"])[:, None]
    hf = dict(mode=abi.HF_VOLUME, z1=z1, z2=z2, molecom=com,
              hftyp=np.where(water, abi.HFTYP_MOLE, abi.HFTYP_ATOM).astype(np.int32))
    vel = md.maxwell_boltzmann(s, 300.0, seed=31)
    mass = s["mass"] / md.MD_CONV
    c = ForceContext(s, prec)
    c.mklist(s["rcut_book"])
    got = c.calforce_heatf(hf, vel, mass)["hf"]
    c.calforce_hf(hf, per_atom=False)
    ref = c.calheatf(vel, mass)
    c.close()
    assert got.shape == ref.shape
    assert np.max(np.abs(got - ref)) < tol * np.max(np.abs(ref))


def test_most_regions_add_up():
    """1024 bins (the most the flux form takes): widths times the bins' flux
    add up to one region over the same range, per term."""
    from thrid_amd.pgk import ForceContext
    s = small_slab()
    lz = float(s["box"][2])
    vel = md.maxwell_boltzmann(s, 300.0, seed=32)
    mass = s["mass"] / md.MD_CONV
    z = np.linspace(0.0, lz, 1025)
    c = ForceContext(s, "fp64")
    c.mklist(s["rcut_book"])
    many = c.calforce_heatf(dict(mode=abi.HF_VOLUME, z1=z[:-1], z2=z[1:]), vel, mass)["hf"]
    one = c.calforce_heatf(dict(mode=abi.HF_VOLUME, z1=z[:1], z2=z[-1:]), vel, mass)["hf"][0]
    c.close()
    total = (many * (z[1:] - z[:-1])[:, None, None]).sum(0) / lz
    assert np.max(np.abs(total - one)) < 1e-10 * np.max(np.abs(one))
