"""The volume mode's flux form, region by region: each region against its own
scale (regions that no pair's segment meets are exactly zero), pairs too close
for a finite share, centres exactly on a region's plane."""
import numpy as np
import pytest

from thrid_amd import abi, md, systems
from helpers import small_slab

pytestmark = pytest.mark.gpu

PAIR = [abi.HFJ_VIRI + abi.HF_NAMES.index(k) for k in ("elin", "ljin", "elc", "vdw")]


def _regions(kind, lz):
    if kind.startswith("tiled"):
        z = np.linspace(0.0, lz, int(kind[5:]) + 1)
        return z[:-1], z[1:]
    if kind == "reversed":   # bounds the wrong way round: counted as the two-step form counts them
        return np.array([0.6, 0.3, 0.9]) * lz, np.array([0.4, 0.5, 0.1]) * lz
    # wide, thin, outside the slab, overlapping
    return (np.array([0.0, 0.0, 0.01, 0.45, 0.3, 0.9]) * lz,
            np.array([1.0, 0.2, 0.02, 0.4501, 0.8, 0.95]) * lz)


def _calls(s, prec, z1, z2, vel, per_atom=False):
    """The flux form, the two-step form (its 64 regions at a time) and, for
    each pair class and region, the sum of the sizes of the atoms' shares."""
    from thrid_amd.pgk import ForceContext
    mass = s["mass"] / md.MD_CONV
    c = ForceContext(s, prec)
    c.mklist(s["rcut_book"])
    got = c.calforce_heatf(dict(mode=abi.HF_VOLUME, z1=z1, z2=z2), vel, mass)["hf"]
    ref, size = [], []
    for k in range(0, len(z1), 64):
        w = c.calforce_hf(dict(mode=abi.HF_VOLUME, z1=z1[k:k + 64], z2=z2[k:k + 64]),
                          per_atom=per_atom)["viri_atm"]
        ref.append(c.calheatf(vel, mass))
        if per_atom:
            size.append((np.abs(w[:, :, :, 2, :]) * np.abs(vel)).sum(axis=(2, 3)))
    c.close()
    if per_atom:
        size = np.concatenate(size, 1) / (s["box"][0] * s["box"][1] * np.abs(z2 - z1))
    return got, np.concatenate(ref), size


# both forms' sums over one region: some 1e4 terms of FP64, whose roundings
# stay below 1e-13 of the sum of the terms' sizes
@pytest.mark.parametrize("kind,prec,vscale", [
    ("tiled2", "fp64", 1.0), ("tiled60", "fp64", 1.0), ("tiled1000", "fp64", 1.0),
    ("any", "fp64", 1.0), ("reversed", "fp64", 1.0), ("tiled60", "fp32", 1.0),
    ("any", "fp32", 1.0), ("tiled60", "fp64", 1e-9), ("any", "fp64", 1e6)])
def test_region_against_its_own_scale(kind, prec, vscale):
    s = small_slab()
    z1, z2 = _regions(kind, float(s["box"][2]))
    vel = vscale * md.maxwell_boltzmann(s, 300.0, seed=41)
    got, ref, size = _calls(s, prec, z1, z2, vel, per_atom=True)
    for row in PAIR[2:] if kind == "reversed" else PAIR:
        d = np.abs(got[:, row, 2] - ref[:, row, 2])
        assert np.all(d <= 1e-13 * size[row - abi.HFJ_VIRI]), row


@pytest.mark.parametrize("kind", ["tiled60", "any"])
def test_empty_regions_are_zero_mixed(kind):
    s = small_slab()
    z1, z2 = _regions(kind, float(s["box"][2]))
    z = s["pos"][:, 2]
    empty = (z2 < z.min()) | (z1 > z.max())
    vel = md.maxwell_boltzmann(s, 300.0, seed=42)
    got, _, _ = _calls(s, "mixed", z1, z2, vel)
    assert empty.sum() > 0 and not np.any(got[empty])
    assert np.all(np.any(got[~empty] != 0.0, axis=(1, 2)))


def _close_pair(s, first, second, dz):
    """s with an atom of type `first` moved to dz above one of type `second`
    of another molecule in the middle of the slab."""
    lz = float(s["box"][2])
    a = int(np.flatnonzero(s["atype"] == systems.TYPE_INDEX[first])[5])
    z = s["pos"][:, 2]
    other = (s["atype"] == systems.TYPE_INDEX[second]) & (s["molid"] != s["molid"][a])
    b = int(np.flatnonzero(other & (np.abs(z - 0.5 * lz) < 2.0) & (z % 1.0 > 0.2) & (z % 1.0 < 0.8))[0])
    pos = s["pos"].copy()
    pos[a] = pos[b] + np.array([0.0, 0.0, dz])
    return dict(s, pos=pos), int(z[b])


# 1e-4 A: a share of 1e50 in FP64, an infinite one of FP32 terms.  The other
# regions agree with the two-step form (mixed: its 2^-32 fixed point, as in
# test_gpu_hf_vol)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 1e-7), ("fp32", 1e-11)])
def test_bad_pair_stays_in_its_region(prec, tol):
    s, bad = _close_pair(small_slab(), "OB", "OB", 1e-4)
    z = np.arange(61.0)
    vel = md.maxwell_boltzmann(s, 300.0, seed=43)
    got, ref, _ = _calls(s, prec, z[:-1], z[1:], vel)
    row = abi.HFJ_VIRI + abi.HF_NAMES.index("vdw")
    rest = np.arange(60) != bad
    assert np.all(np.isfinite(got[rest]))
    assert np.max(np.abs(got[rest] - ref[rest])) < tol * np.max(np.abs(ref[rest]))
    assert not abs(got[bad, row, 2]) < 1e6 * np.max(np.abs(ref[rest, row, 2]))


def test_close_pair_without_lj_mixed():
    """An H atom (no LJ) 5e-4 A from an O: the LJ terms of FP32 overflow and
    count nothing."""
    s, bad = _close_pair(small_slab(), "HB", "OB", 5e-4)
    z = np.arange(61.0)
    vel = md.maxwell_boltzmann(s, 300.0, seed=44)
    got, ref, _ = _calls(s, "mixed", z[:-1], z[1:], vel)
    for row in (abi.HFJ_VIRI + abi.HF_NAMES.index("vdw"),
                abi.HFJ_POT + abi.HF_NAMES.index("vdw")):
        d = np.abs(got[:, row, 2] - ref[:, row, 2])
        assert np.max(d) < 1e-7 * np.max(np.abs(ref[:, row, 2]))


def _weight(z1, z2, ci, cj):
    """calvirihf's weight of a region for the segment cj -> ci."""
    ri1, rj1, ri2, rj2 = ci - z1, cj - z1, ci - z2, cj - z2
    lower, upper = ri1 * rj1 < 0, ri2 * rj2 < 0
    if lower and upper:
        ff = z2 - z1
    elif lower:
        ff = max(ri1, rj1)
    elif upper:
        ff = -min(ri2, rj2)
    elif ri1 * ri2 > 0:
        return 0.0
    else:
        ff = abs(ci - cj)
    return ff if ci >= cj else -ff


# 24 ions on a line along z, one column of the list: the pass's first atom of
# a pair is the one with the lower z.  Their centres are given on a grid of
# half an A, as are the planes, so many lie exactly on one.
# FP64: a few hundred terms; mixed: FP32 pair terms
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 1e-13), ("mixed", 2e-6)])
@pytest.mark.parametrize("tiled", [True, False])
def test_centres_on_planes(prec, tol, tiled):
    from thrid_amd.pgk import ForceContext
    rng = np.random.default_rng(45)
    n, box = 24, np.array([30.0, 30.0, 60.0])
    b = systems._Builder()
    for k in range(n):
        b.add_ion(*(("NA", 1.0), ("CL", -1.0))[k % 2], np.array([15.0, 15.0, 3.0 + 2.3 * k]))
    s = systems._finish(b, box, alpha=0.3, rrcut=10.0, rcut=10.0, rcut_book=11.0,
                        nfft=(32, 32, 60), order=4)
    centre = np.stack([np.full(n, 15.0), np.full(n, 15.0), rng.integers(20, 70, n) * 0.5], 1)
    z1, z2 = ((np.arange(5.0, 40.0), np.arange(6.0, 41.0)) if tiled else
              (10.0 + 0.5 * np.arange(36.0), 11.0 + 0.75 * np.arange(36.0)))
    vel = md.maxwell_boltzmann(s, 300.0, seed=46)
    q, pos = s["charge"], s["pos"]
    want = np.zeros((2, len(z1)))
    size = np.zeros((2, len(z1)))
    ties = [0, 0]
    for i in range(n):
        for j in range(i + 1, n):
            r = pos[i] - pos[j]
            r -= box * np.rint(r / box)
            r2 = r @ r
            if r2 > 100.0 or abs(centre[i, 2] - centre[j, 2]) >= 30.0:
                continue
            ti, tj = s["atype"][i] - 1, s["atype"][j] - 1
            x = s["lj_rmin"][ti, tj] ** 2 / r2
            f = (q[i] * q[j] / r2 ** 1.5,
                 12.0 * s["lj_eps"][ti, tj] * (x ** 6 - x ** 3) / r2)
            rw = 0.5 * (r @ (vel[i] + vel[j]))
            for reg in range(len(z1)):
                ci, cj = centre[i, 2], centre[j, 2]
                ff = _weight(z1[reg], z2[reg], ci, cj)
                true = (np.clip(ci, z1[reg], z2[reg]) - np.clip(cj, z1[reg], z2[reg]))
                if abs(ff - true) > 1e-9:
                    ties[int(ci > cj)] += 1
                for t in range(2):
                    want[t, reg] += ff * f[t] * rw
                    size[t, reg] += abs(ff * f[t] * rw)
    assert min(ties) > 5
    hf = dict(mode=abi.HF_VOLUME, z1=z1, z2=z2, molecom=centre,
              hftyp=np.full(n, abi.HFTYP_MOLE, np.int32))
    c = ForceContext(s, prec)
    c.mklist(s["rcut_book"])
    got = c.calforce_heatf(hf, vel, s["mass"] / md.MD_CONV)["hf"]
    c.close()
    vinv = 1.0 / (box[0] * box[1] * (z2 - z1))
    for t, row in enumerate(PAIR[2:]):
        assert np.all(np.abs(got[:, row, 2] - want[t] * vinv) <= tol * size[t] * vinv), row
