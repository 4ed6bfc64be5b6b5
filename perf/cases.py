"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is a plain dict.  Its "kind" says which public entry points a pass takes:

  force      set_positions, mklist where "rebuild", calforce: the call a host program makes for
             each of its own steps (a Fortran MD driver, an energy minimiser).  The result comes
             back to the host.
  md         a segment of a trajectory kept on the GPU: positions and velocities in, md_run, the
             state and the sampled energies out; plain velocity Verlet, a Nose-Hoover chain
             ("nhc") or RESPA ("respa" inner steps), and the heat flux every step ("flux": "bulk",
             or the number of bins along z).
  ensemble   independent replicas of uneven size stepped together (md_run_batch), each with its
             bulk heat flux every step.
  heatf      one heat-flux call: forces and the flux of the regions (calforce_heatf).
  hf_arrays  calforce_hf with the per-atom arrays on the host, then calheatf.

"fluid" is "water" (rigid three-site water in a cubic box) or "slab" (water between two layers of
1-propanol with vacuum beyond).  Sizes, cutoffs, grids and options are those of the workloads in
systems.py and bench.py, with odd sizes and grids in between.

The inputs are made from the seed alone, on the GPU: molecules on a jittered lattice, the waters
turned so that near neighbours attract, velocities of 300 K.
"""
import math

import numpy as np
import torch

from thrid_amd import abi, md, systems
from thrid_amd.pgk import ForceContext, md_run_batch

DT_FS = 1.0            # time step of every trajectory (the outer one with RESPA)
NSTEP_BOOK = 20        # list rebuilds, as bench.py
TEMPERATURE = 300.0
NHC_FREQ = 0.01        # 1/fs
NHC_LINKS = 4
NUMBER_DENSITY = 0.0334                      # waters per A^3
ALPHA = {9.0: 0.35, 10.0: 0.32, 12.0: 0.26}  # Ewald splitting of each cutoff


# ---- the cases -----------------------------------------------------------------------------
def listed():
    return [
        # the smallest system the tests and the reference's own runs use: launches and latency
        dict(name="force_water_648_fp64", kind="force", fluid="water", nmol=216, rc=9.0, skin=0.3,
             grid=24, order=4, precision="fp64", rebuild=False),
        # a host program that moves the atoms itself and rebuilds the list each time; odd size,
        # a grid without a power of two
        dict(name="force_water_24k_fp64_list", kind="force", fluid="water", nmol=7901, rc=10.0,
             skin=1.0, grid=72, order=6, precision="fp64", rebuild=True),
        # the drop-in call on the 100k water box
        dict(name="force_water_100k_mixed", kind="force", fluid="water", nmol=33333, rc=10.0,
             skin=1.0, grid=128, order=4, precision="mixed", rebuild=False),
        # the headline: a trajectory of the 100k water box, one list rebuild on the way
        dict(name="md_water_100k_mixed", kind="md", fluid="water", nmol=33333, rc=10.0, skin=1.0,
             grid=128, order=4, precision="mixed", nstep=20, nhc=False, respa=1, flux=""),
        # the thermostatted trajectory of a middle size in the FP32 form
        dict(name="md_water_24k_fp32_nvt", kind="md", fluid="water", nmol=8003, rc=10.0, skin=1.0,
             grid=64, order=4, precision="fp32", nstep=20, nhc=True, respa=1, flux=""),
        # flexible molecules: the slab under RESPA, the way the reference's shipped run works
        dict(name="md_slab_6k_fp64_respa", kind="md", fluid="slab", lx=31.25, lz=100.0,
             nwater=1100, nprop=150, rc=12.0, skin=1.0, grid=50, gridz=108, order=6,
             precision="fp64", nstep=10, nhc=False, respa=5, flux=""),
        # the 18.4k-atom slab under the chain
        dict(name="md_slab_18k_mixed_nvt", kind="md", fluid="slab", lx=50.0, lz=150.0, nwater=4096,
             nprop=512, rc=12.0, skin=1.0, grid=64, gridz=192, order=4, precision="mixed",
             nstep=20, nhc=True, respa=1, flux=""),
        # one Green-Kubo replica: the bulk heat flux every step
        dict(name="md_flux_water_5k_mixed", kind="md", fluid="water", nmol=1693, rc=10.0, skin=1.0,
             grid=40, order=4, precision="mixed", nstep=20, nhc=False, respa=1, flux="bulk"),
        # a Green-Kubo ensemble of uneven replicas
        dict(name="ensemble_16_mixed", kind="ensemble", fluid="water", nrep=16, nmin=500,
             nmax=3700, rc=10.0, skin=1.0, order=4, precision="mixed", nstep=10),
        # a heat-flux profile of the 18.4k-atom slab, one bin per A, waters by molecule
        dict(name="heatf_slab_18k_fp64_bins", kind="heatf", fluid="slab", lx=50.0, lz=150.0,
             nwater=4096, nprop=512, rc=12.0, skin=1.0, grid=64, gridz=192, order=4,
             precision="fp64", bins=150),
        # the largest: the 996,000-atom interface, 300 bins
        dict(name="heatf_slab_1M_mixed_bins", kind="heatf", fluid="slab", lx=200.0, lz=300.0,
             nwater=300000, nprop=8000, rc=12.0, skin=1.0, grid=192, gridz=288, order=6,
             precision="mixed", bins=300),
        # per-atom energies and virials for a host that keeps its own calheatf or analysis
        dict(name="hf_arrays_slab_18k_fp64", kind="hf_arrays", fluid="slab", lx=50.0, lz=150.0,
             nwater=4096, nprop=512, rc=12.0, skin=1.0, grid=64, gridz=192, order=4,
             precision="fp64", bins=0),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_water(rng, nmax):
    nmol = int(_log_uniform(rng, 216, nmax))
    box = (nmol / NUMBER_DENSITY) ** (1.0 / 3.0)
    rc = rng.choice([9.0, 10.0, 12.0])
    while rc > 9.0 and rc + 1.0 > 0.49 * box:
        rc = {12.0: 10.0, 10.0: 9.0}[rc]
    skin = 1.0 if rc + 1.0 <= 0.49 * box else 0.5 * box - rc - 0.01
    return dict(fluid="water", nmol=nmol, rc=rc, skin=skin,
                grid=systems.fft_friendly(int(math.ceil(box / rng.uniform(0.75, 1.0)))),
                order=rng.choice([4, 4, 6]))


def _draw_slab(rng, lmax):
    lx = rng.uniform(27.0, lmax)
    side = max(1, int(round(lx / 3.105)))
    layers = rng.randint(6, 20)
    nprop = 2 * int(rng.uniform(0.2, 0.5) * (lx / 5.0) ** 2) + 2
    lz = 3.105 * layers + 2 * 12.0 + rng.uniform(10.0, 40.0)
    spacing = rng.uniform(0.78, 1.04)
    return dict(fluid="slab", lx=lx, lz=max(lz, 30.0), nwater=side * side * layers - rng.randint(0, side),
                nprop=nprop, rc=12.0, skin=1.0, grid=systems.fft_friendly(int(math.ceil(lx / spacing))),
                gridz=systems.fft_friendly(int(math.ceil(max(lz, 30.0) / spacing))),
                order=rng.choice([4, 6]))


def draw(rng):
    kind = rng.choice(["force", "force", "md", "md", "md", "heatf", "heatf", "ensemble", "hf_arrays"])
    precision = rng.choice(["fp64", "mixed", "mixed", "fp32"])
    if kind == "force":
        return dict(kind=kind, **_draw_water(rng, 40000), precision=precision,
                    rebuild=rng.random() < 0.4)
    if kind == "md":
        form = rng.choice(["nve", "nvt", "respa", "flux"])
        if form == "respa" or (form == "nvt" and rng.random() < 0.5):
            fluid = _draw_slab(rng, 60.0)
        else:
            fluid = _draw_water(rng, 12000)
        flux = ""
        if form == "flux":
            flux = rng.choice(["bulk", "bulk", str(rng.randint(2, 40))])
        return dict(kind=kind, **fluid, precision=precision, nstep=rng.randint(5, 25),
                    nhc=form == "nvt", respa=rng.randint(2, 6) if form == "respa" else 1, flux=flux)
    if kind == "heatf":
        return dict(kind=kind, **_draw_slab(rng, 90.0), precision=rng.choice(["fp64", "mixed"]),
                    bins=rng.choice([0, rng.randint(1, 40), rng.randint(41, 300)]))
    if kind == "ensemble":
        return dict(kind=kind, fluid="water", nrep=rng.randint(3, 16), nmin=400,
                    nmax=rng.randint(900, 3700), rc=9.0, skin=1.0, order=4,
                    precision=rng.choice(["mixed", "fp64"]), nstep=rng.randint(4, 10))
    return dict(kind=kind, **_draw_slab(rng, 45.0), precision="fp64",
                bins=rng.choice([0, rng.randint(1, 12)]))


# ---- inputs --------------------------------------------------------------------------------
def _rotations(n, gen):
    q = torch.randn(n, 4, dtype=torch.float64, device="cuda", generator=gen)
    a, b, c, d = (q / q.norm(dim=1, keepdim=True)).T
    return torch.stack([a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c),
                        2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b),
                        2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d],
                       1).reshape(n, 3, 3)


def _waters(nmol, dims, origin, span, box, gen):
    """nmol waters (H, O, H) on a jittered lattice of `dims` sites over origin .. origin + span,
    each turned a few times towards a lower electrostatic energy with its 26 neighbours."""
    f64 = dict(dtype=torch.float64, device="cuda")
    tmpl = systems.TEMPLATES["water"]()
    local = torch.tensor(tmpl["pos"], **f64)
    q = torch.tensor(tmpl["charges"], **f64)
    box = torch.tensor(box, **f64)
    grid = torch.stack(torch.meshgrid(*[torch.arange(k, device="cuda") for k in dims], indexing="ij"), -1)
    step = torch.tensor([s / k for s, k in zip(span, dims)], **f64)
    nsite = dims[0] * dims[1] * dims[2]
    site = torch.tensor(origin, **f64) + (grid + 0.5) * step
    site = site + 0.3 * (torch.rand(*dims, 3, generator=gen, **f64) - 0.5)
    keep = torch.ones(nsite, dtype=torch.bool, device="cuda")
    keep[torch.randperm(nsite, device="cuda", generator=gen)[nmol:]] = False
    here = keep.reshape(*dims).to(torch.float64)
    off = (_rotations(nsite, gen) @ local.T).transpose(1, 2).reshape(*dims, 3, 3)

    def energy(mine):
        e = torch.zeros(dims, **f64)
        for d in [(x, y, z) for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1) if (x, y, z) != (0, 0, 0)]:
            roll = lambda t: torch.roll(t, d, (0, 1, 2))                     # noqa: E731
            r = roll(site) - site
            r = r - box * torch.round(r / box)
            other = roll(off) + r[..., None, :]
            m = roll(here)
            for a in range(3):
                dist = (other - mine[..., a:a + 1, :]).norm(dim=-1).clamp_min(0.5)
                e += m * q[a] * (q / dist).sum(-1)
        return e

    parity = grid[..., 0] % 2 + 2 * (grid[..., 1] % 2) + 4 * (grid[..., 2] % 2)
    for _ in range(2):
        for cls in range(8):
            trial = (_rotations(nsite, gen) @ local.T).transpose(1, 2).reshape(*dims, 3, 3)
            better = (energy(trial) < energy(off)) & (parity == cls)
            off = torch.where(better[..., None, None], trial, off)
    return (site[..., None, :] + off).reshape(nsite, 3, 3)[keep].reshape(-1, 3).cpu().numpy()


def _propanols(n, lx, zlo, up, rng):
    """n 1-propanols standing on a 5 x 5 x 7 A lattice from zlo upwards, the hydroxyl end up."""
    tmpl = systems.TEMPLATES["propanol"]()["pos"]
    local = tmpl - tmpl.mean(axis=0)
    axis = local[3] - local[2]
    axis = axis / np.linalg.norm(axis)
    side = np.cross(axis, [0.0, 0.0, 1.0])
    side = side / np.linalg.norm(side)
    local = local @ np.stack([side, np.cross(axis, side), axis], 1) * (1.0, 1.0, 1.0 if up else -1.0)
    if not up:
        local = local * (-1.0, 1.0, 1.0)       # a rotation, not a mirror image
    k = max(1, int(lx // 5.0))
    nz = -(-n // (k * k))
    site = np.stack(np.meshgrid(np.arange(k), np.arange(k), np.arange(nz), indexing="ij"), -1)
    site = site.transpose(2, 0, 1, 3).reshape(-1, 3)[:n]
    site = (site + 0.5) * (lx / k, lx / k, 7.0) + (0.0, 0.0, zlo)
    return (site[:, None, :] + local[None] + rng.normal(scale=0.03, size=(n, 12, 3))).reshape(-1, 3)


def _tile(rows, nmol, natom, base):
    """1-based index rows of one molecule repeated for nmol molecules whose atoms start at base."""
    rows = np.asarray(rows, np.int64)
    return (rows[None] + base + natom * np.arange(nmol)[:, None, None]).reshape(-1, rows.shape[1]).astype(np.int32)


def _partners(tmpl):
    """The atoms each atom of a molecule is excluded from (1-2, 1-3 and 1-4 neighbours)."""
    n = len(tmpl["types"])
    part = [set() for _ in range(n)]
    ends = [(b[0], b[1]) for b in tmpl["bonds"]] + [(a[0], a[2]) for a in tmpl["angles"]]
    for i, j in ends + [(t[0], t[3]) for t in tmpl["tors"]]:
        part[i - 1].add(j - 1)
        part[j - 1].add(i - 1)
    return part


def _system(pos, counts, box, rc, skin, grid, order):
    """The system dict of `counts` = ((template name, molecules), ...) in the order of pos, and its
    exclusions."""
    base = systems.water_box(nside=1, nmol=1, box=box[0])
    kinds = [(systems.TEMPLATES[k](), k, n) for k, n in counts if n]
    s = dict(base, name="case", natom=len(pos), box=np.array(box, np.float64), pos=pos,
             alpha=ALPHA[rc], rrcut=rc, rcut=rc, rcut_book=rc + skin,
             nspltbl=int(round((rc + 2.0) / 0.01)), nfft=np.array(grid, np.int32), pme_order=order)
    types, charge, molid, bonds, btype, angles, atype, tors, ttype = ([] for _ in range(9))
    idx, lst = [], []
    first, mol, nlist = 0, 0, 0
    for t, _name, n in kinds:
        na = len(t["types"])
        types.append(np.tile([systems.TYPE_INDEX[x] for x in t["types"]], n))
        charge.append(np.tile(t["charges"], n))
        molid.append(np.repeat(mol + 1 + np.arange(n), na))
        bonds.append(_tile([b[:2] for b in t["bonds"]], n, na, first))
        btype.append(np.tile([systems.BOND_INDEX[b[2]] for b in t["bonds"]], n))
        angles.append(_tile([a[:3] for a in t["angles"]], n, na, first))
        atype.append(np.tile([systems.ANGLE_INDEX[a[3]] for a in t["angles"]], n))
        if t["tors"]:
            tors.append(_tile([x[:4] for x in t["tors"]], n, na, first))
            ttype.append(np.tile([systems.RB_INDEX[x[4]] for x in t["tors"]], n))
        above = [sorted(j for j in p if j > i) for i, p in enumerate(_partners(t))]
        row = [(j, True) for p in above for j in (p or [None])]
        start = np.cumsum([0] + [max(len(p), 1) for p in above])
        idx.append((start[None, :-1] + nlist + 1 + start[-1] * np.arange(n)[:, None]).reshape(-1))
        one = np.array([0 if j is None else j + 1 for j, _ in row])
        lst.append(np.where(one[None] > 0, one[None] + first + na * np.arange(n)[:, None], 0).reshape(-1))
        nlist += n * int(start[-1])
        first += n * na
        mol += n
    cat = lambda a, shape: np.concatenate(a).astype(np.int32) if a else np.zeros(shape, np.int32)   # noqa: E731
    s.update(atype=cat(types, 0), molid=cat(molid, 0), nmol=mol,
             charge=np.concatenate(charge) * systems.QSCALE,
             bond_ij=cat(bonds, (0, 2)), bond_type=cat(btype, 0),
             angl_ijk=cat(angles, (0, 3)), angl_type=cat(atype, 0),
             torsrb_ijkl=cat(tors, (0, 4)), torsrb_type=cat(ttype, 0))
    s["mass"] = np.array([t.mass for t in systems.ATOM_TYPES])[s["atype"] - 1]
    s["torsrb_ring14"] = np.ones(len(s["torsrb_type"]))
    return s, (np.append(np.concatenate(idx), nlist + 1).astype(np.int32), np.concatenate(lst).astype(np.int32))


def _fluid(case, seed):
    """The system, its exclusions and its velocities."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    if case["fluid"] == "water":
        nmol = case["nmol"]
        side = math.ceil(nmol ** (1.0 / 3.0) - 1e-9)
        box = (max((nmol / NUMBER_DENSITY) ** (1.0 / 3.0), 2.0 * (case["rc"] + case["skin"]) + 0.01),) * 3
        pos = _waters(nmol, (side,) * 3, (0.0,) * 3, box, box, gen)
        grid = case.get("grid") or systems.fft_friendly(math.ceil(box[0]))
        s, excl = _system(pos, (("water", nmol),), box, case["rc"], case["skin"], (grid,) * 3, case["order"])
    else:
        lx, lz, nw, npr = case["lx"], case["lz"], case["nwater"], case["nprop"]
        side = max(1, int(round(lx / 3.105)))
        layers = -(-nw // (side * side))
        thick = 3.105 * layers
        box = (lx, lx, lz)
        z0 = 0.5 * (lz - thick)
        pos = _waters(nw, (side, side, layers), (0.0, 0.0, z0), (lx, lx, thick), box, gen)
        lower, per = npr // 2, max(1, int(lx // 5.0)) ** 2
        pos = np.concatenate([pos, _propanols(lower, lx, z0 - 2.0 - 7.0 * -(-lower // per), True, rng),
                              _propanols(npr - lower, lx, z0 + thick + 2.0, False, rng)])
        s, excl = _system(pos, (("water", nw), ("propanol", npr)), box, case["rc"], case["skin"],
                          (case["grid"], case["grid"], case["gridz"]), case["order"])
    sd = np.sqrt(md.KB_EREF * TEMPERATURE * md.MD_CONV / s["mass"])
    vel = rng.normal(size=(s["natom"], 3)) * sd[:, None]
    vel -= (s["mass"][:, None] * vel).sum(0) / s["mass"].sum()
    return s, excl, vel


def _replicas(case, seed):
    # sizes spread evenly over their logarithm, in an order that mixes small and large
    nmol = np.geomspace(case["nmin"], case["nmax"], case["nrep"])
    nmol = np.random.default_rng(case["nrep"]).permutation(nmol).astype(int)
    return [_fluid(dict(case, nmol=int(n)), seed + 1 + k) for k, n in enumerate(nmol)]


def _regions(s, bins, mole):
    """bins = 0: one bulk region over the box; else equal bins along z, waters by their centre of
    mass where `mole`."""
    lz = float(s["box"][2])
    if bins == 0:
        return dict(mode=abi.HF_BULK, z1=np.array([0.0]), z2=np.array([lz]))
    z = np.linspace(0.0, lz, bins + 1)
    hf = dict(mode=abi.HF_VOLUME, z1=z[:-1], z2=z[1:])
    if mole:
        water = np.isin(s["atype"], [systems.TYPE_INDEX["OB"], systems.TYPE_INDEX["HB"]])
        hf["hftyp"] = np.where(water, abi.HFTYP_MOLE, abi.HFTYP_ATOM).astype(np.int32)
        com = np.zeros((s["nmol"], 3))
        w = np.zeros(s["nmol"])
        for d in range(3):
            com[:, d] = np.bincount(s["molid"] - 1, s["mass"] * s["pos"][:, d], s["nmol"])
        w = np.bincount(s["molid"] - 1, s["mass"], s["nmol"])
        com /= w[:, None]
        hf["molecom"] = com - s["box"] * np.floor(com / s["box"])
    return hf


def _md_context(s, excl, case):
    c = ForceContext(s, case["precision"], excl=excl)
    cons = md.rigid_constraints(s)
    c.md_setup(s["mass"], *cons, DT_FS)
    if case.get("respa", 1) > 1:
        short, long = abi.MTS_SHORT, abi.MTS_LONG
        c.md_respa(case["respa"], abi.Mts(short, short, short, short, long, long, long))
    flux = case.get("flux", "bulk")
    if flux:
        c.md_heatf(_regions(s, 0 if flux == "bulk" else int(flux), False), 1)
    return c, 3 * s["natom"] - len(cons[1]) - 3


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        reps = _replicas(case, seed)
        return dict(case=case, ctx=[_md_context(s, e, case)[0] for s, e, _ in reps],
                    pos=[s["pos"] for s, _, _ in reps], vel=[v for _, _, v in reps],
                    books=[s["rcut_book"] for s, _, _ in reps])
    s, excl, vel = _fluid(case, seed)
    state = dict(case=case, pos=s["pos"], vel=vel, book=s["rcut_book"])
    if kind == "md":
        state["ctx"], state["nfree"] = _md_context(s, excl, case)
        return state
    state["ctx"] = ForceContext(s, case["precision"], excl=excl)
    state["ctx"].mklist(s["rcut_book"])
    if kind != "force":
        state["hf"] = _regions(s, case["bins"], True)
        state["mass"] = s["mass"] / md.MD_CONV      # m v^2 / 2 in the force calls' energy unit
    return state


# ---- one pass ------------------------------------------------------------------------------
def _segment_out(c, rows, flux):
    pos, vel = c.md_state()
    out = dict(pos=pos, vel=vel, energies=rows)
    if flux:
        out["flux"] = c.md_heatf_series()
    return out


def run(state):
    case, c = state["case"], state["ctx"]
    if case["kind"] == "ensemble":
        for r, p, v in zip(c, state["pos"], state["vel"]):
            r.set_positions(p)
            r.md_set_velocities(v)
        rows = md_run_batch(c, case["nstep"], NSTEP_BOOK, state["books"], case["nstep"])
        return [_segment_out(r, rows[k], True) for k, r in enumerate(c)]
    c.set_positions(state["pos"])
    if case["kind"] == "md":
        if case["nhc"]:      # the chain's state belongs to the segment's start
            c.md_nhc(TEMPERATURE, NHC_FREQ, state["nfree"], NHC_LINKS)
        c.md_set_velocities(state["vel"])
        rows = c.md_run(case["nstep"], NSTEP_BOOK, state["book"], case["nstep"])
        return _segment_out(c, rows, case["flux"])
    if case["kind"] == "force":
        if case["rebuild"]:
            c.mklist(state["book"])
        return c.calforce()
    if case["kind"] == "heatf":
        return c.calforce_heatf(state["hf"], state["vel"], state["mass"])
    out = c.calforce_hf(state["hf"])
    out["hf"] = c.calheatf(state["vel"], state["mass"])
    return out


# ---- what a pass cannot do without ---------------------------------------------------------
def _force_work(natom, density, rc, points):
    """Flops of one force evaluation (49 per pair inside the cutoff, two transforms of the grid and
    its influence function, spreading and gathering of 6 x 6 x 6 points or fewer)."""
    pairs = 0.5 * natom * density * 4.0 / 3.0 * math.pi * rc ** 3
    return 49.0 * pairs + 2 * 2.5 * points * math.log2(points) + 30.0 * points + 1000.0 * natom


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        mean = (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        one = work(dict(case, kind="md", nmol=int(mean), grid=int((mean / NUMBER_DENSITY) ** (1 / 3)) + 1,
                        flux="bulk", respa=1))
        return {k: v * case["nrep"] for k, v in one.items()}
    if case["fluid"] == "water":
        natom, points = 3 * case["nmol"], case["grid"] ** 3
    else:
        natom, points = 3 * case["nwater"] + 12 * case["nprop"], case["grid"] ** 2 * case["gridz"]
    flops = _force_work(natom, 0.1, case["rc"], points)
    nbytes = natom * (24.0 + 24.0 + 16.0) + 2.0 * points * 4       # positions, forces, charges; the grid
    if kind == "md":
        flops = (flops + 2000.0 * natom) * (case["nstep"] + 1) * (2 if case["flux"] else 1)
        nbytes = (nbytes + natom * 96.0) * (case["nstep"] + 1)     # the state read and written each step
    if kind in ("heatf", "hf_arrays"):
        flops *= 2
        nbytes += natom * 32.0
    if kind == "hf_arrays":
        nbytes += 8.0 * abi.NHF * natom * (1 + 9 * max(1, case["bins"]))
    return {"bytes": nbytes, "flops": flops}


# ---- the same results in 64 bits, from plain torch ------------------------------------------
class _Plain:
    """The force field in FP64 torch operations: every pair inside the cutoff from cells, the error
    function itself in place of spline tables, torch's FFT, bonded forces from autograd."""

    def __init__(self, s, excl):
        self.s, self.n = s, s["natom"]
        t = lambda a, d=torch.float64: torch.as_tensor(np.asarray(a), dtype=d, device="cuda")   # noqa: E731
        self.t = t
        self.box = t(s["box"])
        self.q, self.mol = t(s["charge"]), t(s["molid"], torch.int64)
        self.type = t(s["atype"], torch.int64) - 1
        self.eps, self.rm2 = t(s["lj_eps"]), t(s["lj_rmin"]) ** 2
        self.nt = self.eps.shape[0]
        idx, lst = excl
        i = np.repeat(np.arange(self.n), np.diff(idx))
        on = np.asarray(lst) > 0
        self.ex = t(np.stack([i[on], np.asarray(lst)[on] - 1]), torch.int64)
        self.exkey = torch.sort(self.ex[0] * self.n + self.ex[1])[0]
        self.mass = t(s["mass"])

    def image(self, r):
        return r - self.box * torch.round(r / self.box)

    def pairs(self, x, rmax):
        """Blocks of pairs i < j closer than rmax that are not excluded."""
        dims = [max(1, int(float(b) / rmax)) for b in self.box]
        nc = torch.tensor(dims, device="cuda")
        w = x / self.box
        w = w - torch.floor(w)
        ijk = torch.minimum((w * nc).long(), nc - 1)
        cell = (ijk[:, 0] * dims[1] + ijk[:, 1]) * dims[2] + ijk[:, 2]
        order = torch.argsort(cell)
        count = torch.bincount(cell, minlength=dims[0] * dims[1] * dims[2])
        start = torch.cumsum(count, 0) - count
        most = int(count.max())
        table = torch.full((count.numel(), most), -1, dtype=torch.int64, device="cuda")
        table[cell[order], torch.arange(self.n, device="cuda") - start[cell[order]]] = order
        table = table.reshape(*dims, most)
        reach = [(0,) if d == 1 else (0, 1) if d == 2 else (-1, 0, 1) for d in dims]
        slices = max(1, count.numel() * most * most // 100_000_000)
        for d in [(a, b, c) for a in reach[0] for b in reach[1] for c in reach[2]]:
            other = torch.roll(table, d, (0, 1, 2)).reshape(-1, most)
            for mine, its in zip(table.reshape(-1, most).chunk(slices), other.chunk(slices)):
                r = self.image(x[mine][:, :, None, :] - x[its][:, None, :, :])
                near = ((r * r).sum(-1) < rmax * rmax) & (mine[:, :, None] >= 0) & (mine[:, :, None] < its[:, None, :])
                c, a, b = torch.nonzero(near, as_tuple=True)
                i, j = mine[c, a], its[c, b]
                at = torch.searchsorted(self.exkey, i * self.n + j).clamp_max(self.exkey.numel() - 1)
                keep = self.exkey[at] != i * self.n + j
                yield i[keep], j[keep]

    def listed(self, x):
        blocks = list(self.pairs(x, self.s["rcut_book"]))
        return torch.cat([b[0] for b in blocks]), torch.cat([b[1] for b in blocks])

    @staticmethod
    def tensor(f, r):
        return torch.einsum("pa,pn->an", f, r)

    def nonbonded(self, x, blocks):
        """Listed pairs: forces, energies (Coulomb, LJ) and tensors."""
        f = torch.zeros_like(x)
        e = torch.zeros(2, dtype=torch.float64, device="cuda")
        w = torch.zeros(2, 3, 3, dtype=torch.float64, device="cuda")
        al = self.s["alpha"]
        for i0, j0 in blocks:
            for i, j in zip(i0.split(20_000_000), j0.split(20_000_000)):
                r = self.image(x[i] - x[j])
                r2 = (r * r).sum(-1)
                d = torch.sqrt(r2)
                near = (d <= self.s["rrcut"]).to(torch.float64)
                qq = self.q[i] * self.q[j] * near
                ec = qq * torch.erfc(al * d) / d
                fc = (ec + qq * 2 * al / math.sqrt(math.pi) * torch.exp(-(al * d) ** 2)) / r2
                eps, s6 = self.lj(i, j, r2)
                ev, fv = eps * s6 * (s6 - 2.0), 12.0 * eps * s6 * (s6 - 1.0) / r2
                e += torch.stack([ec.sum(), ev.sum()])
                fc, fv = fc[:, None] * r, fv[:, None] * r
                w += torch.stack([self.tensor(fc, r), self.tensor(fv, r)])
                f.index_add_(0, i, fc + fv)
                f.index_add_(0, j, -(fc + fv))
        return f, e, w

    def lj(self, i, j, r2):
        inside = (r2 <= self.s["rcut"] ** 2).to(torch.float64)
        k = self.type[i] * self.nt + self.type[j]
        return self.eps.reshape(-1)[k] * inside, (self.rm2.reshape(-1)[k] / r2) ** 3

    def excluded(self, x):
        al = self.s["alpha"]
        i, j = self.ex
        r = self.image(x[i] - x[j])
        r2 = (r * r).sum(-1)
        d = torch.sqrt(r2)
        qq = self.q[i] * self.q[j]
        e = -qq * torch.erf(al * d) / d
        fs = (e + qq * 2 * al / math.sqrt(math.pi) * torch.exp(-(al * d) ** 2)) / r2
        fv = fs[:, None] * r
        f = torch.zeros_like(x).index_add_(0, i, fv).index_add_(0, j, -fv)
        return f, e.sum(), self.tensor(fv, r)

    def spline(self, w, p):
        """B-spline weights of order p and their derivatives, [p][atoms], for the p grid points that
        end at the atom's own."""
        a = [1.0 - w, w]
        for k in range(3, p + 1):
            if k == p:
                low = [torch.zeros_like(w)] + a + [torch.zeros_like(w)]
                d = [low[m] - low[m + 1] for m in range(p)]
            z = [torch.zeros_like(w)] + a + [torch.zeros_like(w)]
            a = [((w + (k - 1 - m)) * z[m] + (m + 1 - w) * z[m + 1]) / (k - 1) for m in range(k)]
        return a, d

    def influence(self):
        if hasattr(self, "eterm"):
            return
        s, p = self.s, self.s["pme_order"]
        k3 = [int(k) for k in s["nfft"]]
        m = [torch.fft.fftfreq(k, 1.0 / k, dtype=torch.float64, device="cuda") / b for k, b in zip(k3, s["box"])]
        a, _ = self.spline(torch.zeros(1, dtype=torch.float64, device="cuda"), p)
        mod = []
        for k in k3:
            row = torch.zeros(k, dtype=torch.float64, device="cuda")
            for j, v in enumerate(a):
                row[j % k] += v[0]
            mod.append(torch.fft.fft(row).abs() ** 2)
        self.m = (m[0][None, None, :], m[1][None, :, None], m[2][:, None, None])
        msq = self.m[0] ** 2 + self.m[1] ** 2 + self.m[2] ** 2
        half = [0.5 * k / float(b) for k, b in zip(k3, s["box"])]
        rk = half[1] if half[1] < half[0] else half[0]
        rk = half[2] if half[2] < half[1] else rk
        self.fac = math.pi ** 2 / s["alpha"] ** 2
        b = mod[0][None, None, :] * mod[1][None, :, None] * mod[2][:, None, None]
        vol = float(np.prod(s["box"]))
        self.zero = msq == 0
        safe = torch.where(self.zero, torch.ones_like(msq), msq)
        self.eterm = torch.where((msq <= (0.9 * rk) ** 2) & ~self.zero,
                                 torch.exp(-self.fac * msq) / (math.pi * vol * b * safe), torch.zeros_like(msq))
        self.vterm = 2.0 * (self.fac * msq + 1.0) / safe

    def recip(self, x):
        self.influence()
        s, p = self.s, self.s["pme_order"]
        k3 = [int(k) for k in s["nfft"]]
        wts, ders, at = [], [], []
        for d in range(3):
            w = x[:, d] / float(s["box"][d])
            fr = k3[d] * (w - torch.floor(w))
            i0 = torch.floor(fr).clamp_max(k3[d] - 1)
            a, b = self.spline(fr - i0, p)
            wts.append(a)
            ders.append([v * k3[d] / float(s["box"][d]) for v in b])
            at.append([(i0.long() - p + 1 + m) % k3[d] for m in range(p)])
        grid = torch.zeros(k3[0] * k3[1] * k3[2], dtype=torch.float64, device="cuda")
        cells = [(a, b, c, (at[2][c] * k3[1] + at[1][b]) * k3[0] + at[0][a])
                 for a in range(p) for b in range(p) for c in range(p)]
        for a, b, c, k in cells:
            grid.index_add_(0, k, self.q * wts[0][a] * wts[1][b] * wts[2][c])
        spec = torch.fft.fftn(grid.reshape(k3[2], k3[1], k3[0]))
        s2 = spec.real ** 2 + spec.imag ** 2
        e = 0.5 * (self.eterm * s2).sum()
        w = torch.zeros(3, 3, dtype=torch.float64, device="cuda")
        for a in range(3):
            for n in range(3):
                w[a, n] = -0.5 * (self.eterm * s2 * (self.vterm * self.m[a] * self.m[n] - float(a == n))).sum()
        phi = (torch.fft.ifftn(spec * self.eterm).real * grid.numel()).reshape(-1)
        f = torch.zeros_like(x)
        for a, b, c, k in cells:
            g = self.q * phi[k]
            f[:, 0] -= g * ders[0][a] * wts[1][b] * wts[2][c]
            f[:, 1] -= g * wts[0][a] * ders[1][b] * wts[2][c]
            f[:, 2] -= g * wts[0][a] * wts[1][b] * ders[2][c]
        return f, e, w

    def bonded(self, x):
        """Forces, energies (bond, angle, torsion, LJ 1-4, Coulomb 1-4) and the tensors of bonds,
        angles, torsions and 1-4 pairs."""
        s, t = self.s, self.t
        f = torch.zeros_like(x)
        es, ws = [torch.zeros((), dtype=torch.float64, device="cuda")] * 5, [torch.zeros(3, 3, dtype=torch.float64, device="cuda")] * 4
        if not len(s["torsrb_type"]):
            return f, es, ws
        row = lambda k: t(s[k], torch.int64) - 1      # noqa: E731
        bij, bt, aij, at, tij, tt = (row(k) for k in ("bond_ij", "bond_type", "angl_ijk", "angl_type",
                                                      "torsrb_ijkl", "torsrb_type"))
        unit = lambda v: v / v.norm(dim=1, keepdim=True)      # noqa: E731
        sign = t([1.0, -1.0, 1.0, -1.0, 1.0, -1.0])

        def bond(y):
            return (t(s["bond_k"])[bt] * ((y[bij[:, 0]] - y[bij[:, 1]]).norm(dim=1) - t(s["bond_r0"])[bt]) ** 2).sum(),

        def angle(y):
            c = (unit(y[aij[:, 0]] - y[aij[:, 1]]) * unit(y[aij[:, 2]] - y[aij[:, 1]])).sum(1)
            return (t(s["angl_k"])[at] * (torch.acos(c) - t(s["angl_theta0"])[at]) ** 2).sum(),

        def torsion(y):
            i, j, k, l = (y[tij[:, m]] for m in range(4))
            c = (unit(torch.cross(j - i, j - k, dim=1)) * unit(torch.cross(j - k, l - k, dim=1))).sum(1)
            return ((t(s["torsrb_c"])[tt] * sign) * torch.stack([c ** m for m in range(6)], 1)).sum(),

        def pair14(y):
            i, l = tij[:, 0], tij[:, 3]
            r2 = ((y[i] - y[l]) ** 2).sum(1)
            k = self.type[i] * self.nt + self.type[l]
            s6 = (self.rm2.reshape(-1)[k] / r2) ** 3
            lj = self.eps.reshape(-1)[k] * s6 * (s6 - 2.0) / t(s["torsrb_divfac_vdw"])[tt]
            el = self.q[i] * self.q[l] / torch.sqrt(r2) / t(s["torsrb_divfac_elc"])[tt]
            return lj.sum(), el.sum()

        es, ws = [], []
        for term in (bond, angle, torsion, pair14):
            with torch.enable_grad():
                y = x.detach().clone().requires_grad_(True)
                strain = torch.zeros(3, 3, dtype=torch.float64, device="cuda", requires_grad=True)
                parts = term(y + y @ strain.T)
                gy, gs = torch.autograd.grad(sum(parts), (y, strain))
            f -= gy
            es += [v.detach() for v in parts]
            ws.append(-gs)
        return f, es, ws

    def calforce(self, x, blocks=None):
        """The record of a force call: forces, energies and tensors in the library's order."""
        s = self.s
        fp, ep, wp = self.nonbonded(x, self.pairs(x, s["rcut_book"]) if blocks is None else blocks)
        fx, ex, wx = self.excluded(x)
        fr, er, wr = self.recip(x)
        fb, (eb, ea, et, e14v, e14c), (wb, wa, wt, w14) = self.bonded(x)
        ewc = -s["alpha"] / math.sqrt(math.pi) * float((s["charge"] ** 2).sum())
        e = dict.fromkeys(abi.ENE_NAMES, 0.0)
        e.update(pot_vdw=ep[1], pot_elc=ep[0] + ex, pot_ewk=er, pot_ewc=ewc, pot_vdw14=e14v, pot_elc14=e14c,
                 pot_bond=eb, pot_angl=ea, pot_torsrb=et, pot_viri_coul=ep[0] + ex + er, pot_viri_lj=wp[1].trace(),
                 atm_viri_bond=wb.trace(), atm_viri_angl=wa.trace(), atm_viri_tors=wt.trace(), atm_viri_14=w14.trace())
        net = float(s["charge"].sum()) ** 2 * -math.pi / (s["alpha"] ** 2 * float(np.prod(s["box"])))
        e["pot_ewnq"] = 0.5 * net
        e["pot_viri_coul"] = e["pot_viri_coul"] + net
        e["pot_nonbon"] = sum(e[k] for k in ("pot_vdw", "pot_elc", "pot_ewk", "pot_ewc", "pot_ewnq", "pot_vdw14", "pot_elc14"))
        e["pot_tot"] = e["pot_nonbon"] + e["pot_bond"] + e["pot_angl"] + e["pot_torsrb"]
        eye = torch.eye(3, dtype=torch.float64, device="cuda")
        virt = torch.stack([wp[0] + wx + wr + 0.5 * net * eye, wp[1], wb, wa, wt, w14])
        return dict(force=fp + fx + fr + fb, ene=torch.stack([torch.as_tensor(e[k], dtype=torch.float64, device="cuda") for k in abi.ENE_NAMES]), virt=virt)

    # -- trajectories --
    def constraints(self):
        ij, d, _ = md.rigid_constraints(self.s)
        ij = self.t(ij, torch.int64).reshape(-1, 3, 2) - 1          # three per water
        self.ci, self.cj = ij[..., 0], ij[..., 1]
        self.d2 = self.t(d).reshape(-1, 3) ** 2
        self.minv = 1.0 / self.mass
        # change of the separation of constraint k per unit push along constraint l
        same = lambda a, b: (a[:, :, None] == b[:, None, :]).to(torch.float64)      # noqa: E731
        mi, mj = self.minv[self.ci], self.minv[self.cj]
        self.couple = (same(self.ci, self.ci) - same(self.ci, self.cj)) * mi[:, :, None] \
            - (same(self.cj, self.ci) - same(self.cj, self.cj)) * mj[:, :, None]

    def push(self, y, g, r):
        """y with each constraint's push g r / m added to its two atoms."""
        v = g[..., None] * r
        y = y.index_add(0, self.ci.reshape(-1), (v * self.minv[self.ci][..., None]).reshape(-1, 3))
        return y.index_add(0, self.cj.reshape(-1), (-v * self.minv[self.cj][..., None]).reshape(-1, 3))

    def hold_positions(self, x, v, old, dt):
        ro = old[self.ci] - old[self.cj]
        r0 = x[self.ci] - x[self.cj]
        g = torch.zeros_like(self.d2)
        for _ in range(8):      # Newton on |r|^2 = d^2 along the old separations
            r = r0 + torch.einsum("wkl,wl,wla->wka", self.couple, g, ro)
            jac = 2.0 * self.couple * torch.einsum("wka,wla->wkl", r, ro)
            g = g - torch.linalg.solve(jac, ((r * r).sum(-1) - self.d2)[..., None])[..., 0]
        return self.push(x, g, ro), self.push(v, g / dt, ro)

    def hold_velocities(self, x, v):
        r = x[self.ci] - x[self.cj]
        rv = ((v[self.ci] - v[self.cj]) * r).sum(-1)
        g = torch.linalg.solve(self.couple * torch.einsum("wka,wla->wkl", r, r), -rv[..., None])[..., 0]
        return self.push(v, g, r)

    def flux(self, x, v, blocks, flux):
        """calheatf for rigid water with atom centres: [region, term, component]."""
        s = self.s
        reg = _regions(s, 0 if flux == "bulk" else int(flux), False)
        z1, z2 = self.t(reg["z1"]), self.t(reg["z2"])
        lz = float(s["box"][2])
        nreg, bulk = len(z1), flux == "bulk"
        cz = torch.where(x[:, 2] < 0, x[:, 2] + lz, torch.where(x[:, 2] >= lz, x[:, 2] - lz, x[:, 2]))
        e = torch.zeros(2, self.n, dtype=torch.float64, device="cuda")
        col = torch.zeros(2, nreg, 3, dtype=torch.float64, device="cuda")
        for i, j in blocks:
            r = self.image(x[i] - x[j])
            r2 = (r * r).sum(-1)
            d = torch.sqrt(r2)
            ec = self.q[i] * self.q[j] / d * (d <= s["rrcut"])
            eps, s6 = self.lj(i, j, r2)
            sv = 0.5 * (r * (v[i] + v[j])).sum(-1)
            for k, (en, fs) in enumerate(((ec, ec / r2), (eps * s6 * (s6 - 2.0), 12.0 * eps * s6 * (s6 - 1.0) / r2))):
                e[k].index_add_(0, i, 0.5 * en).index_add_(0, j, 0.5 * en)
                if bulk:
                    col[k, 0] += ((fs * sv)[:, None] * r).sum(0)
                    continue
                dz = cz[i] - cz[j]
                lo, hi = torch.minimum(cz[i], cz[j]), torch.maximum(cz[i], cz[j])
                push = torch.where(dz.abs() / lz < 0.5, fs * sv * torch.where(dz >= 0, 1.0, -1.0), torch.zeros_like(dz))
                for m in range(nreg):
                    col[k, m, 2] += (push * (torch.minimum(hi, z2[m]) - torch.maximum(lo, z1[m])).clamp_min(0.0)).sum()
        out = torch.zeros(nreg, abi.NHFJ, 3, dtype=torch.float64, device="cuda")
        kin = 0.5 * self.mass / md.MD_CONV * (v * v).sum(-1)
        vc = v if bulk else v * self.t([0.0, 0.0, 1.0])
        for m in range(nreg):
            inside = ((z1[m] <= cz) & (cz <= z2[m])).to(torch.float64)[:, None] * vc
            out[m, abi.HFJ_KIN] = (kin[:, None] * inside).sum(0)
            for k, name in enumerate(("elc", "vdw")):
                out[m, abi.HFJ_POT + abi.HF_NAMES.index(name)] = (e[k][:, None] * inside).sum(0)
                out[m, abi.HFJ_VIRI + abi.HF_NAMES.index(name)] = col[k, m]
            out[m] /= float(s["box"][0] * s["box"][1]) * (z2[m] - z1[m])
            out[m, abi.HFJ_TOT] = out[m, :abi.HFJ_TOT].sum(0)
        return out

    def kinetic(self, v):
        return 0.5 * (self.mass[:, None] * v * v).sum() / md.MD_CONV

    def trajectory(self, x, v, case):
        self.constraints()
        v = self.hold_velocities(x, v)
        inner = case.get("respa", 1)
        dts = DT_FS / inner
        flux = case.get("flux", "bulk")
        acc = (md.MD_CONV * self.minv)[:, None]
        chain = _Chain(3 * self.n - self.d2.numel() - 3) if case.get("nhc") else None
        blocks = [self.listed(x)]

        def forces():
            rec = self.calforce(x, blocks)
            if inner == 1:
                return None, rec["force"], rec["ene"][0]
            fb, parts, _ = self.bonded(x)
            short = fb - self.pair14(x)
            return short, rec["force"] - short, rec["ene"][0]

        def kick(v, f, dt):
            return chain.kick(v, f * acc) if chain else v + 0.5 * dt * acc * f

        def sample():
            ke = float(self.kinetic(v))
            return [ke, float(pot), ke + float(pot) + (chain.energy() if chain else 0.0)]

        short, long, pot = forces()
        rows, series = [sample()], [self.flux(x, v, blocks, flux)] if flux else []
        if chain:
            chain.move(float(self.kinetic(v)))
        for step in range(1, case["nstep"] + 1):
            for k in range(inner):
                if inner > 1 and k == 0:
                    v = v + 0.5 * DT_FS * acc * long
                v = kick(v, long if inner == 1 else short, dts)
                old, x = x, x + dts * v
                x, v = self.hold_positions(x, v, old, dts)
                if k == 0 and step % NSTEP_BOOK == 0:
                    blocks = [self.listed(x)]
                if inner == 1 or k == inner - 1:
                    short, long, pot = forces()
                else:
                    short = self.bonded(x)[0] - self.pair14(x)
                v = kick(v, long if inner == 1 else short, dts)
                if inner > 1 and k == inner - 1:
                    v = v + 0.5 * DT_FS * acc * long
                v = self.hold_velocities(x, v)
            if chain:
                chain.move(float(self.kinetic(v)))
            if step == case["nstep"]:
                rows.append(sample())
            if flux:
                series.append(self.flux(x, v, blocks, flux))
            if chain:
                chain.move(float(self.kinetic(v)))
        out = dict(pos=x, vel=v, energies=torch.tensor(rows, dtype=torch.float64))
        if flux:
            out["flux"] = torch.stack(series)
        return out

    def pair14(self, x):
        """The forces of the 1-4 pairs (long with RESPA), which bonded() holds too."""
        s, t = self.s, self.t
        f = torch.zeros_like(x)
        if not len(s["torsrb_type"]):
            return f
        tt = t(s["torsrb_type"], torch.int64) - 1
        ends = t(s["torsrb_ijkl"], torch.int64) - 1
        i, l = ends[:, 0], ends[:, 3]
        r = x[i] - x[l]
        r2 = (r * r).sum(1)
        k = self.type[i] * self.nt + self.type[l]
        s6 = (self.rm2.reshape(-1)[k] / r2) ** 3
        fs = 12.0 * self.eps.reshape(-1)[k] * s6 * (s6 - 1.0) / r2 / t(s["torsrb_divfac_vdw"])[tt]
        fs = fs + self.q[i] * self.q[l] / r2 ** 1.5 / t(s["torsrb_divfac_elc"])[tt]
        return f.index_add_(0, i, fs[:, None] * r).index_add_(0, l, -fs[:, None] * r)


class _Chain:
    """A Nose-Hoover chain of NHC_LINKS links (third-order Yoshida-Suzuki, one sub-step)."""

    def __init__(self, nfree):
        self.kt = md.KB_EREF * TEMPERATURE
        self.nkt = nfree * self.kt
        self.mass = [(self.nkt if i == 0 else self.kt) / NHC_FREQ ** 2 for i in range(NHC_LINKS)]
        self.x, self.v = [0.0] * NHC_LINKS, [0.0] * NHC_LINKS
        w = 1.0 / (2.0 - 2.0 ** (1.0 / 3.0))
        self.weights = (w, 1.0 - 2.0 * w, w)

    def move(self, kinetic):
        q, x, v, m = self.mass, self.x, self.v, NHC_LINKS
        g1 = (2.0 * kinetic - self.nkt) / q[0]
        pull = lambda i: (q[i - 1] * v[i - 1] ** 2 - self.kt) / q[i]      # noqa: E731
        for w in self.weights:
            h2 = w * DT_FS / 2.0
            h4, h8 = h2 / 2.0, h2 / 4.0

            def damp(i, g):
                e = math.exp(-h8 * v[i + 1])
                v[i] = v[i] * e * e + h4 * g * e
            v[m - 1] += pull(m - 1) * h4
            for i in range(m - 2, 0, -1):
                damp(i, pull(i))
            damp(0, g1)
            for i in range(m):
                x[i] += v[i] * h2
            damp(0, g1)
            for i in range(1, m - 1):
                damp(i, pull(i))
            v[m - 1] += pull(m - 1) * h4

    def kick(self, v, a):
        u = 0.25 * DT_FS * self.v[0]
        e = math.exp(-u)
        shape = 1.0 + u * u / 6.0 * (1.0 + u * u / 20.0 * (1.0 + u * u / 42.0 * (1.0 + u * u / 72.0)))
        return v * (e * e) + a * (e * shape * 0.5 * DT_FS)

    def energy(self):
        return sum(0.5 * m * v * v for m, v in zip(self.mass, self.v)) + self.nkt * self.x[0] + self.kt * sum(self.x[1:])


def exact(case, seed):
    """What run() returns, in 64 bits.  The heat flux of the slabs (bonded terms, molecule centres)
    and the per-atom arrays have no value here."""
    torch.set_grad_enabled(False)
    try:
        if case["kind"] == "ensemble":
            return [_host(_Plain(s, e).trajectory(torch.as_tensor(s["pos"], device="cuda"), torch.as_tensor(v, device="cuda"), case))
                    for s, e, v in _replicas(case, seed)]
        s, excl, vel = _fluid(case, seed)
        plain = _Plain(s, excl)
        x = torch.as_tensor(s["pos"], device="cuda")
        if case["kind"] == "md":
            return _host(plain.trajectory(x, torch.as_tensor(vel, device="cuda"), case))
        out = dict(_host(plain.calforce(x)))
        if case["kind"] == "heatf":
            out["hf"] = None
        if case["kind"] == "hf_arrays":
            out.update(pot_atm=None, viri_atm=None, hf=None)
        return out
    finally:
        torch.set_grad_enabled(True)


def _host(out):
    return {k: v.cpu().numpy() for k, v in out.items()}
