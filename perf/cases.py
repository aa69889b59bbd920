"""The calls this engine is timed on: map sets, an ensemble, the
differentiable mode and ligand scoring, from the smallest docking box to a
blind-docking one.

A case is a dict of plain values.  ``prepare`` builds what a program holds
before the call (a parsed receptor, a plan, a scorer, output buffers),
``run`` makes the call, ``work`` states its algorithmic bytes and FLOPs, and
``exact`` gives the same outputs in FP64 from torch alone.

Receptors are seeded globules at protein density (0.068 atoms / A^3, polar
hydrogens included, the atom mix of the x1hpv receptor): residue-sized chains
with bonds of 1.0 to 1.8 A on a jittered lattice, so donors, carbonyl,
hydroxyl and ring acceptors all get the bond vectors a protein gives them.
They go through a PDBQT file and a GPF as a user's receptor does.
"""
from __future__ import annotations

import dataclasses
import math
import os
import tempfile

import torch  # first: one HIP runtime for torch and the engine

import numpy as np

import autogrid_amd as ag
from autogrid_amd import fit, synth
from autogrid_amd.poses import make_poses

DENSITY = 0.068          # receptor atoms per A^3
LIGAND_TYPES = ["C", "A", "HD", "OA", "N", "NA", "SA", "S", "F", "Cl", "Br", "I", "P"]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _case(name, kind, atoms, nx, ny, nz, types, spacing=0.375, dielectric="distance", centre=0.0, poses=0,
          conformations=0):
    """nx ny nz: GPF npts (one fewer than the points per axis); types: affinity
    maps, the first of LIGAND_TYPES; centre: box centre along x from the
    receptor's, in receptor radii."""
    return {"name": name, "kind": kind, "atoms": atoms, "nx": nx, "ny": ny, "nz": nz, "types": types,
            "spacing": spacing, "dielectric": dielectric, "centre": centre, "poses": poses,
            "conformations": conformations}


def listed():
    return [
        # A docking box around one site of a small domain: the smallest call
        # of a screening program that keeps its plan, where launches count.
        _case("site", "plan", 1000, 40, 40, 40, 6, centre=0.5),
        # AutoDock's default box (npts 60) on a protein the size of x1hpv
        # with its map set of 11 ligand types: the everyday grid run.
        _case("pocket", "plan", 1849, 60, 60, 60, 11, centre=0.4),
        # The headline benchmark's shape: 5,000 atoms, 127^3 points, 13 types.
        _case("whole", "plan", 5000, 126, 126, 126, 13),
        # Blind docking over a large receptor: 20,000 atoms, 257^3 points.
        _case("blind", "plan", 20000, 256, 256, 256, 13),
        # A long, flat, fine box over a groove: no edge a multiple of a
        # tile, 0.25 A spacing, a few ligand types.
        _case("groove", "plan", 2743, 46, 82, 118, 4, spacing=0.25, centre=0.6),
        # Floating and constriction grids beside the maps, with a constant
        # dielectric, on an ordinary box.
        _case("grids", "grids", 3000, 80, 80, 80, 6, dielectric="constant"),
        # The Vina potential on the headline box: table sums only.
        _case("vina", "vina", 5000, 126, 126, 126, 13),
        # One receptor from host arrays to maps in pinned host memory: what a
        # program that sees each receptor once calls.
        _case("host", "host", 1849, 80, 80, 80, 6, centre=0.4),
        # Receptor conformations of ensemble docking in one resident batch.
        _case("ensemble", "batch", 6000, 80, 80, 80, 6, conformations=12),
        # One step of fitting the differentiable maps to 256 poses: forward,
        # scores, both adjoints (the analytic benchmark's shape).
        _case("fit", "fit", 5000, 64, 64, 64, 5, poses=256),
        # The same step on a site box, as a per-site refit runs it.
        _case("fit_site", "fit", 1000, 40, 40, 40, 5, centre=0.5, poses=64),
        # One step of minimising 256 poses in resident maps: new positions,
        # scores and the gradient on every ligand atom.
        _case("dock", "dock", 1849, 64, 64, 64, 6, centre=0.4, poses=256),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["plan"] * 6 + ["grids", "vina", "host", "batch", "fit", "fit", "dock"])
    fitted = kind in ("fit", "dock")
    atoms = int(_log_uniform(rng, 600, 6000 if fitted or kind == "batch" else 12000))
    edge = _log_uniform(rng, *((40, 72) if fitted else (30, 100 if kind == "batch" else 170)))
    n = [2 * int(edge * rng.uniform(0.75, 1.25) / 2) for _ in range(3)]
    types = rng.randint(3, 8) if kind == "fit" else rng.randint(3, 13)
    return {"kind": kind, "atoms": atoms, "nx": n[0], "ny": n[1], "nz": n[2], "types": types,
            "spacing": rng.choice([0.375, 0.375, 0.375, 0.25, 0.3, 0.5]),
            "dielectric": rng.choice(["distance"] * 4 + ["constant"]),
            "centre": round(rng.uniform(0.0, 0.8), 2),
            "poses": rng.randint(16, 384) if fitted else 0,
            "conformations": rng.randint(2, 10) if kind == "batch" else 0}


# ---------------------------------------------------------------------------
# receptors
# ---------------------------------------------------------------------------

# (parent, bond length, type, charge) per atom; the backbone first
_BACKBONE = [(-1, 0.0, "N", -0.35), (0, 1.01, "HD", 0.16), (0, 1.46, "C", 0.16), (2, 1.53, "C", 0.24),
             (3, 1.23, "OA", -0.27)]
_CB = (2, 1.53, "C", 0.04)
_SIDE = [
    (0.0, []), (0.0, [_CB]), (0.0, [_CB, (5, 1.43, "OA", -0.40), (6, 0.96, "HD", 0.21)]),
    (-1.0, [_CB, (5, 1.52, "C", 0.17), (6, 1.25, "OA", -0.65), (6, 1.25, "OA", -0.65)]),
    (0.0, [_CB, (5, 1.52, "C", 0.27), (6, 1.23, "OA", -0.27), (6, 1.33, "N", -0.37), (8, 1.01, "HD", 0.16),
           (8, 1.01, "HD", 0.16)]),
    (1.0, [_CB, (5, 1.52, "C", 0.03), (6, 1.52, "C", 0.03), (7, 1.49, "N", -0.08), (8, 1.01, "HD", 0.27),
           (8, 1.01, "HD", 0.27), (8, 1.01, "HD", 0.27)]),
    (0.0, [_CB, (5, 1.53, "C", 0.0), (6, 1.53, "C", 0.01), (6, 1.53, "C", 0.01)]),
    (0.0, [_CB, (5, 1.51, "A", -0.05), (6, 1.39, "A", 0.0), (6, 1.39, "A", 0.0), (7, 1.39, "A", 0.0),
           (8, 1.39, "A", 0.0)]),
    (0.0, [_CB, (5, 1.50, "A", 0.08), (6, 1.38, "N", -0.33), (7, 1.01, "HD", 0.17), (6, 1.38, "NA", -0.25)]),
    (0.0, [_CB, (5, 1.52, "C", 0.08), (6, 1.80, "SA", -0.17), (7, 1.79, "C", 0.09)]),
]
_SIDE_P = np.array([8, 14, 12, 12, 9, 12, 18, 8, 3, 4.0])


def _receptor(n_atoms, rng):
    """(coord [n, 3], types [n], charges [n], radius): residues on the
    lattice sites nearest the origin, each grown atom by atom in the
    direction (of 24 drawn) that keeps farthest from its other atoms."""
    mean = float(np.dot(_SIDE_P / _SIDE_P.sum(), [5 + len(s) for _, s in _SIDE]))
    a = (mean / DENSITY) ** (1.0 / 3.0)
    n_res = int(n_atoms / 5) + 1
    m = int(math.ceil((n_res * 0.75 / math.pi) ** (1.0 / 3.0))) + 2
    site = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.25
    site = site[np.argsort((site ** 2).sum(1), kind="stable")[:n_res]]
    kind = rng.choice(len(_SIDE), size=n_res, p=_SIDE_P / _SIDE_P.sum())
    kind[0] = 2
    n_of = np.array([5 + len(s) for _, s in _SIDE])[kind]
    keep = int(np.searchsorted(np.cumsum(n_of), n_atoms)) + 1     # residues that give n_atoms
    order = np.lexsort((site[:keep, 0], site[:keep, 1], site[:keep, 2]))
    site, kind = site[:keep][order] * a + rng.uniform(-0.5, 0.5, (keep, 3)), kind[:keep][order]
    width = 5 + max(len(s) for _, s in _SIDE)
    xyz = np.full((keep, width, 3), np.nan)
    typ = np.full((keep, width), "", dtype="<U2")
    chg = np.zeros((keep, width))
    for k, (net, side) in enumerate(_SIDE):
        rows = np.flatnonzero(kind == k)
        if not rows.size:
            continue
        atoms = _BACKBONE + side
        p = np.zeros((rows.size, len(atoms), 3))
        p[:, 0] = site[rows] + rng.normal(0.0, 0.3, (rows.size, 3))
        for j in range(1, len(atoms)):
            parent, length = atoms[j][0], atoms[j][1]
            d = rng.normal(size=(rows.size, 24, 3))
            d *= length / np.linalg.norm(d, axis=2, keepdims=True)
            cand = p[:, parent, None, :] + d
            others = [i for i in range(j) if i != parent]
            gap = np.full(cand.shape[:2], 9.0)
            for i in others:
                gap = np.minimum(gap, np.linalg.norm(cand - p[:, i, None, :], axis=2))
            gap = np.minimum(gap, 2.4) - 0.35 * np.linalg.norm(cand - site[rows][:, None, :], axis=2)
            p[:, j] = cand[np.arange(rows.size), np.argmax(gap, axis=1)]
        q = np.array([t[3] for t in atoms])[None, :] + rng.normal(0.0, 0.03, (rows.size, len(atoms)))
        q += (net - q.sum(1, keepdims=True)) / len(atoms)
        xyz[rows, :len(atoms)], chg[rows, :len(atoms)] = p, q
        typ[rows, :len(atoms)] = [t[2] for t in atoms]
    use = typ.reshape(-1) != ""
    return (xyz.reshape(-1, 3)[use][:n_atoms], typ.reshape(-1)[use][:n_atoms], chg.reshape(-1)[use][:n_atoms],
            (n_atoms / DENSITY * 0.75 / math.pi) ** (1.0 / 3.0))


def _state(case, rng):
    """PreparedState of the case's receptor, box and map set, read by the
    front end from the PDBQT and GPF a user would write."""
    coord, types, charges, radius = _receptor(case["atoms"], rng)
    rec_types = list(dict.fromkeys(types.tolist()))
    centre = np.round([case["centre"] * radius, 0.0, 0.0], 3)
    extra = ["constriction_distance_cutoff 6.5", "fmap r.f.map", "cmap r.c.map"] if case["kind"] == "grids" else []
    cwd = os.getcwd()
    with tempfile.TemporaryDirectory(prefix="agcase_") as d:
        synth.write_pdbqt(os.path.join(d, "r.pdbqt"), coord, types, charges)
        gpf = os.path.join(d, "r.gpf")
        synth.write_gpf(gpf, "r", "r.pdbqt", rec_types, LIGAND_TYPES[:case["types"]],
                        (case["nx"], case["ny"], case["nz"]), centre, spacing=case["spacing"], extra=extra)
        if case["dielectric"] == "constant":
            with open(gpf) as f:
                text = f.read()
            with open(gpf, "w") as f:
                f.write(text.replace("dielectric -0.1465", "dielectric 4.0"))
        os.chdir(d)
        try:
            job = ag.Job("r.gpf")
            return (job.prepare_vina() if case["kind"] == "vina" else job.prepare()).state()
        finally:
            os.chdir(cwd)


def _conformations(case, rng):
    """The case's ensemble: conformations of one receptor with 25 to 100 % of
    its atoms and boxes of half to one and a half the case's edges (both the
    case's own), Gaussian jitter."""
    base = _state(case, rng)
    size = np.random.default_rng([case["atoms"], case["nx"], case["conformations"]])
    out = []
    for _ in range(case["conformations"]):
        n = max(300, int(base.n_atoms * size.uniform(0.25, 1.0)))
        first = int(rng.integers(0, base.n_atoms - n + 1))
        part = slice(first, first + n)
        move = np.repeat(rng.normal(0.0, 0.4, (n // 8 + 1, 3)), 8, axis=0)[:n]
        coord = base.coord[part] + move + rng.normal(0.0, 0.02, (n, 3))
        npts = [2 * int(case[k] * size.uniform(0.5, 1.5) / 2) for k in ("nx", "ny", "nz")]
        out.append(dataclasses.replace(
            base, coord=coord - coord.mean(0), charge=base.charge[part], vol=base.vol[part],
            solpar=base.solpar[part], type=base.type[part], hbond=base.hbond[part], rexp=base.rexp[part],
            rvector=base.rvector[part], rvector2=base.rvector2[part], disorder=base.disorder[part],
            n1=tuple(k + 1 for k in npts), ne=tuple(k // 2 for k in npts), _keep=[]))
    return ag.bond_vectors_batch(out)


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------

_context = None


def _ctx():
    global _context
    if _context is None:
        torch.cuda.init()
        _context = ag.Context(0)
    return _context


def _grid(st):
    return (st.n1[2], st.n1[1], st.n1[0])


def _split(st, maps):
    """A map set by what its maps are: affinity maps, e and d."""
    m = st.n_atom_maps
    return {"affinity": maps[:m], "e": maps[st.elec_index], "d": maps[st.dsolv_index]}


def _poses(case, st, seed):
    """Seeded poses of 20 to 60 atoms; how many atoms each has is the case's."""
    lig = {LIGAND_TYPES[k]: k for k in range(case["types"])}
    count = np.random.default_rng(case["poses"]).integers(20, 61, case["poses"])
    full = make_poses(st, lig, n_poses=case["poses"], seed=seed, atoms_range=(60, 60))
    return [tuple(a[:n] for a in pose) for n, pose in zip(count, full)]


def _inputs(case, seed):
    """The seeded host inputs alone (prepare puts them on the GPU; exact
    starts from the same ones)."""
    rng = np.random.default_rng([int(seed), 977])
    if case["kind"] == "batch":
        return {"states": _conformations(case, rng)}
    s = {"st": _state(case, rng)}
    if case["kind"] in ("fit", "dock"):
        s["poses"] = _poses(case, s["st"], int(seed))
    if case["kind"] == "fit":
        s["target"] = rng.normal(-4.0, 3.0, case["poses"]).astype(np.float32)
        s["scale"] = rng.uniform(0.8, 1.2, 4)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = kind = case["kind"]
    ctx = _ctx()
    if kind == "batch":
        s["plan"] = ctx.batch(s["states"], tune={"cell_size": 4.0, "cube": True})
        s["maps"] = torch.empty(s["plan"].map_floats, dtype=torch.float32, device="cuda")
        return s
    st = s["st"]
    if kind == "host":
        s["out"] = torch.empty((st.n_maps,) + _grid(st), dtype=torch.float32, pin_memory=True).numpy()
        return s
    if kind == "fit":
        s["engine"] = ag.Analytic(ctx, st)
        s["scorer"] = fit.PoseScorer(ctx, st, s["poses"])
        e = s["engine"]
        s["par"] = [torch.tensor(np.asarray(a), dtype=torch.float32).requires_grad_() for a in
                    (st.coord, st.charge, e.rij0, e.eps0, e.weights0 * s["scale"])]
        s["goal"] = torch.from_numpy(s["target"]).cuda()
        return s
    if kind == "dock":
        s["maps"] = _docking_maps(st, seed)
        s["scorer"] = ag.Scorer(ctx, st, s["poses"])
        # the minimiser's step away from the poses the scorer was made with
        s["xyz"] = _moved(s["poses"], seed)
        s["scores"] = torch.empty(len(s["poses"]), dtype=torch.float32, device="cuda")
        s["grad"] = torch.empty((s["scorer"].n_atoms, 3), dtype=torch.float32, device="cuda")
        return s
    s["maps"] = torch.empty((st.n_maps,) + _grid(st), dtype=torch.float32, device="cuda")
    if kind == "grids":
        s["fmap"] = torch.empty(_grid(st), dtype=torch.float32, device="cuda")
        s["cmap"] = torch.empty(_grid(st), dtype=torch.int32, device="cuda")
    s["plan"] = ctx.plan(st, potential=ag.AG_POTENTIAL_VINA if kind == "vina" else ag.AG_POTENTIAL_AD4)
    return s


def _docking_maps(st, seed):
    """Maps a minimiser reads, already on the GPU: wells of a few kcal/mol
    and, at every eighth point (inside the receptor), clashes up to 1e5."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 17)
    shape = (st.n_maps,) + _grid(st)
    u = torch.rand(shape, device="cuda", generator=g)
    return torch.where(u < 0.125, 10.0 ** (40.0 * u), torch.randn(shape, device="cuda", generator=g) - 0.5)


def _moved(poses, seed):
    rng = np.random.default_rng([int(seed), 311])
    xyz = np.concatenate([p[2] for p in poses])
    return xyz + rng.normal(0.0, 0.2, xyz.shape)


def run(s):
    kind = s["kind"]
    if kind == "batch":
        s["plan"].execute(s["maps"].data_ptr())
        out = []
        for i, st in enumerate(s["states"]):
            o = int(s["plan"].map_offsets[i])
            out.append(_split(st, s["maps"][o:o + st.n_maps * st.points].view((st.n_maps,) + _grid(st))))
        return out
    if kind == "host":
        return _split(s["st"], _ctx().maps_plain(s["st"], out=s["out"]))
    if kind == "fit":
        for p in s["par"]:
            p.grad = None
        maps = fit.AnalyticMaps.apply(*s["par"], s["engine"])
        scores = s["scorer"](maps)
        loss = torch.mean(((scores - s["goal"]) / (1.0 + s["goal"].abs() + scores.detach().abs())) ** 2)
        loss.backward()
        return {**_split(s["st"], maps.detach()), "scores": scores.detach(),
                "grad": dict(zip(("coord", "charge", "rij", "eps", "weights"), [p.grad for p in s["par"]]))}
    if kind == "dock":
        s["scorer"].set_positions(s["xyz"])
        s["scorer"].score(s["maps"].data_ptr(), s["scores"].data_ptr(), s["grad"].data_ptr())
        return {"scores": s["scores"], "grad": s["grad"]}
    if kind == "grids":
        s["plan"].execute(s["maps"].data_ptr(), s["fmap"].data_ptr(), s["cmap"].data_ptr())
        return {**_split(s["st"], s["maps"]), "fmap": s["fmap"], "cmap": s["cmap"]}
    s["plan"].execute(s["maps"].data_ptr())
    return _split(s["st"], s["maps"])


def work(case):
    """Bytes: the receptor (96 bytes an atom), the pair tables and every map
    written once.  FLOPs, as the reference forms a map set: 16 per (point,
    atom) pair of the e map, 16 + 4 per affinity map + 2 for d per pair within
    8 A (atoms at DENSITY, where the 8 A sphere meets the receptor); the
    adjoint of the fit counts the map set's again, over the fifth of the
    points its poses touch.  A ligand atom reads 24 map values and writes its
    gradient."""
    n, m = case["atoms"], case["types"]
    p = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    h, r = case["spacing"], (n / DENSITY * 0.75 / math.pi) ** (1.0 / 3.0)
    if case["kind"] == "dock":
        a = 40 * case["poses"]
        return {"bytes": a * (24 * 4 + 24 + 12 + 8), "flops": a * 8 * 20}
    inside = min(1.0, 4.0 / 3.0 * math.pi * (r + 4.0) ** 3 / (p * h ** 3))
    near = p * inside * DENSITY * 4.0 / 3.0 * math.pi * 512.0
    b = 96 * n + 7 * m * 4096 + 4 * p * (m + 2) + (8 * p if case["kind"] == "grids" else 0)
    f = near * (2 * m if case["kind"] == "vina" else 16 + 4 * m + 2) + (0 if case["kind"] == "vina" else 16.0 * p * n)
    if case["kind"] == "grids":
        f += 6.0 * p * n
    if case["kind"] == "batch":
        b, f = case["conformations"] * b, case["conformations"] * 0.625 * f
    if case["kind"] == "fit":
        b, f = 2 * b, 1.2 * f
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same outputs in FP64
# ---------------------------------------------------------------------------

DS, D1, AS, A1, A2, AD = 1, 2, 3, 4, 5, 6        # H-bond classes of the state


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(dtype)


def _axes(st):
    return [(torch.arange(st.n1[d], device="cuda", dtype=torch.float64) - st.ne[d]) * st.spacing for d in range(3)]


def _e_fmap_cmap(st, charge, eps_of):
    """The sums over every atom: e, the floating grid's distance and the
    constriction count; eps_of(r) is 332 / eps."""
    x = _t(st.coord)
    ax = _axes(st)
    P, N, nx = st.points, st.n_atoms, st.n1[0]
    e = torch.empty(P, dtype=torch.float64, device="cuda")
    f = torch.empty(P, dtype=torch.float64, device="cuda") if st.floating_grid else None
    c = torch.empty(P, dtype=torch.int32, device="cuda") if st.constriction_grid else None
    dx2 = (x[None, :, 0] - ax[0][:, None]).square()
    step = max(1, int(2e8) // (nx * N))
    for a in range(0, P // nx, step):            # rows of points along x
        row = torch.arange(a, min(P // nx, a + step), device="cuda")
        dyz2 = (x[None, :, 1] - ax[1][row % st.n1[1]][:, None]).square()
        dyz2 += (x[None, :, 2] - ax[2][row // st.n1[1]][:, None]).square()
        r = (dx2[None] + dyz2[:, None, :]).sqrt_().view(-1, N)
        i = slice(a * nx, a * nx + len(r))
        if f is not None:
            f[i] = r.amin(1).clamp_(min=1e-6)
        if c is not None:
            c[i] = (r <= st.constriction_cutoff).sum(1).to(torch.int32)
        e[i] = eps_of(r).div_(r.clamp_(min=0.5)) @ charge
    return e, f, c


def _closest_h(st, limit=None):
    """Index of each point's nearest donor hydrogen (-1 past `limit`)."""
    hb = _t(st.hbond, torch.int64)
    idx = torch.nonzero((hb == DS) | (hb == D1)).reshape(-1)
    x = _t(st.coord)[idx]
    ax = _axes(st)
    out = torch.empty(st.points, dtype=torch.int64, device="cuda")
    step = max(1, int(1.5e8) // max(len(idx), 1))
    for a in range(0, st.points, step):
        i = torch.arange(a, min(st.points, a + step), device="cuda")
        pt = (ax[0][i % st.n1[0]], ax[1][(i // st.n1[0]) % st.n1[1]], ax[2][i // (st.n1[0] * st.n1[1])])
        r = sum((x[None, :, d] - pt[d][:, None]).square_() for d in range(3)).sqrt_()
        v, k = r.min(1)
        out[i] = idx[k] if limit is None else torch.where(v < limit, idx[k], torch.full_like(k, -1))
    return out


def _pairs_within_8(st, coord):
    """Batches of (point index, atom index, r, unit vector) of the pairs
    within 8 A; coord may carry a gradient."""
    h = st.spacing
    w = int(math.ceil(8.0 / h)) + 1
    off = torch.arange(-w, w + 1, device="cuda")
    ax = _axes(st)
    n1 = torch.tensor(st.n1, device="cuda")
    base = torch.round(coord.detach() / h).long() + torch.tensor(st.ne, device="cuda")
    step = max(1, int(6e6) // (2 * w + 1) ** 3)
    for a in range(0, st.n_atoms, step):
        at = torch.arange(a, min(st.n_atoms, a + step), device="cuda")
        ok, sq = [], []
        for d in range(3):
            k = base[at, d][:, None] + off
            ok.append((k >= 0) & (k < n1[d]))
            sq.append((coord.detach()[at, d][:, None] - ax[d][k.clamp(0, st.n1[d] - 1)]).square())
        r2 = sq[0][:, None, None, :] + sq[1][:, None, :, None] + sq[2][:, :, None, None]
        m = (r2 <= 64.0) & ok[0][:, None, None, :] & ok[1][:, None, :, None] & ok[2][:, :, None, None]
        ia, kz, ky, kx = torch.nonzero(m, as_tuple=True)
        if not len(ia):
            continue
        ia = at[ia]
        g = [base[ia, d] + off[k] for d, k in enumerate((kx, ky, kz))]
        delta = torch.stack([coord[ia, d] - ax[d][g[d]] for d in range(3)], 1)
        r = (delta[:, 0] ** 2 + delta[:, 1] ** 2 + delta[:, 2] ** 2).sqrt()
        yield g[0] + st.n1[0] * (g[1] + st.n1[1] * g[2]), ia, r, delta / r.clamp(min=1e-6)[:, None]


def _directional(st, ia, dn, rv, rv2, closest):
    """racc, rdon and Hramp of pairs of ordered atoms."""
    hb, rexp = _t(st.hbond, torch.int64)[ia], _t(st.rexp, torch.int64)[ia]
    one = torch.ones(len(ia), dtype=torch.float64, device="cuda")
    v, v2 = rv[ia], rv2[ia]
    c = -(dn * v).sum(1)
    power = torch.where(rexp == 2, c ** 2, torch.where(rexp == 4, c ** 4, c))
    racc = torch.where(hb == D1, torch.where(c > 0, power, 0 * c), one)
    ct = (rv[closest.clamp(min=0)] * v).sum(1).clamp(-1, 1)
    ramp = 0.5 - 0.5 * torch.cos(torch.acos(ct) * (120.0 / 90.0))
    hramp = torch.where((hb == D1) & (c > 0) & (closest != ia) & (closest >= 0), ramp, one)
    t0 = math.pi / 2 - torch.acos((dn * v2).sum(1).clamp(-1, 1))
    cross = torch.linalg.cross(dn, v2)
    ti = (cross * v).sum(1) / (cross ** 2).sum(1).clamp(min=1e-6).sqrt()
    ti = (torch.acos(ti.clamp(-1, 1)) - math.pi / 2).abs()
    lone = torch.where(c >= 0, (0.9 + 0.1 * torch.sin(2 * ti)) * torch.cos(t0),
                       torch.where(c >= -0.34202, 562.25 * (0.116978 - c ** 2) ** 3 * torch.cos(t0), 0 * c))
    rdon = torch.where(hb == A1, torch.where(c > 0, c ** 2, 0 * c), torch.where(hb == A2, lone, one))
    return racc, rdon, hramp


def _cases_of(map_desc):
    """Per atom class 0..6: 0 plain, 1 acceptor probe, 2 / 3 the min / max
    mix with racc / rdon."""
    mh = int(map_desc["hbond"])
    out = []
    for ah in range(7):
        donor = ah in (DS, D1, AD)
        k = 0
        if map_desc["is_hbonder"]:
            if mh in (AS, A2, AD) and donor:
                k = 1
            elif mh in (A1, AD) and donor:
                k = 2
            elif mh in (DS, D1, AD) and ah > 2:
                k = 3
        out.append(k)
    return torch.tensor(out, device="cuda")


def _affinity_terms(st, m, e, ia, racc, rdon, hramp):
    """(summed term, term of the min / max mix, where the mix applies) of
    map m's pair energies e."""
    k = _cases_of(st.maps[m])[_t(st.hbond, torch.int64)[ia]]
    ramp = (e / 100.0).clamp(0, 1)
    acc = e * hramp * (racc + (1 - racc) * ramp)
    f = torch.where(k == 2, racc, rdon)
    return torch.where(k == 0, e, torch.where(k == 1, acc, 0 * e)), e * (f + (1 - f) * ramp), k >= 2


def _near_maps(st, vina):
    """Affinity maps and d of the table model."""
    M, P = st.n_atom_maps, st.points
    x, rv, rv2 = _t(st.coord), _t(st.rvector), _t(st.rvector2)
    tab, sol = _t(st.e_vdw_hb), _t(st.sol_fn)
    typ, vol, q = _t(st.type, torch.int64), _t(st.vol), _t(st.charge)
    solq = _t(st.solpar) + st.solpar_q * q.abs()
    aff = torch.zeros((M, P), dtype=torch.float64, device="cuda")
    lo, hi = torch.full_like(aff, 999999.0), torch.full_like(aff, -999999.0)
    d = torch.zeros(P, dtype=torch.float64, device="cuda")
    near_h = None if vina else _closest_h(st)
    for pt, ia, r, dn in _pairs_within_8(st, x):
        b = (r * 128.0).long()
        rows = tab[typ[ia], :, b.clamp(max=1023)]
        if vina:
            aff.index_add_(1, pt, rows.t().contiguous())
            continue
        dirs = _directional(st, ia, dn, rv, rv2, near_h[pt])
        s = sol[b.clamp(max=1024)]
        d.index_add_(0, pt, st.solpar_q * vol[ia] * s)
        for m in range(M):
            term, v, mixed = _affinity_terms(st, m, rows[:, m], ia, *dirs)
            des = (st.maps[m]["solpar_probe"] * vol[ia] + st.maps[m]["vol_probe"] * solq[ia]) * s
            aff[m].index_add_(0, pt, term + des)
            lo[m].scatter_reduce_(0, pt[mixed], v[mixed], "amin")
            hi[m].scatter_reduce_(0, pt[mixed], v[mixed], "amax")
    return aff + torch.where(lo < 999999.0, lo + hi.clamp(min=0), torch.zeros_like(lo)), d


def _exact_maps(st, vina=False):
    grid = _grid(st)
    aff, d = _near_maps(st, vina)
    if vina:
        e, f, c = torch.zeros(st.points, dtype=torch.float64, device="cuda"), None, None
    elif float(st.points) * st.n_atoms > 4e11:
        e = f = c = None         # over 20 s of FP64
    else:
        eps = _t(st.r_eps) if st.dddiel else torch.full((8192,), st.inv_diel_cal, dtype=torch.float64, device="cuda")
        e, f, c = _e_fmap_cmap(st, _t(st.charge) * st.coeff_estat,
                               lambda r: eps[(r * 128.0).long().clamp_(max=8191)])
    out = {"affinity": aff.view((st.n_atom_maps,) + grid), "e": None if e is None else e.view(grid), "d": d.view(grid)}
    if st.floating_grid:
        out.update(fmap=f.view(grid), cmap=c.view(grid))
    return out


def _trilinear(st, maps, poses, xyz):
    """(scores, per-atom gradient) of poses in maps [n_maps, P]; an atom off
    the grid scores 0."""
    mi = _t(np.concatenate([p[0] for p in poses]), torch.int64)
    q = _t(np.concatenate([p[1] for p in poses]))
    pose = torch.cat([torch.full((len(p[0]),), k, device="cuda") for k, p in enumerate(poses)])
    g = xyz / st.spacing + _t(st.ne)
    n1 = torch.tensor(st.n1, device="cuda")
    on = ((g >= 0) & (g < n1 - 1)).all(1)
    i0 = torch.floor(torch.where(on[:, None], g, torch.zeros_like(g)))
    f = g - i0
    i0 = i0.long()
    e = torch.zeros(len(q), dtype=torch.float64, device="cuda")
    grad = torch.zeros((len(q), 3), dtype=torch.float64, device="cuda")
    for c in range(8):
        k = [c & 1, (c >> 1) & 1, c >> 2]
        pt = (i0[:, 0] + k[0]) + st.n1[0] * ((i0[:, 1] + k[1]) + st.n1[1] * (i0[:, 2] + k[2]))
        v = maps[mi, pt] + q * maps[st.elec_index, pt] + q.abs() * maps[st.dsolv_index, pt]
        w = [f[:, d] if k[d] else 1 - f[:, d] for d in range(3)]
        e = e + w[0] * w[1] * w[2] * v
        for d in range(3):
            grad[:, d] += (1.0 if k[d] else -1.0) / st.spacing * w[(d + 1) % 3] * w[(d + 2) % 3] * v.detach()
    scores = torch.zeros(len(poses), dtype=torch.float64, device="cuda").index_add(0, pose, torch.where(on, e, 0 * e))
    return scores, grad * on[:, None]


class _Model:
    """The differentiable model's closed forms (map energies at the exact
    distance, switched off from 7.5 to 8 A)."""

    def __init__(self, st, par):
        self.st = st
        self.charge, self.rij, self.eps, self.w = par
        self.rv, self.rv2, self.typ = _t(st.rvector), _t(st.rvector2), _t(st.type, torch.int64)
        self.half = math.floor(st.r_smooth * 64.0) / 128.0
        self.hb = _t(st.pairs["hbonder"], torch.int64) > 0
        self.ab = [_t(st.pairs[k]) for k in ("xA", "xB")]

    def pair_terms(self, ia, r):
        """(switch, [energy of each map], desolvation Gaussian) of pairs."""
        u = ((r - 7.5) * 2.0).clamp(0, 1)
        s = 1 - u ** 3 * (10 - 15 * u + 6 * u ** 2)
        t = self.typ[ia]
        out = []
        for m in range(self.st.n_atom_maps):
            R, a, b = self.rij[m][t], self.ab[0][m][t], self.ab[1][m][t]
            eps = (self.eps[m] * torch.where(self.hb[m], self.w[1], self.w[0]))[t]
            x = torch.where(r < R - self.half, r + self.half, torch.where(r > R + self.half, r - self.half, R))
            e = eps / (a - b) * (b * (R / x) ** a - a * (R / x) ** b)
            out.append(e.clamp(max=1e5) * s)
        return out, self.w[3] * torch.exp(-r ** 2 / 25.92) * s

    def eps_of(self, r):
        if not self.st.dddiel:
            return torch.full_like(r, self.st.inv_diel_cal)
        b = 78.4 + 8.5525
        return 332.0 / (-8.5525 + b / (1.0 + 7.7839 * torch.exp(-0.003627 * b * r)))


def _exact_fit(s):
    """Maps, scores and the gradients of the loss.  The coordinates' gradient
    has no value here: it also runs through the bond vectors."""
    st, poses = s["st"], s["poses"]
    M, P, grid = st.n_atom_maps, st.points, _grid(st)
    w0 = np.asarray(st.weights, np.float64)
    wk = np.where(st.pairs["hbonder"] > 0, w0[1], w0[0])
    f32 = [np.asarray(a, np.float32) for a in (st.coord, st.charge, st.pairs["Rij"], st.pairs["eps"] / wk,
                                               w0 * s["scale"])]
    coord = f32[0].astype(np.float64)
    rexp, rv, rv2, _ = ag.bond_vectors(st, coord, st.type, st.hbond)
    st = dataclasses.replace(st, coord=coord, rexp=rexp, rvector=rv, rvector2=rv2, _keep=[])
    par = [_t(a).requires_grad_() for a in f32[1:]]
    model = _Model(st, par)
    vol, solpar = _t(st.vol), _t(st.solpar)
    near_h = _closest_h(st, 8.0)

    def batch_terms(pt, ia, r, dn):
        energies, g = model.pair_terms(ia, r)
        dirs = _directional(st, ia, dn, model.rv, model.rv2, near_h[pt])
        solq = solpar[ia] + st.solpar_q * model.charge[ia].abs()
        for m in range(M):
            des = (st.maps[m]["solpar_probe"] * vol[ia] + st.maps[m]["vol_probe"] * solq) * g
            yield (*_affinity_terms(st, m, energies[m], ia, *dirs), des)
        yield st.solpar_q * vol[ia] * g

    x = _t(st.coord)
    maps = torch.zeros((M + 2, P), dtype=torch.float64, device="cuda")
    lo = torch.full((M, P), 999999.0, dtype=torch.float64, device="cuda")
    hi = torch.full_like(lo, -999999.0)
    with torch.no_grad():
        for pt, ia, r, dn in _pairs_within_8(st, x):
            for m, t in enumerate(batch_terms(pt, ia, r, dn)):
                if m == M:
                    maps[st.dsolv_index].index_add_(0, pt, t)
                    continue
                maps[m].index_add_(0, pt, t[0] + t[3])
                lo[m].scatter_reduce_(0, pt[t[2]], t[1][t[2]], "amin")
                hi[m].scatter_reduce_(0, pt[t[2]], t[1][t[2]], "amax")
        maps[:M] += torch.where(lo < 999999.0, lo + hi.clamp(min=0), torch.zeros_like(lo))
        maps[st.elec_index] = _e_fmap_cmap(st, model.charge * model.w[2], model.eps_of)[0]
    maps.requires_grad_()
    scores, _ = _trilinear(st, maps, poses, _t(np.concatenate([p[2] for p in poses])))
    goal = _t(s["target"])
    torch.mean(((scores - goal) / (1.0 + goal.abs() + scores.detach().abs())) ** 2).backward()
    up = maps.grad
    for pt, ia, r, dn in _pairs_within_8(st, x):
        keep = (up[:, pt] != 0).any(0)
        if not keep.any():
            continue
        pt, ia, r, dn = pt[keep], ia[keep], r[keep], dn[keep]
        loss = 0.0
        for m, t in enumerate(batch_terms(pt, ia, r, dn)):
            if m == M:
                loss = loss + (up[st.dsolv_index][pt] * t).sum()
                continue
            v = t[1].detach()
            times = t[2] * ((v == lo[m][pt]).double() + ((v == hi[m][pt]) & (v > 0)).double())
            loss = loss + (up[m][pt] * (t[0] + t[3] + times * t[1])).sum()
        loss.backward()
    on = torch.nonzero(up[st.elec_index]).reshape(-1)
    ax = _axes(st)
    per_atom = torch.zeros(st.n_atoms, dtype=torch.float64, device="cuda")
    for i in on.split(max(1, int(1.0e8) // st.n_atoms)):
        pt = torch.stack((ax[0][i % st.n1[0]], ax[1][(i // st.n1[0]) % st.n1[1]], ax[2][i // (st.n1[0] * st.n1[1])]), 1)
        r = sum((x[None, :, d] - pt[:, None, d]).square() for d in range(3)).sqrt()
        per_atom += up[st.elec_index][i] @ (model.eps_of(r) / r.clamp(min=0.5))
    (model.charge * model.w[2] * per_atom).sum().backward()
    maps = maps.detach().view((M + 2,) + grid)
    return {**_split(st, maps), "scores": scores.detach(),
            "grad": dict(zip(("coord", "charge", "rij", "eps", "weights"), [None] + [p.grad for p in par]))}


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batch":
        return [_exact_maps(st) for st in s["states"]]
    if kind == "fit":
        return _exact_fit(s)
    if kind == "dock":
        st = s["st"]
        maps = _docking_maps(st, seed).view(st.n_maps, -1).double()
        scores, grad = _trilinear(st, maps, s["poses"], _t(_moved(s["poses"], seed)))
        return {"scores": scores, "grad": grad}
    return _exact_maps(s["st"], vina=kind == "vina")
