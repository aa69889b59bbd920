"""The far-field kernel (direct pairs near a patch, interpolation from its
nodes beyond) against the FP64 sum over all pairs, where its parts can go
wrong: patch and run edges, atom counts at the group of 64, patches shared by
workgroups, spacings that move the radius and the table's end, atoms far
outside the box, and dielectric tables that are flat, rough or kinked.

Tolerance, per point, from the design: an interpolated term follows its table
to 1e-5 (the radius is chosen so) and its steps stay below 6.5e-5 of the value,
half a step on average with random sign, so 3e-5 of the sum of the terms'
magnitudes bounds the sum; a direct pair whose FP32 bin differs from the FP64
one moves by one table step, at most 1.1e-3 of the term (r > 8 A), and a few
such pairs meet at one point: 5e-3 of its largest term.
"""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

import autogrid_amd as ag
import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base(tmp_path_factory):
    d = tmp_path_factory.mktemp("far")
    gpf = cases.materialize("small", str(d))
    cwd = os.getcwd()
    os.chdir(d)
    try:
        return ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)


def state(base, n_atoms, n1, spacing, radius, seed, r_eps=None, constant=None, offset=0.0):
    """The base's map set cut to e and d, n_atoms random atoms in a ball of the
    given radius (A), its centre offset along x, on a grid of n1 points."""
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n_atoms, 3))
    x *= radius * rng.uniform(size=(n_atoms, 1)) ** (1 / 3) / np.linalg.norm(x, axis=1, keepdims=True)
    x[:, 0] += offset
    q = rng.normal(0.0, 0.25, n_atoms)
    pick = rng.integers(0, base.n_atoms, n_atoms)
    keep = dict(vol=base.vol[pick], solpar=base.solpar[pick], type=base.type[pick], hbond=base.hbond[pick],
                rexp=base.rexp[pick], rvector=base.rvector[pick], rvector2=base.rvector2[pick],
                disorder=np.zeros(n_atoms, np.uint8))
    st = dataclasses.replace(base, coord=np.round(x, 3), charge=q, n1=tuple(n1), ne=tuple(k // 2 for k in n1),
                             spacing=spacing, maps=base.maps[:0], elec_index=0, dsolv_index=1, n_maps=2,
                             e_vdw_hb=base.e_vdw_hb[:, :0], pairs=None, _keep=[], **keep)
    if r_eps is not None:
        st = dataclasses.replace(st, r_eps=r_eps, _keep=[])
    if constant is not None:
        st = dataclasses.replace(st, dddiel=0, inv_diel_cal=332.0 / constant, _keep=[])
    return st


def check(st, got, seed=0, points=3000, floor_charge=0.0):
    """e at sampled points (the grid's corners among them) against FP64."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = st.n1
    P = st.points
    pick = np.unique(np.concatenate([[0, nx - 1, P - 1, P - nx], rng.integers(0, P, points)]))
    ijk = np.stack([pick % nx, (pick // nx) % ny, pick // (nx * ny)], 1)
    pt = (ijk - np.array(st.ne)) * st.spacing
    tab = np.asarray(st.r_eps if st.dddiel else np.full(8192, st.inv_diel_cal), np.float32).astype(np.float64)
    e, mag, top = np.zeros(len(pick)), np.zeros(len(pick)), np.zeros(len(pick))
    for a in range(0, st.n_atoms, 4096):
        r = np.linalg.norm(pt[:, None, :] - st.coord[None, a:a + 4096], axis=2)
        t = st.charge[a:a + 4096] * st.coeff_estat * tab[np.minimum((r * 128.0).astype(np.int64), 8191)] / \
            np.maximum(r, 0.5)
        e += t.sum(1)
        unit = abs(st.coeff_estat) * tab[np.minimum((r * 128.0).astype(np.int64), 8191)] / np.maximum(r, 0.5)
        mag += (unit * np.maximum(np.abs(st.charge[a:a + 4096]), floor_charge)).sum(1)
        top = np.maximum(top, np.abs(t).max(1))
    err = np.abs(got.reshape(-1)[pick].astype(np.float64) - e)
    lim = 3e-5 * mag + 5e-3 * top
    worst = int(np.argmax(err / lim))
    assert np.all(err <= lim), f"point {ijk[worst]}: error {err[worst]:.3g}, allowed {lim[worst]:.3g}"


def run(st):
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)
        again = ctx.maps_plain(st)
    assert np.array_equal(got, again)
    check(st, got[0])


@pytest.mark.parametrize("n1", [(1, 1, 1), (15, 7, 9), (16, 8, 8), (17, 9, 9), (33, 6, 10), (16, 11, 41), (48, 41, 61)])
def test_patch_edges(base, n1):
    print(f"[gpu] far patches {n1}", flush=True)
    run(state(base, 1500, n1, 0.375, 32.0, 1))


@pytest.mark.parametrize("n_atoms", [1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 2049, 4100])
def test_atom_groups(base, n_atoms):
    """Group-of-64 edges, and (29^3 points: 24 patches) the atom counts where
    a patch goes from one workgroup to up to eight."""
    print(f"[gpu] far atoms {n_atoms}", flush=True)
    run(state(base, n_atoms, (29, 29, 29), 0.375, 35.0, n_atoms))


@pytest.mark.parametrize("spacing", [0.1, 0.25, 0.5, 0.9, 1.1, 2.0, 4.0])
def test_spacings(base, spacing):
    """The radius grows with the spacing; from about 1 A a direct pair can pass
    the table's end."""
    print(f"[gpu] far spacing {spacing}", flush=True)
    run(state(base, 1200, (35, 21, 27), spacing, 40.0, 5))


@pytest.mark.parametrize("offset", [30.0, 70.0, 150.0])
def test_atoms_outside_the_box(base, offset):
    print(f"[gpu] far offset {offset}", flush=True)
    run(state(base, 700, (33, 33, 33), 0.375, 20.0, 6, offset=offset))


@pytest.mark.parametrize("table", ["flat", "rough", "kinked", "zero past 30 A"])
def test_dielectric_tables(base, table):
    """A table the nodes cannot follow is summed pair by pair as far out as
    needed."""
    print(f"[gpu] far table {table}", flush=True)
    if table == "flat":
        run(state(base, 2500, (40, 40, 40), 0.375, 45.0, 7, constant=4.0))
        return
    k = np.arange(8192)
    tab = base.r_eps.copy()
    if table == "rough":
        tab *= 1.0 + 1e-3 * np.random.default_rng(8).uniform(-1, 1, 8192)
    elif table == "kinked":
        tab *= np.where(k > 40 * 128, 1.0 - 5e-5 * (k - 40 * 128), 1.0)
    else:
        tab[30 * 128:] = 0.0
    run(state(base, 2500, (40, 40, 40), 0.375, 45.0, 7, r_eps=tab))


@pytest.mark.parametrize("charges", ["four decades", "one large", "all zero", "half zero"])
@pytest.mark.parametrize("spacing", [0.25, 0.5])
def test_charge_levels(base, charges, spacing):
    """An atom of a small charge is interpolated from nearer, to the absolute
    error of one of the reference charge (0.85 rms): the bound's first part
    takes every charge as the rms at least."""
    print(f"[gpu] far charges {charges} {spacing}", flush=True)
    st = state(base, 2500, (40, 33, 41), spacing, 36.0, 9)
    rng = np.random.default_rng(10)
    q = st.charge
    if charges == "four decades":
        q = rng.choice([-1.0, 1.0], len(q)) * 10.0 ** rng.uniform(-4, 0, len(q))
    elif charges == "one large":
        q = np.where(np.arange(len(q)) == 7, 20.0, 0.01 * q)
    elif charges == "all zero":
        q = np.zeros(len(q))
    else:
        q = np.where(np.arange(len(q)) % 2, q, 0.0)
    st = dataclasses.replace(st, charge=q, _keep=[])
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)
        assert np.array_equal(ctx.maps_plain(dataclasses.replace(st, charge=-q, _keep=[]))[0], -got[0])
    check(st, got[0], floor_charge=float(np.sqrt(np.mean(q ** 2))))


@pytest.mark.parametrize("n1, spacing, constant, offset", [
    ((1, 1, 1), 0.375, 1.0, 0.0), ((33, 41, 17), 0.25, 4.0, 0.0), ((35, 21, 27), 0.9, 80.0, 3.0),
    ((30, 21, 20), 2.0, 4.0, 0.0), ((33, 33, 33), 0.375, 2.5, 90.0)])
def test_constant_dielectric(base, n1, spacing, constant, offset):
    """One value past the near kernel's pairs: summed without the table, at
    any spacing, with atoms at and inside the near limit of a patch."""
    print(f"[gpu] far constant {n1} {spacing} {constant}", flush=True)
    run(state(base, 1600, n1, spacing, 30.0, 11, constant=constant, offset=offset))


def test_zero_past_the_near_limit(base):
    """A table that is zero from bin 1025 on: the far kernel adds nothing."""
    print("[gpu] far zero table", flush=True)
    tab = base.r_eps.copy()
    tab[1025:] = 0.0
    run(state(base, 1600, (33, 33, 33), 0.375, 30.0, 12, r_eps=tab))


@pytest.mark.parametrize("n_atoms, n1, spacing, constant", [
    (9000, (97, 65, 66), 0.375, None),     # boxes of 4 x 4 patches, ragged ones at the ends
    (9001, (33, 60, 140), 0.375, None),    # one x-run past a box; patches not 8 x 8
    (12000, (90, 90, 90), 0.3, None),
    (16000, (60, 61, 63), 0.6, None),      # wide boxes: a longer distance
    (20000, (97, 65, 66), 0.375, 4.0),     # no table
])
def test_coarse_boxes(base, n_atoms, n1, spacing, constant):
    """Atoms beyond a box of patches are summed at the box's nodes; alone and
    in a batch the same bits."""
    print(f"[gpu] far boxes {n_atoms} {n1}", flush=True)
    radius = (n_atoms / 0.068 * 0.75 / np.pi) ** (1 / 3)
    st = state(base, n_atoms, n1, spacing, radius, n_atoms, constant=constant, offset=0.4 * radius)
    small = state(base, 700, (17, 18, 19), spacing, 17.0, 13, constant=constant)
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)
        assert np.array_equal(got, ctx.maps_plain(st))
        beside = ctx.maps_batch([small, st], tune={"cell_size": 4.0, "cube": True})
    assert np.array_equal(np.asarray(beside[1]).reshape(-1), np.asarray(got).reshape(-1))
    check(st, got[0])
