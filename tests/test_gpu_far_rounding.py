"""The far field's accuracy where no near term hides it: boxes outside the
receptor, the error's 2-norm over the box against FP64.

Unit: u = 2^-24, the most that one FP32 operation loses, relatively; its rms over
mantissas is 0.42 u.  T = sqrt(sum over atoms of term^2), rms over the box:
independent roundings of the terms add up to a multiple of it.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import autogrid_amd as ag
from test_gpu_far import base, state  # noqa: F401

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def terms(st, points, rounds=1.0, flips=0.0):
    """(sum of the terms, mean square error that `rounds` roundings of each and putting
    `flips` of the pairs on the wrong side of a table step leaves) at points, FP64."""
    tab = np.asarray(st.r_eps if st.dddiel else np.full(8192, st.inv_diel_cal), np.float32).astype(np.float64)
    step = np.abs(np.diff(tab, append=tab[-1]))
    e, sq = np.zeros(len(points)), np.zeros(len(points))
    q = st.charge * st.coeff_estat
    for a in range(0, st.n_atoms, 2048):
        r = np.linalg.norm(points[:, None, :] - st.coord[None, a:a + 2048], axis=2)
        b = np.minimum((r * 128.0).astype(np.int64), 8191)
        w = q[a:a + 2048] / np.maximum(r, 0.5)
        e += (w * tab[b]).sum(1)
        sq += ((w * tab[b] * U * rounds) ** 2 + flips * (w * step[b]) ** 2).sum(1)
    return e, sq


def grid_points(st):
    x = [(np.arange(st.n1[d]) - st.ne[d]) * st.spacing for d in range(3)]
    return np.stack(np.meshgrid(x[2], x[1], x[0], indexing="ij"), -1).reshape(-1, 3)[:, ::-1]


@pytest.mark.parametrize("n_atoms, spacing", [(6000, 0.375), (12000, 0.9)])
def test_node_sums(base, n_atoms, spacing):  # noqa: F811
    """All atoms interpolated, no table steps; the error's part that changes over
    the box (an atom's rounded charge and place are the same for all of it).  A
    term's distance and reciprocal root lose 0.75 u rms, a partial sum of up to 16
    terms of random signs 0.42 u sqrt(1 + ... + 16) / 4 = 1.22 u a term, FP64 sums of
    those nothing: 1.43 u a term at a node, 1.3 times that over the points of a patch,
    1.86 u T, and a tenth for the estimate.  (Partial sums of 64 terms, added up in
    FP32: 0.42 u sqrt(1 + ... + 64) / 8 = 2.4 u a term and more.)"""
    print(f"[gpu] far node sums {n_atoms} {spacing}", flush=True)
    st = state(base, n_atoms, (33, 25, 27), spacing, 35.0, n_atoms, constant=4.0, offset=260.0)
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)[0].reshape(-1)
    want, sq = terms(st, grid_points(st))
    err, t = np.std(got - want), np.sqrt(np.mean(sq))
    out = 0.42 * U * np.sqrt(np.mean(want ** 2))      # the result's own rounding
    assert err <= np.hypot(2.05 * t, out), f"{err / t:.2f} u T"


@pytest.mark.parametrize("spacing, constant", [(0.9, None), (0.75, 4.0)])
def test_box_nodes(base, spacing, constant):  # noqa: F811
    """One charge ahead of a coarse box's face, at the distances from which the box
    takes it: its nodes leave no more than a patch's own at the distance from
    which that interpolates (6.5 half-lengths of a run, 10 without table steps),
    5.2e-6 of the term there (8.4e-7), once for each axis."""
    print(f"[gpu] far box nodes {spacing} {constant}", flush=True)
    n = 40000
    st = state(base, n, (64, 64, 64), spacing, 50.0, n, constant=constant)
    edge = 0.5 * 31 * spacing                               # half of a box of 32 points
    far = (10.0 if constant else 6.5) * 7.5 * spacing
    tab = np.asarray(st.r_eps if st.dddiel else np.full(8192, st.inv_diel_cal), np.float64)
    q = np.zeros(n)
    q[n // 2] = 1.0
    pts = grid_points(st)
    allowed = 3 * (8.4e-7 if constant else 5.2e-6) * abs(st.coeff_estat) * tab[min(int(128 * far), 8191)] / far
    with ag.Context(0) as ctx:
        for d in np.arange(1.3, 3.6, 0.15) * edge:          # from the face, in half-edges
            x = st.coord.copy()
            x[n // 2] = [edge - 32 * spacing, -32 * spacing - d, edge - 32 * spacing]
            one = dataclasses.replace(st, coord=x, charge=q, _keep=[])
            got = ctx.maps_plain(one)[0].reshape(-1)
            box = np.all(pts < -0.5 * spacing, axis=1)      # the first box's points
            r = np.linalg.norm(pts[box] - x[n // 2], axis=1)
            b = np.minimum((128 * r).astype(int), 8190)
            want = st.coeff_estat * tab[b] / r
            off = st.coeff_estat * np.abs(tab[b] - tab[b + 1]) / r + 3e-7 * np.abs(want)   # a table step; FP32
            err = np.abs(got[box] - want)
            assert np.all(err <= allowed + np.abs(off)), (d, float((err / (allowed + np.abs(off))).max()))


# Share of the pairs that FP32 distances put on the wrong side of a table step,
# where all are summed pair by pair: 128 r is good to some 1e-4 of a step.
FLIPS = 1.6e-4


def shell_error(st, got):
    """(rms error, rms error that rounded terms and flipped bins leave) by
    distance from the nearest atom, in shells of 4 A from 8 A on, at sampled points."""
    pick = np.random.default_rng(st.n_atoms).choice(st.points, 9000, replace=False)
    pts, got = grid_points(st)[pick], got[pick]
    want, sq = terms(st, pts, 2.0, FLIPS)
    near = np.full(len(pts), np.inf)
    for a in range(0, st.n_atoms, 2048):
        near = np.minimum(near, np.linalg.norm(pts[:, None, :] - st.coord[None, a:a + 2048], axis=2).min(1))
    out = []
    for lo in np.arange(8.0, 64.0, 4.0):
        m = (near >= lo) & (near < lo + 4.0)
        if m.sum() >= 200:
            out.append((lo, np.sqrt(np.mean((got[m] - want[m]) ** 2)), np.sqrt(np.mean(sq[m]))))
    return out


@pytest.mark.parametrize("n_atoms, spacing, charges", [
    (30, 0.375, "all"), (600, 0.375, "all"), (5000, 0.375, "all"), (5000, 0.375, "one"), (5000, 0.375, "ion"),
    (2500, 0.5, "all"), (1200, 1.0, "all"), (12000, 0.375, "all")])
def test_shells_outside_the_receptor(base, n_atoms, spacing, charges):  # noqa: F811
    """The shells 8 to 60 A outside: no table step there is hidden by larger ones
    nearer.  Against what a sum pair by pair leaves (its rounded terms 2 u each,
    FLIPS of the pairs one table step off), three times as much: flips are few
    and a shell is a small sample of them."""
    print(f"[gpu] far shells {n_atoms} {spacing} {charges}", flush=True)
    radius = (n_atoms / 0.068 * 0.75 / np.pi) ** (1 / 3)
    n1 = (97, 33, 33) if spacing < 0.5 else (81, 33, 33)
    st = state(base, n_atoms, n1, spacing, radius, n_atoms, offset=-(radius + 4.0 + 0.5 * (n1[0] - 1) * spacing))
    if charges != "all":     # one charge alone, or an ion's among the others
        q = 1e-3 * st.charge if charges == "one" else st.charge.copy()
        q[n_atoms // 2] = 2.0
        st = dataclasses.replace(st, charge=q, _keep=[])
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)[0].reshape(-1)
    worst = [(lo, err / left) for lo, err, left in shell_error(st, got)]
    print(" ".join(f"{lo:.0f}:{x:.2f}" for lo, x in worst), flush=True)
    assert len(worst) >= 4 and all(x <= 3.0 for _, x in worst), worst


@pytest.mark.parametrize("n_atoms, n1, spacing, constant", [
    (257, (29, 29, 29), 0.375, None),      # a patch's atoms in one workgroup, the last atom in a group of its own
    (2049, (29, 29, 29), 0.375, None),     # in eight
    (2049, (29, 29, 29), 0.375, 4.0),
    (9000, (97, 65, 66), 0.375, None),     # coarse boxes, ragged ones at the ends
    (9001, (33, 60, 140), 0.375, None),
    (20000, (97, 65, 66), 0.375, 4.0)])
def test_every_atom_counts_once(base, n_atoms, n1, spacing, constant):  # noqa: F811
    """One charge alone, on atoms at the ends of the groups of 64 and of the workgroups'
    parts: left out or taken twice, by a patch, its box or both, it would be off by
    all of itself.  A pair's bin is at most one table step off, 1.7e-3 of the term at
    8 A, and interpolation less."""
    print(f"[gpu] far every atom {n_atoms} {n1}", flush=True)
    radius = (n_atoms / 0.068 * 0.75 / np.pi) ** (1 / 3)
    st = state(base, n_atoms, n1, spacing, radius, 3, constant=constant, offset=0.4 * radius)
    tab = np.asarray(st.r_eps if st.dddiel else np.full(8192, st.inv_diel_cal), np.float32).astype(np.float64)
    last = n_atoms - 1
    pts = grid_points(st)
    with ag.Context(0) as ctx:
        for a in sorted({0, 1, 63, 64, 65, 127, 128, 255, 256, n_atoms // 2, last // 64 * 64 - 1, last // 64 * 64, last - 1, last}):
            q = np.zeros(n_atoms)
            q[a] = 1.0
            got = ctx.maps_plain(dataclasses.replace(st, charge=q, _keep=[]))[0].reshape(-1)
            r = np.linalg.norm(pts - st.coord[a], axis=1)
            want = st.coeff_estat * tab[np.minimum((128 * r).astype(int), 8191)] / np.maximum(r, 0.5)
            off = np.abs(got - want) / np.abs(want)
            assert np.all(off[r > 8.0] <= 2e-3), (a, float(off[r > 8.0].max()))
            assert np.all(off[r <= 8.0] <= 2e-5), (a, float(off[r <= 8.0].max()))
