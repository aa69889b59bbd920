"""The analytic e map's accuracy where its nearest atoms do not hide it.

Unit: u = 2^-24, the most that one FP32 operation loses, relatively (0.42 u rms).
T = sqrt(sum over atoms of term^2)."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import autogrid_amd as ag
from test_gpu_analytic import Dev
from test_gpu_analytic_boxes import base, state  # noqa: F401

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def forward(st):
    d = Dev(4 * st.n_maps * st.points)
    try:
        with ag.Context(0) as ctx, ag.Analytic(ctx, st) as an:
            an.forward(d.p.value)
            return d.get(st.n_maps * st.points).reshape(st.n_maps, -1)[st.elec_index].astype(np.float64)
    finally:
        d.free()


def place(st, pt):
    nx, ny, _ = st.n1
    return (np.stack([pt % nx, pt // nx % ny, pt // (nx * ny)], 1) - np.array(st.ne)) * st.spacing


def sums(st, xyz):
    """(sum of the terms, sum of their squares, distance of the nearest atom) in
    FP64, the pairs' squared distance with the half-run's 2^-19 added, as the kernels
    have it."""
    nx = st.n1[0]
    run = 13 if 13 * -(-nx // 13) < 16 * -(-nx // 16) else 16
    added = (0.5 * (run - 1) * st.spacing) ** 2 * 2.0 ** -19
    e, sq, near = np.zeros(len(xyz)), np.zeros(len(xyz)), np.full(len(xyz), np.inf)
    for a in range(0, st.n_atoms, 2048):
        r2 = np.sum((xyz[:, None] - st.coord[None, a:a + 2048]) ** 2, axis=2)
        near = np.minimum(near, np.sqrt(r2.min(1)))
        r = np.sqrt(r2 + added)
        f = 332.0 / (-8.5525 + 86.9525 / (1.0 + 7.7839 * np.exp(-0.003627 * 86.9525 * r))) if st.dddiel else \
            np.full_like(r, st.inv_diel_cal)
        t = st.charge[a:a + 2048] * st.weights[2] * f / r
        e += t.sum(1)
        sq += (t * t).sum(1)
    return e, sq, near


@pytest.mark.parametrize("spacing, constant", [(0.375, None), (0.25, None), (0.6, None), (0.375, 4.0)])
def test_box_nodes(base, spacing, constant):  # noqa: F811
    """One charge ahead of a box's face, from where boxes might take it to where
    they do: eight nodes leave at most 1.2e-7 of the term on each of three axes; a
    term's roundings and those of the places (20 A, 8 A apart) 12 u at most."""
    print(f"[gpu] analytic box nodes {spacing} {constant}", flush=True)
    n = 12000
    st = state(base, n, (48, 48, 48), spacing, 5, constant)
    edge = 7.5 * spacing
    pts = place(st, np.arange(st.points))
    box = np.all(pts < (-8.5) * spacing, axis=1)            # the first box's points
    q = np.zeros(n)
    q[n // 2] = 1.0
    for d in np.arange(2.0, 6.0, 0.25) * edge:
        x = st.coord.copy()
        x[n // 2] = [edge - 24 * spacing, -24 * spacing - d, edge - 24 * spacing]
        one = dataclasses.replace(st, coord=x, charge=q, _keep=[])
        got = forward(one)[box]
        want, _, _ = sums(dataclasses.replace(one, coord=x[n // 2:n // 2 + 1], charge=q[n // 2:n // 2 + 1], _keep=[]),
                          pts[box])
        off = np.abs(got - want).max() / np.abs(want).max()
        assert off <= 3 * 1.2e-7 + 12 * U, (d / edge, off)


def test_sums_of_many_pairs(base):  # noqa: F811
    """Wide boxes, so that each leaves thousands of atoms to its points, a quarter to a
    wave, and takes thousands at its nodes; places and charges that FP32 holds
    exactly, a constant dielectric, points 6 A and more from any atom.  Partial sums
    of up to 95 terms of random signs lose 0.42 u sqrt(95 / 2) = 2.9 u a term, a
    term itself 1 u (distance, root): 3.1 u T, 3.7 with a fifth for the estimate.
    (One FP32 sum over n terms loses 0.42 u sqrt(n / 2): 5.5 u for 350.)"""
    print("[gpu] analytic sums of many pairs", flush=True)
    st = state(base, 60000, (97, 48, 48), 1.0, 3, 20.0)
    x = np.round(64.0 * st.coord) / 64.0
    x[:, 0] -= 62.0                  # the receptor's surface inside the box
    w = st.weights[2] * st.inv_diel_cal
    q = (st.charge * w).astype(np.float32).astype(np.float64) / w
    st = dataclasses.replace(st, coord=x, charge=q, _keep=[])
    e = forward(st)
    xyz = place(st, np.arange(st.points))
    far = np.flatnonzero(np.linalg.norm(xyz - x.mean(0), axis=1) > 59.5 + 6.0)
    pick = np.random.default_rng(1).choice(far, 2500, replace=False)
    want, sq, near = sums(st, xyz[pick])
    m = near >= 6.0
    ratio = np.sqrt(np.mean((e[pick][m] - want[m]) ** 2) / np.mean(sq[m])) / U
    print(f"{ratio:.2f} u T", flush=True)
    assert m.sum() > 1500 and ratio <= 3.7


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_cotangent_past_the_cutoff(base, axis):  # noqa: F811
    """A cotangent that is not a number, 8.0004 A from the only atom: not that
    atom's.  At 7.9 A it is."""
    print(f"[gpu] analytic cutoff {axis}", flush=True)
    st = state(base, 2, (33, 33, 33), 0.375, 7)
    for distance, finite in ((8.0004, True), (7.9, False)):
        x = np.array([[0.0, 0.0, 0.0], [200.0, 0.0, 0.0]])
        x[0, axis] = 4.0
        x[0, (axis + 1) % 3] = np.sqrt(distance ** 2 - 16.0)
        one = dataclasses.replace(st, coord=x, _keep=[])
        cot = np.zeros((one.n_maps, one.points), np.float32)
        cot[0, 16 + 33 * (16 + 33 * 16)] = np.nan
        maps, dmaps = Dev(cot.nbytes), Dev(cot.nbytes)
        dmaps.put(cot)
        try:
            with ag.Context(0) as ctx, ag.Analytic(ctx, one) as an:
                an.forward(maps.p.value)
                g = an.adjoint(dmaps.p.value)
        finally:
            maps.free()
            dmaps.free()
        assert np.isfinite(g["coord"]).all() == finite and np.isfinite(g["eps"]).all() == finite
