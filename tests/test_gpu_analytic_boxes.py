"""The analytic e map with boxes (atoms beyond a box at its nodes) against the
FP64 sum over all atoms: ends of runs, patches and boxes, both run lengths,
groups of 64 atoms, spacings that move the distance, a constant dielectric,
and receptors around the size from which boxes are used.

Tolerance per point, from the design.  A term by pairs has FP32 roundings (six
of 6e-8, and the run's expansion: 2^-21 of (8 spacings)^2 on r^2, so at most
4e-6 / r^2 A^2 at 0.375 A, 3e-5 at the 0.5 A where r is clamped), one by nodes
3e-7 of itself at the box's nearest; coordinates are FP32 (2e-6 A at 30 A): 2e-6
of the sum of magnitudes and, for the expansion at the nearest atoms,
(spacing / 0.375)^2 1e-4 of the largest term.
"""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

import autogrid_amd as ag
import cases
from test_gpu_analytic import Dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base(tmp_path_factory):
    d = tmp_path_factory.mktemp("anbox")
    gpf = cases.materialize("small", str(d))
    cwd = os.getcwd()
    os.chdir(d)
    try:
        return ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)


def state(base, n, n1, spacing, seed, constant=None):
    """n atoms at protein density in a ball, its centre a third of its radius
    off the grid's; one affinity map, e and d."""
    rng = np.random.default_rng(seed)
    radius = (n / 0.068 * 0.75 / np.pi) ** (1 / 3)
    x = rng.normal(size=(n, 3))
    x *= radius * rng.uniform(size=(n, 1)) ** (1 / 3) / np.linalg.norm(x, axis=1, keepdims=True)
    x[:, 0] += radius / 3
    pick = np.concatenate([np.flatnonzero(base.hbond == 2)[:1], rng.integers(0, base.n_atoms, n - 1)])
    st = dataclasses.replace(
        base, coord=np.round(x, 3), charge=rng.normal(0.0, 0.25, n), vol=base.vol[pick], solpar=base.solpar[pick],
        type=base.type[pick], hbond=base.hbond[pick], rexp=base.rexp[pick], rvector=base.rvector[pick],
        rvector2=base.rvector2[pick], disorder=np.zeros(n, np.uint8), n1=tuple(n1), ne=tuple(k // 2 for k in n1),
        spacing=spacing, maps=base.maps[:1], pairs=base.pairs[:1].copy(), e_vdw_hb=base.e_vdw_hb[:, :1],
        elec_index=1, dsolv_index=2, n_maps=3, _keep=[])
    return st if constant is None else dataclasses.replace(st, dddiel=0, inv_diel_cal=332.0 / constant, _keep=[])


def check(st, e):
    """e at the grid's corners and 4,000 points against FP64."""
    nx, ny, nz = st.n1
    P = st.points
    pt = np.unique(np.concatenate([[0, nx - 1, P - 1, P - nx, nx * ny - 1],
                                   np.random.default_rng(1).integers(0, P, 4000)]))
    xyz = (np.stack([pt % nx, pt // nx % ny, pt // (nx * ny)], 1) - np.array(st.ne)) * st.spacing
    # the pairs' squared distance has 2^-19 of the half-run's added, which keeps it positive
    run = 13 if 13 * -(-nx // 13) < 16 * -(-nx // 16) else 16
    added = (0.5 * (run - 1) * st.spacing) ** 2 * 2.0 ** -19
    want, mag, top = np.zeros(len(pt)), np.zeros(len(pt)), np.zeros(len(pt))
    for a in range(0, st.n_atoms, 2048):
        r = np.sqrt(np.sum((xyz[:, None] - st.coord[None, a:a + 2048]) ** 2, axis=2) + added)
        if st.dddiel:
            f = 332.0 / (-8.5525 + 86.9525 / (1.0 + 7.7839 * np.exp(-0.003627 * 86.9525 * r)))
        else:
            f = np.full_like(r, st.inv_diel_cal)
        t = st.charge[a:a + 2048] * st.weights[2] * f / np.maximum(r, 0.5)
        want += t.sum(1)
        mag += np.abs(t).sum(1)
        top = np.maximum(top, np.abs(t).max(1))
    err = np.abs(e[pt].astype(np.float64) - want)
    lim = 2e-6 * mag + 1e-4 * max(1.0, st.spacing / 0.375) ** 2 * top
    k = int(np.argmax(err / lim))
    assert np.all(err <= lim), f"point {pt[k]}: off {err[k]:.3g}, allowed {lim[k]:.3g}"


@pytest.mark.parametrize("n, n1, spacing, constant", [
    (2000, (65, 65, 65), 0.375, None),     # runs of 13
    (2047, (64, 48, 33), 0.375, None),     # runs of 16, one row past a box
    (2049, (33, 41, 57), 0.375, 4.0),
    (1000, (48, 48, 48), 0.375, None),     # too few atoms for boxes
    (3000, (49, 17, 80), 0.25, None),
    (6000, (50, 45, 40), 0.6, None),
    (5000, (79, 16, 16), 0.3, 20.0),
])
def test_e_map(base, n, n1, spacing, constant):
    print(f"[gpu] analytic boxes {n} {n1} {spacing}", flush=True)
    st = state(base, n, n1, spacing, n, constant)
    d = Dev(4 * st.n_maps * st.points)
    try:
        with ag.Context(0) as ctx, ag.Analytic(ctx, st) as an:
            an.forward(d.p.value)
            got = d.get(st.n_maps * st.points)
            an.set(coord=st.coord[::-1].copy(), charge=st.charge)      # other inputs, then these again
            an.forward(d.p.value)
            an.set(coord=st.coord, charge=st.charge)
            an.forward(d.p.value)
            assert np.array_equal(got, d.get(st.n_maps * st.points))
    finally:
        d.free()
    check(st, got.reshape(st.n_maps, -1)[st.elec_index])
