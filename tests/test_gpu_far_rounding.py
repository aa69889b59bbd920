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


def terms(st, points, flips=0.0):
    """(sum of the terms, mean square error that rounding each to U and putting
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
        sq += ((w * tab[b] * U) ** 2 + flips * (w * step[b]) ** 2).sum(1)
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
