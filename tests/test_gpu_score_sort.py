"""The scorer's device-built contribution lists: atom counts at the sort's
tile (256 atoms are 2,048 corners), many atoms in one cell, grids whose points
need one to three sort passes, coinciding map slots, moved positions.

dL/dmaps against S^T g in FP64.  A corner's weight is a product of three FP32
factors, each within 6e-8 of 1 - f or f of a position rounded to 6e-8 of up to
128 grid units (8e-6 of a unit), the rest is FP64 with one rounding at the end:
2.5e-5 of the sum of the touched terms' charges bounds an entry.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import autogrid_amd as ag
from test_gpu_analytic import Dev

pytestmark = pytest.mark.gpu


@dataclasses.dataclass
class Grid:
    n1: tuple
    n_maps: int
    elec_index: int
    dsolv_index: int
    spacing: float = 0.375

    @property
    def ne(self):
        return tuple(k // 2 for k in self.n1)

    @property
    def points(self):
        return int(np.prod(self.n1))


def _poses(st, n, per_pose, rng, spread=1.0, maps=None):
    lo = np.array([-e * st.spacing for e in st.ne])
    size = (np.array(st.n1) - 1) * st.spacing
    x = lo + size * (0.5 + spread * (rng.uniform(size=(n, 3)) - 0.5)) * 0.999
    m = rng.integers(-1, st.n_maps if maps is None else maps, n)
    q = rng.normal(0, 0.3, n)
    return [(m[a:a + per_pose], q[a:a + per_pose], x[a:a + per_pose]) for a in range(0, n, per_pose)]


def _expected(st, poses, g):
    """(S^T g, the sum of the magnitudes) in FP64."""
    out, mag = np.zeros((st.n_maps, st.points)), np.zeros((st.n_maps, st.points))
    for k, (m, q, x) in enumerate(poses):
        u = x / st.spacing + np.array(st.ne)
        on = np.all((u >= 0) & (u < np.array(st.n1) - 1), axis=1)
        m, q, u = m[on], q[on], u[on]
        i0 = np.floor(u).astype(np.int64)
        f = u - i0
        for c in range(8):
            b = np.array([c & 1, (c >> 1) & 1, c >> 2])
            w = np.prod(np.where(b, f, 1 - f), axis=1)
            p = (i0 + b) @ np.array([1, st.n1[0], st.n1[0] * st.n1[1]])
            for slot, v in ((m, np.ones_like(q)), (np.full(len(q), st.elec_index), q),
                            (np.full(len(q), st.dsolv_index), np.abs(q))):
                ok = slot >= 0
                np.add.at(out, (slot[ok], p[ok]), (w * v * g[k])[ok])
                np.add.at(mag, (slot[ok], p[ok]), (np.abs(v) * abs(g[k]))[ok])
    return out, mag


def _check(st, poses, moved=None):
    rng = np.random.default_rng(9)
    g = rng.normal(size=len(poses)).astype(np.float32)
    dg, dm = Dev(4 * len(poses)), Dev(4 * st.n_maps * st.points)
    try:
        dg.put(g)
        with ag.Context(0) as ctx, ag.Scorer(ctx, st, poses) as sc:
            if moved is not None:
                sc.set_positions(np.concatenate([p[2] for p in moved]))
                poses = moved
            sc.adjoint(dg.p.value, dm.p.value)
            got = dm.get(st.n_maps * st.points).reshape(st.n_maps, -1)
            sc.adjoint(dg.p.value, dm.p.value)
            assert np.array_equal(got, dm.get(st.n_maps * st.points).reshape(st.n_maps, -1))
    finally:
        dg.free()
        dm.free()
    ref, mag = _expected(st, poses, g.astype(np.float64))
    assert np.all(np.abs(got - ref) <= 2.5e-5 * mag + 1e-30)
    assert np.all(got[mag == 0] == 0)


@pytest.mark.parametrize("n", [1, 31, 255, 256, 257, 5000])
def test_adjoint_counts(n):
    print(f"[gpu] scorer lists, {n} atoms", flush=True)
    st = Grid((41, 33, 27), 6, 4, 5)
    _check(st, _poses(st, n, 40, np.random.default_rng(n)))


@pytest.mark.parametrize("n1", [(2, 2, 2), (6, 6, 6), (7, 6, 6), (41, 40, 39), (128, 128, 5)])
def test_adjoint_grids(n1):
    """Points below and above 256 and 65,536: one, two and three passes."""
    print(f"[gpu] scorer lists on {n1}", flush=True)
    st = Grid(n1, 3, 1, 2)
    _check(st, _poses(st, 700, 25, np.random.default_rng(1)))


def test_adjoint_crowded_cell():
    print("[gpu] scorer lists, one cell", flush=True)
    st = Grid((21, 21, 21), 4, 2, 3)
    _check(st, _poses(st, 3000, 30, np.random.default_rng(2), spread=0.02))


@pytest.mark.parametrize("slots", [(0, 1), (1, 1), (-1, 2), (2, -1), (-1, -1)])
def test_adjoint_coinciding_slots(slots):
    print(f"[gpu] scorer slots {slots}", flush=True)
    st = Grid((15, 14, 13), 3, *slots)
    _check(st, _poses(st, 500, 20, np.random.default_rng(3)))


def test_moved_positions():
    print("[gpu] scorer moved positions", flush=True)
    st = Grid((41, 33, 27), 6, 4, 5)
    a = _poses(st, 900, 30, np.random.default_rng(4))
    b = _poses(st, 900, 30, np.random.default_rng(5), spread=1.2)   # some of them off the grid
    moved = [(p[0], p[1], r[2]) for p, r in zip(a, b)]
    _check(st, a, moved=moved)


@pytest.mark.parametrize("n", [64 * 256, 64 * 256 + 1])
def test_sort_tiles(n):
    """Tiles of 2,048 corners: up to 64 of them, each workgroup adds up the
    counts itself, and for more a launch of its own does."""
    print(f"[gpu] scorer lists, {n} atoms", flush=True)
    st = Grid((41, 43, 47), 5, 3, 4)
    _check(st, _poses(st, n, 300, np.random.default_rng(n), spread=1.05))
