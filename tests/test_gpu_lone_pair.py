"""The lone-pair factor of ordered acceptors with two bonds near its axis, where
1 - (dn . rvector2)^2 has no digits left of its own: one such atom, a donor's
map on a fine grid along its rvector2, against the FP64 oracle.

Tolerance, u = 2^-24, theta the angle between the point's direction dn and the
axis: dn is good to 2 u a component and its cross product with the axis to 4 u, so
sin(theta) to 4 u / theta of itself, and y = (dn x rvector2).rvector / sin(theta) to
twice that, which the factor takes as 0.2 / 0.9 of y sqrt(1 - y^2)."""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

import autogrid_amd as ag
import cases
import oracle_lib as ol

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


@pytest.mark.parametrize("axis", [(1.0, 0.031, -0.017), (1.0, -0.2, 0.35), (0.0, 0.0, 0.0)])
def test_near_the_axis(tmp_path, axis):
    print(f"[gpu] lone pair {axis}", flush=True)
    gpf = cases.materialize("small", str(tmp_path))
    cwd = os.getcwd()
    os.chdir(tmp_path)
    try:
        st = ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)
    pick = [int(np.flatnonzero(st.hbond == 5)[0]), int(np.flatnonzero(st.hbond == 2)[0])]
    n1, h = (81, 21, 23), 0.05
    rv2 = np.array(axis)
    if rv2.any():
        rv2 /= np.linalg.norm(rv2)
        rv = np.cross(rv2, [0.3, -0.5, 0.8])
        rv /= np.linalg.norm(rv)
    else:                                       # no axis (the reference's vectors may be zero)
        rv = np.array([0.6, 0.0, 0.8])
    toward = rv2 if rv2.any() else np.array([1.0, 0.0, 0.0])
    x = np.array([-4.2 * toward, [0.0, 60.0, 0.0]])
    zero = np.zeros(2)
    st = dataclasses.replace(
        st, coord=x, charge=zero, vol=zero, solpar=zero, type=st.type[pick], hbond=st.hbond[pick],
        rexp=np.zeros(2, np.int32), rvector=np.array([rv, [1.0, 0, 0]]), rvector2=np.array([rv2, [0, 0, 0.0]]),
        disorder=np.zeros(2, np.uint8), n1=n1, ne=tuple(k // 2 for k in n1), spacing=h, _keep=[])
    m = [k for k in range(st.n_atom_maps) if st.maps[k]["is_hbonder"] and st.maps[k]["hbond"] in (1, 2)][0]
    want = ol.maps(st)[m].reshape(-1)
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)[m].reshape(-1).astype(np.float64)
    g = [(np.arange(n1[d]) - st.ne[d]) * h for d in range(3)]
    pt = np.stack(np.meshgrid(g[2], g[1], g[0], indexing="ij"), -1).reshape(-1, 3)[:, ::-1]
    d = x[0] - pt
    dn = d / np.linalg.norm(d, axis=1, keepdims=True)
    cross = np.cross(dn, rv2)
    theta = np.maximum(np.linalg.norm(cross, axis=1), 1e-3) if rv2.any() else np.ones(len(dn))
    y = np.minimum(np.abs(cross @ rv) / theta, 1.0)
    dy = 8 * U / theta
    ds = np.minimum(dy / np.sqrt(np.maximum(1 - y * y, 1e-12)), np.sqrt(2 * dy)) + dy
    rel = 4 * U / theta + 0.2 / 0.9 * ds + 16 * U
    # the branch of the other side, (0.117 - c^2)^3 with its zero at c = -0.342
    c = -(dn @ rv)
    other = c < 0
    rel = np.where(other, 4 * U / theta + 16 * U + 3 * 4 * U / np.maximum(0.116978 - c * c, 1e-6), rel)
    use = (want < -1e-4 * np.abs(want.min())) & (np.abs(c) > 1e-5) & (c > -0.33)
    off = np.abs(got - want)[use] / (rel * np.abs(want))[use]
    assert use.sum() > 3000 and (not rv2.any() or theta[use].min() < 0.02)
    assert np.all(off <= 1.0), (float(off.max()), float(theta[use][off.argmax()]))
