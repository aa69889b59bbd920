"""The floating grid's culled search against the FP64 distance to the nearest of
all atoms: ragged boxes, atom counts at the group of 256 that is tested at a
time, atoms far outside the box, and a single one.

Tolerance: a coordinate difference of two FP32 values is off by three roundings
(2^-24 of the largest coordinate each), so the distance by 2^-22 of the largest
coordinate and three axes' worth of it at most, plus the square root's own.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import autogrid_amd as ag
from test_gpu_far import base, state  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1", [(1, 1, 1), (8, 8, 8), (9, 17, 7), (41, 33, 12)], ids=str)
@pytest.mark.parametrize("n_atoms,radius,offset", [(1, 3.0, 0.0), (255, 12.0, 0.0), (256, 12.0, 0.0), (257, 12.0, 9.0),
                                                   (3000, 20.0, 5.0), (700, 20.0, 90.0)])
def test_nearest_atom(base, n1, n_atoms, radius, offset):  # noqa: F811
    print(f"[gpu] floating grid {n1} {n_atoms} {offset}", flush=True)
    st = state(base, n_atoms, n1, 0.375, radius, 3, offset=offset)
    st = dataclasses.replace(st, floating_grid=1, _keep=[])
    with ag.Context(0) as ctx:
        ctx.maps_plain(st)
        got = ctx.last_fmap
    ax = [(np.arange(n1[d]) - st.ne[d]) * st.spacing for d in range(3)]
    pt = np.stack(np.meshgrid(ax[2], ax[1], ax[0], indexing="ij"), -1)[..., ::-1].reshape(-1, 3)
    best = np.full(len(pt), np.inf)
    for a in range(0, n_atoms, 256):
        best = np.minimum(best, np.linalg.norm(pt[:, None] - st.coord[None, a:a + 256], axis=2).min(1))
    top = max(np.abs(st.coord).max(), np.abs(pt).max())
    assert np.all(np.abs(got.reshape(-1) - best) <= 3 * 2.0 ** -22 * top + 2.0 ** -22 * best)
