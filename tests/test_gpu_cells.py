"""The cell list made by one workgroup against the one made in four launches:
the same records in the same order, so the same maps bit for bit.  A receptor
alone takes the first, and in a batch beside a large one the second."""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

import autogrid_amd as ag
import cases

pytestmark = pytest.mark.gpu
ONE = 6144          # atoms of a cell list made by one workgroup


@pytest.fixture(scope="module")
def base(tmp_path_factory):
    d = tmp_path_factory.mktemp("cells")
    gpf = cases.materialize("small", str(d))
    cwd = os.getcwd()
    os.chdir(d)
    try:
        return ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)


def state(base, n, n1, edge, seed):
    """n atoms of the base's, spread over a cube of the given edge (A)."""
    rng = np.random.default_rng(seed)
    pick = np.concatenate([np.flatnonzero(base.hbond == 2)[:1], rng.integers(0, base.n_atoms, n - 1)])
    return dataclasses.replace(
        base, coord=np.round(rng.uniform(-edge / 2, edge / 2, (n, 3)), 3), charge=base.charge[pick], vol=base.vol[pick],
        solpar=base.solpar[pick], type=base.type[pick], hbond=base.hbond[pick], rexp=base.rexp[pick],
        rvector=base.rvector[pick], rvector2=base.rvector2[pick], disorder=np.zeros(n, np.uint8),
        n1=tuple(n1), ne=tuple(k // 2 for k in n1), _keep=[])


@pytest.mark.parametrize("n, n1, edge", [
    (1, (5, 5, 5), 2.0),             # one atom, one cell in use
    (64, (9, 9, 9), 0.5),            # all atoms in a few cells
    (1025, (21, 21, 21), 30.0),      # one past the workgroup; atoms outside every cell
    (1500, (21, 97, 5), 40.0),       # cells not a multiple of 64
    (ONE, (25, 25, 25), 44.0),       # the most that one workgroup takes
    (ONE + 1, (25, 25, 25), 44.0),   # the fewest in four launches
])
def test_one_workgroup(base, n, n1, edge):
    print(f"[gpu] cells {n} {n1}", flush=True)
    st, large = state(base, n, n1, edge, n), state(base, ONE + 64, (9, 9, 9), 45.0, 5)
    with ag.Context(0) as ctx:
        alone = ctx.maps_plain(st)
        beside = ctx.maps_batch([st, large], tune={"cell_size": 4.0, "cube": True})
    assert np.array_equal(np.asarray(alone).reshape(-1), np.asarray(beside[0]).reshape(-1))
    assert np.isfinite(alone).all()
