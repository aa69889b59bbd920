"""The near kernel with one, two and four waves to a cube's atoms, on both
sides of the brick counts where the number changes (1,024 and 4,096 bricks of
8x8x4 points) and on ragged grids, for each row width of its tables and with
the options its general form handles.

Maps are held to the parity bar against the FP64 oracle.  The oracle's e map
takes hypot() distances, as the reference does, and the engine sqrt of the sum of
squares: where an atom's distance is a bin edge to the last place the two may take
different bins, so a point of e beyond the bar must be such a point.  How a wave's lanes lie
on the points (the tuning's cube switch) may not change a bit of them.
"""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

import autogrid_amd as ag
import cases
import oracle_lib as ol
import parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["small", "disorder", "all13"])
def base(request, tmp_path_factory):
    d = tmp_path_factory.mktemp("share")
    gpf = cases.materialize(request.param, str(d))
    cwd = os.getcwd()
    os.chdir(d)
    try:
        return request.param, ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)


# (points, spacing): 4 shares (a single point, one cube, ragged, the line), 2 (past the
# line, the next line), 1 (past it)
GRIDS = [((1, 1, 1), 0.375), ((4, 4, 4), 0.375), ((13, 9, 6), 0.375), ((256, 256, 4), 0.07),
         ((257, 251, 4), 0.07), ((512, 509, 3), 0.04), ((513, 512, 2), 0.04)]


def only_ties(st, got, ref, z):
    """Every point beyond the bar has an atom at a bin edge to 1e-12 bins."""
    off = np.abs(got - ref) > np.maximum(parity.TOL_ABS, parity.TOL_REL * np.abs(ref))
    for y, x in zip(*np.nonzero(off)):
        bins = np.linalg.norm(st.coord - (np.array([x, y, z]) - st.ne) * st.spacing, axis=1) * 128.0
        if not np.any(np.abs(bins - np.rint(bins)) < 1e-12):
            return False
    return True


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g[0])))
@pytest.mark.parametrize("count", [0, 1], ids=["", "constriction"])
def test_shared_cubes(base, grid, count):
    name, st = base
    n1, spacing = grid
    print(f"[gpu] near shares {name} {n1} {count}", flush=True)
    st = dataclasses.replace(st, n1=n1, ne=tuple(n // 2 for n in n1), spacing=spacing, constriction_grid=count,
                             constriction_cutoff=6.5, _keep=[])
    z = n1[2] // 2
    ref = ol.maps(ol.oracle_state(st), z, z + 1, cmap=bool(count))
    if count:
        ref, _, rcm = ref
    with ag.Context(0) as ctx:
        got = ctx.maps_plain(st)
        if count:
            assert np.array_equal(ctx.last_cmap[z], rcm[z])
        cubes, slabs = [ctx.maps_batch([st, st], tune={"cell_size": 4.0, "cube": c}) for c in (True, False)]
    for k in range(st.n_maps):
        ok, mx, rms, bad = parity.within(got[k, z], ref[k, z])
        assert ok or (k == st.elec_index and only_ties(st, got[k, z], ref[k, z], z)), \
            f"map {k}: max {mx} rms {rms} bad {bad}"
    for m in cubes + slabs:
        assert np.array_equal(m.view(np.uint32), got.view(np.uint32))
