"""ag_context_timing: the phases of a map set, wherever their kernels run."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import autogrid_amd as ag
from test_gpu_analytic import Dev
from test_gpu_far import base, state  # noqa: F401

pytestmark = pytest.mark.gpu


def phases(st, n=9):
    """The medians of a plan's phases, in ms."""
    d = Dev(4 * st.n_maps * st.points)
    try:
        with ag.Context(0) as ctx, ctx.plan(st) as p:
            out = []
            for _ in range(n + 2):
                p.execute(d.p.value)
                t = ctx.timing()
                out.append([t[k] for k in ("cell_ms", "near_ms", "far_ms", "total_ms")])
    finally:
        d.free()
    return np.median(np.array(out[2:]), axis=0)


def without_e(st):
    return dataclasses.replace(st, elec_index=-1, dsolv_index=0, n_maps=1, _keep=[])


def test_fields_beside_each_other(base):  # noqa: F811
    """In a constant dielectric the two fields overlap; each has its own time, the
    longer one most of the total."""
    st = state(base, 3000, (81, 81, 81), 0.375, 22.0, 1, constant=4.0)
    cells, near, far, total = phases(st)
    print(f"[gpu] beside {cells:.4f} {near:.4f} {far:.4f} {total:.4f}", flush=True)
    assert cells > 0 and near > 0.1 * total and far > 0.1 * total
    assert max(near, far) <= total and near + far + cells > 0.8 * total


def test_coarse_boxes_are_far_field(base):  # noqa: F811
    """The coarse boxes run before the patches and count with them: the near field
    takes what it takes in a map set without an e map, and the two of its some 50
    operations a pair that add the near pairs to e: 8 % with the e map's stores."""
    st = state(base, 16000, (129, 129, 129), 0.375, 38.0, 2)
    _, near, far, total = phases(st)
    _, alone, _, _ = phases(without_e(st))
    print(f"[gpu] boxes near {near:.4f} alone {alone:.4f} far {far:.4f} total {total:.4f}", flush=True)
    assert near <= 1.08 * alone + 0.02 and far > 0


def test_cell_list_beside_the_far_field(base):  # noqa: F811
    """A small plan's cell list (counts, their sum and two passes over the atoms by
    one workgroup, then the records) against the same plan's without a far field."""
    st = state(base, 1500, (41, 41, 41), 0.375, 17.0, 3)
    cells, near, far, total = phases(st)
    alone = phases(without_e(st))[0]
    print(f"[gpu] small cells {cells:.4f} alone {alone:.4f} near {near:.4f} far {far:.4f} total {total:.4f}", flush=True)
    assert cells >= 0.6 * alone and near > 0 and far > 0
    assert near + far <= total + 1e-3
