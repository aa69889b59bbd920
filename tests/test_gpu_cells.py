"""The cell list made by one workgroup against the one made in four launches:
the same records in the same order, so the same maps bit for bit.  A receptor
alone takes the first, and in a batch beside a large one the second."""
from __future__ import annotations

import ctypes as C
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


class Dev:
    """A device buffer through the engine's own HIP runtime."""

    def __init__(self, nbytes):
        self.hip, self.p = C.CDLL("libamdhip64.so"), C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.p), C.c_size_t(nbytes)) == 0

    def put(self, a):
        assert self.hip.hipMemcpy(self.p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0

    def get(self, n):
        a = np.empty(n, np.float32)
        assert self.hip.hipMemcpy(a.ctypes.data_as(C.c_void_p), self.p, C.c_size_t(a.nbytes), 2) == 0
        return a

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        assert self.hip.hipFree(self.p) == 0


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


@pytest.mark.parametrize("n, n1, edge", [
    (600, (33, 33, 33), 25.0),       # two parts: the far field first, the cell list in it
    (2500, (25, 31, 17), 33.0),      # eight parts, ragged patches
    (5000, (5, 5, 5), 42.0),         # one patch
    (ONE, (41, 41, 41), 44.0),
    (600, (33, 33, 157), 25.0),      # more cells than fit beside the far kernel's other workgroups
    (200, (33, 33, 33), 18.0),       # one part: the usual order
])
def test_far_field_first(base, n, n1, edge):
    """A map set on the device and one copied to the host take the far field
    in other places of the same sum."""
    print(f"[gpu] far first {n} {n1}", flush=True)
    st = state(base, n, n1, edge, n)
    with ag.Context(0) as ctx:
        host = np.asarray(ctx.maps_plain(st)).reshape(-1)
        blank = np.full(host.size, np.nan, np.float32)
        with ctx.plan(st) as plan, Dev(host.nbytes) as out:
            for _ in range(3):
                out.put(blank)
                plan.execute(out.p.value)
                assert np.array_equal(out.get(host.size), host)
            t = ctx.timing()
    assert all(v >= 0.0 for v in t.values()) and max(t.values()) < 1e3


def test_more_plans_than_reports(base):
    """Plans past the 64 that a context has reports for keep their flag on the
    device; a report given back is used again."""
    print("[gpu] plans without reports", flush=True)
    st = state(base, 300, (17, 17, 17), 20.0, 3)
    n = st.n_maps * st.points
    with ag.Context(0) as ctx, Dev(4 * n) as out:
        def run(plan):
            out.put(np.full(n, np.nan, np.float32))
            plan.execute(out.p.value)
            return out.get(n)

        plans = [ctx.plan(st) for _ in range(66)]
        first = run(plans[0])
        assert np.isfinite(first).all()
        assert all(np.array_equal(run(p), first) for p in plans[1:])
        plans[3].close()
        plans.append(ctx.plan(st))
        assert np.array_equal(run(plans[-1]), first)
        for p in plans:
            p.close()


@pytest.mark.parametrize("n, n1", [(500, (41, 42, 43)), (1500, (81, 33, 80)), (9000, (97, 65, 66))])
def test_far_field_beside(base, n, n1):
    """In a constant dielectric the far field runs beside the near one for a map
    set on the device, and behind it for one copied to the host."""
    print(f"[gpu] far beside {n} {n1}", flush=True)
    st = dataclasses.replace(state(base, n, n1, (n / 0.068) ** (1 / 3), n), dddiel=0, inv_diel_cal=332.0 / 4.0, _keep=[])
    with ag.Context(0) as ctx:
        host = np.asarray(ctx.maps_plain(st)).reshape(-1)
        with ctx.plan(st) as plan, Dev(host.nbytes) as out:
            for _ in range(3):
                out.put(np.full(host.size, np.nan, np.float32))
                plan.execute(out.p.value)
                assert np.array_equal(out.get(host.size), host)
