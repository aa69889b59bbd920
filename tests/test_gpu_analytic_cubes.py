"""The analytic mode's cube kernels where they can go wrong: grids at the cube's
and the bit word's edges, every count of affinity maps a kernel is built for,
pair exponents off the 12-6 / 12-10 path, receptors denser than one list.

Forward: against the oracle's FP64 model, under the plain path's tolerance.
Adjoint: it is linear in the cotangent, so the gradients of a sparse cotangent
and of its complement add up to the whole's.  Each is an FP32 sum in its own
order; 2e-5 of the largest component is 170 roundings of 1.2e-7, for sums of
up to 30,000 terms that grow as their square root.
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
from test_gpu_analytic import Dev

pytestmark = pytest.mark.gpu


def _state(tmp_path, name, n1, naff):
    """The named case on a grid of n1 points with its first naff affinity maps."""
    gpf = cases.materialize(name, str(tmp_path))
    cwd = os.getcwd()
    os.chdir(tmp_path)
    try:
        st = ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)
    return dataclasses.replace(st, n1=tuple(n1), ne=tuple(k // 2 for k in n1), maps=st.maps[:naff],
                               pairs=st.pairs[:naff].copy(), e_vdw_hb=st.e_vdw_hb[:, :naff], elec_index=naff,
                               dsolv_index=naff + 1, n_maps=naff + 2, _keep=[])


def _forward(st):
    with ag.Context(0) as ctx, ag.Analytic(ctx, st) as an:
        d = Dev(4 * st.n_maps * st.points)
        try:
            an.forward(d.p.value)
            return d.get(st.n_maps * st.points).reshape(st.n_maps, -1)
        finally:
            d.free()


def _check(st):
    got = _forward(st)
    pts = np.unique(np.random.default_rng(2).integers(0, st.points, min(st.points, 1500)))
    ref = ol.analytic_maps(st, pts)
    for m in range(st.n_maps):
        ok, mx, rms, bad = parity.within(got[m, pts], ref[m])
        assert ok, f"map {m}: max {mx} rms {rms}, {bad} points over tolerance"


@pytest.mark.parametrize("n1,naff", [((1, 1, 1), 1), ((4, 4, 4), 4), ((5, 3, 9), 5), ((17, 8, 7), 6), ((13, 12, 11), 7),
                                     ((9, 10, 21), 8)])
def test_forward_grids_and_map_counts(tmp_path, n1, naff):
    print(f"[gpu] analytic forward {n1} {naff} maps", flush=True)
    _check(_state(tmp_path, "all13", n1, naff))


@pytest.mark.parametrize("what", ["exponents", "coefficients", "no smoothing"])
def test_forward_pair_forms(tmp_path, what):
    print(f"[gpu] analytic forward, {what}", flush=True)
    if what == "coefficients":
        _check(_state(tmp_path, "nbp_coeffs", (13, 9, 11), 4))
        return
    st = _state(tmp_path, "all13", (13, 9, 11), 6)
    if what == "exponents":
        st.pairs["xA"][1], st.pairs["xB"][1] = 9, 6
        st.pairs["xA"][3, 0], st.pairs["xB"][3, 0] = 12, 4
    else:
        st = dataclasses.replace(st, r_smooth=0.0, _keep=[])
    _check(st)


@pytest.mark.parametrize("n_atoms", [255, 257, 767, 769, 1400])
def test_forward_dense_receptor(tmp_path, n_atoms):
    """Every atom within 8 A of every point: lists at and past the places a
    cube's donor H (256) and atoms (1,024, worked off from 768 on) take."""
    print(f"[gpu] analytic forward, {n_atoms} atoms a cube", flush=True)
    st = _state(tmp_path, "all13", (5, 5, 5), 5)
    rng = np.random.default_rng(n_atoms)
    x = rng.normal(size=(n_atoms, 3))
    x *= 4.5 * rng.uniform(0.5, 1.0, (n_atoms, 1)) / np.linalg.norm(x, axis=1, keepdims=True)
    pick = rng.integers(0, st.n_atoms, n_atoms)
    pick[:n_atoms // 3] = rng.choice(np.flatnonzero(st.hbond == 2), n_atoms // 3)   # donor H
    f = {k: getattr(st, k)[pick] for k in ("charge", "vol", "solpar", "type", "hbond", "rexp", "rvector", "rvector2",
                                           "disorder")}
    _check(dataclasses.replace(st, coord=x, _keep=[], **f))


@pytest.mark.parametrize("n1,share", [((64, 5, 6), 0.3), ((65, 7, 5), 0.9), ((130, 3, 4), 0.05), ((20, 21, 22), 0.5)])
def test_adjoint_adds_up(tmp_path, n1, share):
    print(f"[gpu] analytic adjoint {n1}", flush=True)
    st = _state(tmp_path, "all13", n1, 5)
    rng = np.random.default_rng(4)
    G = rng.normal(size=(st.n_maps, st.points)).astype(np.float32)
    pick = rng.uniform(size=st.points) < share
    with ag.Context(0) as ctx, ag.Analytic(ctx, st) as an:
        dm, dg = Dev(4 * G.size), Dev(4 * G.size)
        try:
            an.forward(dm.p.value)
            g = []
            for part in (G, G * pick, G * ~pick):
                dg.put(part)
                g.append(an.adjoint(dg.p.value))
        finally:
            dm.free()
            dg.free()
    for k in g[0]:
        scale = max(float(np.abs(x[k]).max()) for x in g)
        assert scale > 0, k
        off = float(np.abs(g[1][k] + g[2][k] - g[0][k]).max())
        assert off <= 2e-5 * scale, f"{k}: {off / scale:.2g} of the largest component"
