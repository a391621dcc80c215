"""Whole trajectories of the rows path: every run here ends, through rebuilds.

Rows against tiles (GEMS_HIP_LIST_BUILD=coop): the same bits after 60 steps of a
liquid at its own time step (0.005 tau, T* = 1) or a warm solid, in boxes whose
atoms all, or all but one, fill the groups of 16 lanes.

The update inside the force pass against the one in kernels of its own (each=1
observes every step): at most 5 roundings a step of coordinates below 32 A (2^-48
each) over 60 steps and a growth of at most e^2 give 60 * 5 * 3.6e-15 * 7.4 =
8e-12 A; velocities that over one step (5.1e-5 ps liquid, 1e-3 ps solid) 1.6e-7 and
8e-9 A/ps.
"""
import os

import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")

TAU = 0.01018047  # ps: sqrt(m sigma^2 / eps) for 1 amu, 1 A, 1 eV
V_LIQUID = 98.2   # A/ps: sqrt(eps / m)


def _ctx(tiled=False):
    if tiled:
        os.environ["GEMS_HIP_LIST_BUILD"] = "coop"
    try:
        return hip.Context(0, hip.GH_FP64)
    finally:
        os.environ.pop("GEMS_HIP_LIST_BUILD", None)


def _setup(c, pot, x, t, L, pbc):
    c.set_box(L, *([pbc] if L is not None else []))
    c.set_atoms(x, t)
    rng = np.random.default_rng(9)
    if pot in ("au", "agcu"):
        if pot == "au":
            c.set_masses([cm.MASS_AU])
            c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        else:
            c.set_masses(cm.agcu_masses("Ag"))
            c.set_smatb(2, *cm.matrices(cm.agcu_params("Ag"), 2))
        c.set_skin(0.5)
        c.set_velocities(rng.normal(0.0, 4.0, x.shape))
        return 0.002
    e, s = np.array([[1.0, 0.9], [0.9, 0.8]]), np.array([[1.0, 0.97], [0.97, 0.94]])
    c.set_masses([1.0, 1.3])
    if pot == "lj":
        c.set_lj(1.0, 1.0, 2.5)
    elif pot == "plj":
        c.set_plj(e, s, 2.5)
    elif pot == "slj":
        c.set_slj(e, s, 1.6 * s)
    else:
        c.set_wca(e, 2.0 * s)  # cut at 2.2 A
    c.set_skin(0.3)
    v = rng.normal(0.0, V_LIQUID, x.shape)
    if pot == "wca":
        v *= 0.3
    c.set_velocities(v - v.mean(0))
    return 0.005 * TAU


def _box(pot, n, cut):
    a = {"au": 4.078, "agcu": 3.87, "wca": 3.2}.get(pot, (4.0 / 0.8442) ** (1.0 / 3.0))
    x = cm.fcc(n[0], a, n[1], n[2])
    L = np.array(n) * a
    x += np.random.default_rng(2).normal(0.0, 0.01 * a, x.shape)
    x = np.mod(x, L)[:len(x) - cut]
    t = (np.arange(len(x)) % 2 if pot not in ("au", "lj") else np.zeros(len(x))).astype(np.int32)
    return x, t, L


@pytest.mark.parametrize("pot,n,cut", [
    ("lj", (10, 10, 10), 0), ("lj", (8, 9, 10), 3), ("plj", (8, 8, 8), 1), ("slj", (10, 8, 9), 2),
    ("wca", (8, 8, 8), 1), ("au", (8, 8, 9), 1), ("agcu", (9, 8, 8), 15),
])
def test_rows_and_tiles_walk_the_same_path(pot, n, cut):
    x, t, L = _box(pot, n, cut)
    res = []
    for tiled in (False, True):
        with _ctx(tiled) as c:
            c.integrator_vv(_setup(c, pot, x, t, L, (1, 1, 1)))
            c.compute()
            s0 = c.stats()
            assert s0["list_mode"] == 1 and (s0["list_build"] == 3) == (not tiled)
            rows = c.run(60, 30)
            s1 = c.stats()
            assert s1["steps"] == 60 and s1["nupd"] > s0["nupd"]
            res.append([rows, np.array([s1["nupd"]])] + list(c.state()))
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("pot,n,free", [
    ("lj", (8, 8, 8), False), ("plj", (8, 8, 8), False), ("au", (8, 8, 8), False),
    ("lj", (6, 6, 6), True), ("agcu", (5, 5, 4), True), ("agcu", (8, 8, 8), True),
])
@pytest.mark.parametrize("integ", ["vv", "ermak"])
def test_updates_in_and_out_of_the_force_pass(pot, n, free, integ):
    x, t, L = _box(pot, n, 2)
    out = []
    for each in (0, 1):
        with _ctx() as c:
            dt = _setup(c, pot, x, t, None if free else L, (1, 1, 1))
            if pot in ("au", "agcu"):
                dt = 0.001
            if integ == "vv":
                c.integrator_vv(dt)
            else:
                T = 300.0 if pot in ("au", "agcu") else 1.0 / 8.617385e-05
                c.integrator_ermak(dt, T, 0.5, rng=hip.GH_RNG_PHILOX, seed=11)
            c.compute()
            before = c.stats()["nupd"]
            c.run(60, each)
            s = c.stats()
            assert s["steps"] == 60 and s["list_mode"] == (0 if free else 1)
            out.append(list(c.state())[:2] + [s["nupd"] - before])
    assert out[0][2] == out[1][2] > 0
    for a, b, bar in zip(out[0], out[1], (8e-12, 8e-12 / dt)):
        assert np.max(np.abs(a - b)) <= bar
