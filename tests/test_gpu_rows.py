"""Passes over rows of atom numbers (smaller FP64 boxes) against the tiled
passes on the same box, and integrator updates inside the force pass against
those of their own kernels.

The tiled path (GEMS_HIP_LIST_BUILD=coop) lists the same neighbours in the same
order and sums them in the same order: forces, energies and trajectories
through rebuilds agree bit for bit, and so does where a run that outgrows the
rows stops (the dense liquids' steps are long).  Cases: one and two types, every pair
potential's kernel, slabs (guard cells), cells without atoms, atom counts that
leave a group of 16 lanes or a whole workgroup idle, the first count beyond the
rows and the last within.

Updates: `each=1` observes every step, which keeps the update out of the force
pass.  Their arithmetic differs at most by the contraction of a few products: 5
roundings a step of coordinates below 128 A (2^-46 each) over 60 steps, and a
growth of at most e^2 in 60 fs: bar 60 * 5 * 1.5e-14 * 7.4 = 3.3e-11 A,
velocities that over one step (1e-3 ps) 3.3e-8 A/ps.
"""
import os

import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


def _ctx(tiled, prec=None):
    if tiled:
        os.environ["GEMS_HIP_LIST_BUILD"] = "coop"
    try:
        return hip.Context(0, hip.GH_FP64 if prec is None else prec)
    finally:
        os.environ.pop("GEMS_HIP_LIST_BUILD", None)


def _pot(c, pot):
    if pot == "au":
        c.set_masses([cm.MASS_AU])
        c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        c.set_skin(1.0)
    elif pot == "agcu":
        c.set_masses(cm.agcu_masses("Ag"))
        c.set_smatb(2, *cm.matrices(cm.agcu_params("Ag"), 2))
        c.set_skin(1.0)
    else:
        c.set_masses([1.0, 1.3])
        e, s = np.array([[1.0, 0.9], [0.9, 0.8]]), np.array([[1.0, 0.97], [0.97, 0.94]])
        if pot == "lj":
            c.set_lj(1.0, 1.0, 2.5)
        elif pot == "plj":
            c.set_plj(e, s, 2.5)
        else:
            c.set_slj(e, s, 1.6 * s)
        c.set_skin(0.3)


def _box(pot, n, cut=0, seed=1, gap=0.0):
    a = {"au": 4.078, "agcu": 3.87}.get(pot, (4.0 / 0.8442) ** (1.0 / 3.0))
    nx, ny, nz = n
    x = cm.fcc(nx, a, ny, nz)
    x += np.random.default_rng(seed).normal(0.0, 0.02 * a, x.shape)
    x = x[:len(x) - cut]
    t = (np.arange(len(x)) % 2 if pot != "au" and pot != "lj" else np.zeros(len(x))).astype(np.int32)
    return x, t, np.array([nx * a, ny * a, nz * a + gap])


@pytest.mark.parametrize("pot,n,cut,pbc,gap,steps", [
    ("au", (8, 8, 8), 0, (1, 1, 1), 0.0, 60),
    ("au", (8, 7, 9), 1, (1, 1, 0), 30.0, 60),
    ("agcu", (9, 8, 8), 15, (1, 1, 1), 0.0, 60),
    ("agcu", (8, 8, 8), 17, (0, 1, 1), 20.0, 0),
    ("lj", (10, 10, 10), 3, (1, 1, 1), 0.0, 60),
    ("plj", (8, 8, 8), 1, (1, 1, 1), 0.0, 60),
    ("slj", (8, 9, 10), 2, (1, 1, 0), 9.0, 0),
    ("au", (32, 32, 32), 1, (1, 1, 1), 0.0, 0),
    ("au", (32, 32, 32), 0, (1, 1, 1), 0.0, 0),
    ("lj", (26, 26, 26), 4769, (1, 1, 1), 0.0, 0),
    ("lj", (26, 26, 26), 4768, (1, 1, 1), 0.0, 0),
])
def test_rows_match_tiles(pot, n, cut, pbc, gap, steps):
    x, t, L = _box(pot, n, cut, gap=gap)
    res = []
    for tiled in (False, True):
        with _ctx(tiled) as c:
            c.set_box(L, pbc)
            c.set_atoms(x, t)
            _pot(c, pot)
            F, e, et = c.compute()
            assert c.stats()["list_mode"] == 1
            within = len(x) < (131072 if pot == "au" else 65536)
            assert (c.stats()["list_build"] == 3) == (within and not tiled)
            out = [F, e, np.array([et])]
            if len(x) < 5000:
                nn, idx = c.neighbors(cap=256)
                out += [nn, idx]
            if steps:
                c.set_velocities(np.random.default_rng(3).normal(0.0, 8.0 if gap else 5.0, x.shape))
                c.integrator_vv(0.002)
                try:
                    out += [c.run(steps, steps // 2)]
                except hip.GhError as err:  # (a close collision outgrew the row capacity)
                    assert "row capacity" in str(err)
                    out += [np.array([str(err).split(" at ")[1]])]
                out += list(c.state())
                out += [np.array([c.stats()["nupd"]])]
            res.append(out)
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,cut", [((32, 32, 32), 0), ((46, 46, 47), 4592), ((46, 46, 47), 4593)])
def test_rows_match_tiles_two_types_large(n, cut):
    # several types keep the rows where the tiles take one lane per atom: the
    # same pairs summed in another order, ~60 terms of up to a few rms(F) at 2^-53
    x, t, L = _box("agcu", n, cut)
    res = []
    for tiled in (False, True):
        with _ctx(tiled) as c:
            c.set_box(L, (1, 1, 1))
            c.set_atoms(x, t)
            _pot(c, "agcu")
            res.append(c.compute())
            assert (c.stats()["list_build"] == 3) == (not tiled and len(x) < 393216)
    (F, e, et), (F2, e2, et2) = res
    assert np.max(np.abs(F - F2)) <= 1e-13 * 60 * np.sqrt(np.mean(F2 ** 2))
    assert np.max(np.abs(e - e2)) <= 1e-13 * np.max(np.abs(e2)) and abs(et - et2) <= 1e-13 * abs(et2)


@pytest.mark.parametrize("pot,n,kind,prec", [
    ("au", (5, 5, 4), "free", "fp64"), ("agcu", (5, 5, 4), "free", "fp64"),
    ("au", (7, 7, 6), "free", "fp64"), ("au", (5, 5, 4), "free", "mixed"),
    ("agcu", (7, 7, 6), "free", "mixed"), ("lj", (6, 6, 6), "free", "fp64"),
    ("au", (8, 8, 8), "box", "fp64"), ("lj", (8, 8, 8), "box", "fp64"),
])
@pytest.mark.parametrize("integ", ["vv", "ermak"])
def test_update_inside_the_force_pass(pot, n, kind, prec, integ):
    x, t, L = _box(pot, n, 2)
    v = np.random.default_rng(5).normal(0.0, 3.0, x.shape)
    out = []
    for each in (0, 1):
        with _ctx(False, hip.GH_MIXED if prec == "mixed" else hip.GH_FP64) as c:
            c.set_box(L if kind == "box" else None, *([(1, 1, 1)] if kind == "box" else []))
            c.set_atoms(x, t)
            _pot(c, pot)
            c.set_velocities(v)
            if integ == "vv":
                c.integrator_vv(0.001)
            else:
                c.integrator_ermak(0.001, 300.0, 0.5, rng=hip.GH_RNG_PHILOX, seed=11)
            stop = ""
            try:
                c.run(60, each)
            except hip.GhError as err:  # as above
                assert "row capacity" in str(err)
                stop = str(err).split(" at ")[1]
            out.append(list(c.state())[:2] + [stop])
            assert c.stats()["list_mode"] == (1 if kind == "box" else 0)
    bars = (3.3e-11, 3.3e-8)
    if prec == "mixed":
        # the FP32 pair terms of coordinates that differ by the bar may round the
        # other way: 2^-24 of a pair force below 3 eV/A, 50 pairs, on 1/2 dt^2
        # of 60 steps and the same growth
        bars = (1e-6, 1e-3)
    assert out[0][2] == out[1][2]
    for a, b, bar in zip(out[0], out[1], bars):
        assert np.max(np.abs(a - b)) <= bar
