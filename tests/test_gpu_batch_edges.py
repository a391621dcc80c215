"""Batched clusters at the edges of their lane groups: systems of 1 to 65
atoms side by side (several in one wavefront, 16, 48 and 64 pairs around the
prefetched part of a row), a system too large for the LDS staging of FIRE, and
one with an atom 64 A and more from the first (beyond the staging's fixed
point).

Bars: forces FP64 1e-10 and mixed 1e-5 of rms against the oracle (as
test_gpu_batch.py); energies reported by a Langevin run against a new batch at
its final positions 1e-12 (FP64: the same arithmetic up to the order of rows);
FIRE energies against the oracle's FIRE 1e-8 eV/atom (as test_gpu_batch.py).
"""
import numpy as np
import pytest

from gems_amd import clusters as CL
from oracle import oracle as O
from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")

SIZES = [1, 2, 3, 13, 15, 16, 17, 38, 47, 63, 64, 65, 1, 55]


def _systems(sizes, seed=3, squeeze=1.0):
    rng = np.random.default_rng(seed)
    xs, ts, off = [], [], [0]
    for n in sizes:
        x = CL.fcc_sphere(n, CL.AGCU["r0"] * np.sqrt(2.0) * squeeze, rng.uniform(-0.4, 0.4, 3))
        xs.append(x + rng.normal(0.0, 0.05, x.shape))
        ts.append((rng.random(n) < 0.5).astype(np.int32))
        off.append(off[-1] + n)
    return np.array(off, np.int32), np.concatenate(xs), np.concatenate(ts)


def _batch(prec, off, x, t, nt):
    b = hip.Batch(0, prec)
    b.set_systems(off, x, t if nt == 2 else np.zeros(len(x), np.int32))
    if nt == 2:
        b.set_smatb(2, *CL.agcu_params())
        b.set_masses([CL.MASS_AG, CL.MASS_CU])
    else:
        b.set_smatb(1, *[m[:1, :1] for m in CL.agcu_params()])
        b.set_masses([CL.MASS_AG])
    return b


def _oracle(nt):
    m = CL.agcu_params()
    rows = [(i, j) + tuple(mm[i, j] for mm in m) for i in range(nt) for j in range(i, nt)]
    return O.smatb_params(rows, nt)


def _check_forces(off, x, t, nt, F, tol):
    s, box = _oracle(nt), O.make_box(None)
    for k in range(len(off) - 1):
        a0, a1 = off[k], off[k + 1]
        if a1 - a0 < 2:
            continue  # a lone atom has no density: its 1/sqrt(rho) is infinite here and there
        tt = t[a0:a1] if nt == 2 else np.zeros(a1 - a0, np.int32)
        nn, lst, _ = O.neighbours(x[a0:a1], box, O.smatb_rcut(s) + 1.0)
        Fo = O.smatb_force(x[a0:a1], tt, box, s, nn, lst)[0]
        assert cm.force_err(F[a0:a1], Fo) <= tol, (k, a1 - a0)


@pytest.mark.parametrize("nt", [1, 2])
@pytest.mark.parametrize("squeeze", [1.0, 0.88], ids=["rows-under-64", "rows-over-64"])
def test_small_systems_side_by_side(nt, squeeze):
    off, x, t = _systems(SIZES + [300] if squeeze < 1 else SIZES, squeeze=squeeze)
    for prec, tol in ((hip.GH_FP64, 1e-10), (hip.GH_MIXED, 1e-5)):
        with _batch(prec, off, x, t, nt) as b:
            F, ep = b.compute()
        _check_forces(off, x, t, nt, F, tol)


def test_many_atoms_take_the_other_lane_count():
    off, x, t = _systems([64] * 3200 + [65, 17])  # 204,882 atoms
    with _batch(hip.GH_FP64, off, x, t, 2) as b:
        F, ep = b.compute()
        b.set_temperatures(np.full(len(off) - 1, 300.0))
        ep1, _ = b.langevin(7, 0.002, 1.0, 5)
        x1, _ = b.state()
    keep = np.r_[0:3, len(off) - 4:len(off) - 1]
    for k in keep:
        a0, a1 = off[k], off[k + 1]
        _check_forces(np.array([0, a1 - a0]), x[a0:a1], t[a0:a1], 2, F[a0:a1], 1e-10)
    with _batch(hip.GH_FP64, off, x1, t, 2) as b:
        assert np.allclose(b.compute()[1], ep1, rtol=1e-12, atol=0)


@pytest.mark.parametrize("steps", [1, 2, 31])
def test_langevin_leaves_the_state_it_reports(steps):
    off, x, t = _systems([n for n in SIZES if n > 2])
    with _batch(hip.GH_FP64, off, x, t, 2) as b:
        b.set_temperatures(np.full(len(off) - 1, 900.0))
        b.langevin(5, 0.002, 1.0, 4)
        ep, ek = b.langevin(steps, 0.002, 1.0, 5)
        b.set_skin(0.6)  # new rows for the next call
        b.langevin(0, 0.002, 1.0, 5)
        x1, v1 = b.state()
    with _batch(hip.GH_FP64, off, x1, t, 2) as b:
        assert np.allclose(b.compute()[1], ep, rtol=1e-12, atol=0)
    m = np.where(t == 0, CL.MASS_AG, CL.MASS_CU)
    for k in range(len(off) - 1):
        a = slice(off[k], off[k + 1])
        cmv = (m[a, None] * v1[a]).sum(0) / m[a].sum()
        assert ek[k] == pytest.approx(
            0.5 * (m[a, None] * (v1[a] - cmv) ** 2).sum() * cm.UI_EV, rel=1e-12)


@pytest.mark.parametrize("case", ["far-atom", "large"])
def test_mixed_systems_outside_the_staging(case):
    if case == "far-atom":
        off, x, t = _systems([55, 40])
        x[54] += 80.0  # alone, 80 A away on each axis ...
        x[53] = x[54] + [2.6, 0.0, 0.0]  # ... but for one neighbour
    else:
        off, x, t = _systems([4000, 38])
    with _batch(hip.GH_MIXED, off, x, t, 1) as b:
        F, ep = b.compute()
        _check_forces(off, x, t, 1, F, 1e-5)
        r = b.fire(max_iter=3, fswitch=1e-9)
        xm, _ = b.state()
    with _batch(hip.GH_FP64, off, x, t, 1) as b:
        b.fire(max_iter=3)
        xd, _ = b.state()
    assert np.all(r["iters"] == 3)
    # three steps of at most 0.6 fs: displacements ~1e-3 A, mixed forces within 1e-5
    assert np.max(np.abs(xm - xd)) < 1e-7
    assert np.max(np.abs(xd - x)) > 1e-5
