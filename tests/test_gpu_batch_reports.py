"""What a batch reports where there is nothing to iterate, little to pair and
much to list.

FIRE without iterations reports the forces it starts from: max|F| of compute()
in the same precision (FP64: the same pair terms summed in another order,
1e-12; mixed: FP32 pair terms, 1e-5 of rms as test_gpu_batch.py, doubled).
"""
import numpy as np
import pytest

from gems_amd import clusters as CL
from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")


def _au(n, seed):
    x = CL.fcc_sphere(n, 4.078, np.array([0.3, 0.1, -0.2]))
    return x + np.random.default_rng(seed).normal(0.0, 0.1, x.shape)


def _smatb(b):
    b.set_smatb(1, *cm.matrices(cm.au_params(), 1))
    b.set_masses([cm.MASS_AU])


@pytest.mark.parametrize("prec,tol", [(hip.GH_FP64, 1e-12), (hip.GH_MIXED, 2e-5)],
                         ids=["fp64", "mixed"])
def test_fire_without_iterations_reports_its_forces(prec, tol):
    sizes = [13, 55, 147]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    x = np.concatenate([_au(n, n) for n in sizes])
    with hip.Batch(0, prec) as b:
        b.set_systems(off, x)
        _smatb(b)
        for earlier in (False, True):  # a new batch, and one that holds a quench's figures
            if earlier:
                b.fire(max_iter=7)
            F, ep = b.compute()
            r = b.fire(max_iter=0)
            f = np.sqrt((F ** 2).sum(1)) * cm.UI_EV
            for s in range(len(sizes)):
                want = f[off[s]:off[s + 1]].max()
                assert abs(r["fmax"][s] - want) <= tol * want
            assert np.all(r["iters"] == 0) and np.all(r["converged"] == 0)
            assert np.allclose(r["epot"], ep, rtol=max(tol, 1e-12), atol=0)


def test_rows_longer_than_32767_pairs():
    # a skin that lists every pair of 36,000 atoms (the pairs outside the inner
    # bound number more than 15 bits); the same pairs are within the cut as with
    # the usual skin: ~45 terms of a few rms(F) at 2^-53 each in another order
    x = _au(36000, 5)
    res = []
    for skin in (1.0, 150.0):
        with hip.Batch(0, hip.GH_FP64) as b:
            b.set_skin(skin)
            b.set_systems(np.array([0, len(x)], np.int32), x)
            _smatb(b)
            res.append(b.compute())
    (F0, e0), (F1, e1) = res
    assert cm.force_err(F1, F0) <= 1e-12
    assert abs(e1[0] - e0[0]) <= 1e-12 * abs(e0[0])


@pytest.mark.parametrize("prec", [hip.GH_FP64, hip.GH_MIXED], ids=["fp64", "mixed"])
def test_types_without_parameters_do_not_interact(prec):
    # an atom whose type the potential has no parameters for: no force on it and
    # none from it, whatever the tables in LDS held before
    rng = np.random.default_rng(2)
    off, x, t = np.array([0, 38, 93], np.int32), np.concatenate([_au(38, 1), _au(55, 2)]), \
        (rng.random(93) < 0.5).astype(np.int32)
    t[[5, 60]] = 3
    keep = t != 3
    many = np.arange(400, dtype=np.int32)
    with hip.Batch(0, prec) as b:  # every entry of the tables filled, on every CU
        b.set_systems(np.concatenate([many, [400]]) * 55, np.tile(_au(55, 2), (400, 1)),
                      np.tile(np.arange(55, dtype=np.int32) % 8, 400))
        b.set_smatb(8, *[m[0, 0] for m in CL.agcu_params()])
        b.set_masses([100.0] * 8)
        b.fire(max_iter=1)
        b.compute()
    res = []
    for sel in (np.ones(93, bool), keep):
        with hip.Batch(0, prec) as b:
            b.set_systems(np.array([0, sel[:38].sum(), sel.sum()], np.int32), x[sel], t[sel])
            b.set_smatb(2, *CL.agcu_params())
            b.set_masses([CL.MASS_AG, CL.MASS_CU])
            F, ep = b.compute()
            r = b.fire(max_iter=0)
            res.append((F, ep, r["epot"]))
    (F, ep, er), (Fk, epk, erk) = res
    tol = 1e-12 if prec == hip.GH_FP64 else 2e-5
    assert np.all(F[~keep] == 0.0)
    assert cm.force_err(F[keep], Fk) <= tol
    assert np.allclose(ep, epk, rtol=tol, atol=0) and np.allclose(er, erk, rtol=tol, atol=0)


@pytest.mark.parametrize("sizes", [[5], [40, 30, 20, 300]])
@pytest.mark.parametrize("why", ["type", "size", "first"])
def test_refused_systems_leave_the_batch_as_it_was(sizes, why):
    off = np.array([0, 13, 68], np.int32)
    x = np.concatenate([_au(13, 1), _au(55, 2)])
    new = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    t = np.zeros(new[-1], np.int32)
    if why == "type":
        t[-1] = 8
    elif why == "size":
        new = np.concatenate([new, new[-1:]])  # a system without atoms
    else:
        new[0] = 1
    with hip.Batch(0, hip.GH_FP64) as b:
        b.set_systems(off, x)
        _smatb(b)
        F, ep = b.compute()
        with pytest.raises(hip.GhError):
            b.set_systems(new, np.zeros((len(t), 3)), t)
        assert np.array_equal(b.state()[0], x)
        F2, ep2 = b.compute()
        assert np.array_equal(F, F2) and np.array_equal(ep, ep2)
