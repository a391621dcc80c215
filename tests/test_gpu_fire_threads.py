"""FIRE with 1024, 512 and 256 threads per system (by the number of systems and
the largest one): the same quench whatever the workgroup.

Clusters at both sides of each limit against the same clusters among enough small
ones to take 256 threads.  The forces are the same sums; only the sums over a
system (F.v, |v|^2, |F|^2) round differently, 2^-53 times the square root of 900
atoms a step on velocities that move atoms at most 0.1 A: below 1e-14 A a step,
30 steps and a growth below e^2 give 2.3e-12 A; bar 1e-11.
"""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


def _quench(clusters, nt, prec):
    off = np.cumsum([0] + [len(c) for c in clusters]).astype(np.int32)
    x = np.concatenate(clusters)
    t = np.concatenate([np.arange(len(c)) % nt for c in clusters]).astype(np.int32)
    with hip.Batch(0, prec) as b:
        if nt == 1:
            b.set_masses([cm.MASS_AU])
            b.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        else:
            b.set_masses(cm.agcu_masses("Ag"))
            b.set_smatb(2, *cm.matrices(cm.agcu_params("Ag"), 2))
        b.set_skin(0.8)
        b.set_systems(off, x, t)
        b.fire(max_iter=30)
        return [b.state()[0][off[s]:off[s + 1]] for s in range(len(clusters))]


def _ball(rng, n, a):
    m = int(np.ceil((n / 4) ** (1 / 3))) + 2
    x = cm.fcc(m, a) - 0.5 * m * a
    x = x[np.argsort((x * x).sum(1))[:n]]
    return x + rng.normal(0.0, 0.05, x.shape)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("nt,nsys,sizes", [
    (1, 3, (900, 257, 20)), (1, 256, (130, 64)), (1, 257, (130, 65)), (2, 5, (300, 128, 129)),
    (2, 768, (129, 13)), (2, 769, (129, 13)),
])
def test_same_quench(nt, nsys, sizes, prec):
    rng = np.random.default_rng(nsys + nt)
    a = 4.078 if nt == 1 else 3.87
    few = [_ball(rng, sizes[k % len(sizes)] if k < 6 else 13, a) for k in range(nsys)]
    many = few[:6] + [_ball(rng, 13, a) for _ in range(800)]
    p = hip.GH_FP64 if prec == "fp64" else hip.GH_MIXED
    A, B = _quench(few, nt, p), _quench(many, nt, p)
    for k in range(min(6, nsys)):
        assert np.max(np.abs(A[k] - B[k])) <= 1e-11
