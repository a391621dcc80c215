"""Binning of small boxes by one workgroup, at its limits: 4,096 atoms (four per
thread) and 8,192 cells with guard and padding cells; atoms in shuffled order,
two types, many empty cells, a slab.

A run through rebuilds at a small skin against one at a skin that needs none:
every atom keeps its position, velocity and type.  Both integrate the same
forces, whose sums round differently (1e-15 of coordinates below 200 A, 2^-45,
per step); 30 steps at a growth below e give 30 * 2^-45 * 2.7 = 2.3e-12 A, and
that over a step of 1e-3 ps 2.3e-9 A/ps: bars 1e-11 and 1e-8.  Forces of the first
evaluation against the oracle as in test_gpu_parity.py, 1e-10 of their rms.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")

EPS, SIG, RC = np.array([[0.01, 0.012], [0.012, 0.015]]), np.array([[2.5, 2.6], [2.6, 2.7]]), 6.0


def _ctx(x, t, L, pbc, skin):
    c = hip.Context(0, hip.GH_FP64)
    c.set_box(L, pbc)
    c.set_atoms(x, t)
    c.set_masses([20.0, 40.0])
    c.set_plj(EPS, SIG, RC)
    c.set_skin(skin)
    return c


@pytest.mark.parametrize("n,L,pbc", [
    (4095, 60.0, (1, 1, 1)), (4096, 60.0, (1, 1, 1)), (4097, 60.0, (1, 1, 1)),
    (4096, 60.0, (1, 1, 0)), (700, 122.0, (1, 1, 1)), (700, 160.0, (1, 1, 1)),
    (65, 30.0, (1, 1, 1)),
])
def test_state_through_rebuilds(n, L, pbc):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = rng.permutation(g)[:n]
    x = (g + 0.5 + rng.uniform(-0.1, 0.1, g.shape)) * (L / m)
    t = rng.integers(0, 2, n).astype(np.int32)
    v = rng.normal(0.0, 20.0, x.shape)
    box = np.array([L] * 3) + (1 - np.array(pbc)) * 40.0
    ob = O.make_box(box, pbc)
    p = O.plj_params(EPS, SIG, RC)
    nn, lst, _ = O.neighbours(x, ob, RC + 0.3)
    Fo = O.plj_force(x, t, ob, p, nn, lst)[0]
    out = []
    for skin in (0.3, 3.0):
        with _ctx(x, t, box, pbc, skin) as c:
            F = c.compute()[0]
            assert np.max(np.abs(F - Fo)) <= 1e-10 * np.sqrt(np.mean(Fo ** 2))  # (0 in the sparsest)
            c.set_velocities(v)
            c.integrator_vv(0.001)
            c.run(30)
            out.append(list(c.state()[:2]) + [c.stats()["nupd"], c.stats()["list_mode"]])
    assert out[0][3] == 1 and out[0][2] >= out[1][2] + 2
    d = out[0][0] - out[1][0]
    d -= np.where(np.array(pbc) == 1, np.round(d / box) * box, 0.0)
    assert np.max(np.abs(d)) <= 1e-11
    assert np.max(np.abs(out[0][1] - out[1][1])) <= 1e-8
