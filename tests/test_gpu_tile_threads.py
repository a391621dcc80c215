"""Force passes whose workgroups have fewer threads than their brick has atoms
(mixed SMA-TB sizes them to the typical brick, in multiples of 256): every atom
is summed and moved once, whatever round it falls into.

A gold slab of 256,000 atoms (bricks cut by its surfaces, empty ones in the
vacuum) at brick shapes from under one round to over 768 atoms, mixed precision
against FP64: forces within 1e-5 of their rms (the bar of mixed forces), and
after three fused steps of 2 fs positions within 1e-5 rms(F)/m * (6 fs)^2 / 2 of
FP64's, at most 1e-7 A for rms(F) below 1 eV/A.
"""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


def _run(prec, x, v, L, tile):
    with hip.Context(0, prec) as c:
        c.set_box(L, (1, 1, 0))
        c.set_atoms(x, np.zeros(len(x), np.int32))
        c.set_masses([cm.MASS_AU])
        c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        c.set_skin(1.0)
        c.set_tile(np.array(tile))
        F = c.compute()[0]
        c.set_velocities(v)
        c.integrator_vv(0.002)
        c.run(3)
        return F, c.state()[0]


@pytest.mark.parametrize("tile", [(2, 2, 2), (3, 3, 2), (4, 3, 3), (4, 4, 4)])
def test_second_rounds(tile):
    a = 4.078
    x = cm.fcc(40, a)
    rng = np.random.default_rng(sum(tile))
    x += rng.normal(0.0, 0.05, x.shape)
    v = rng.normal(0.0, 1.5, x.shape)
    L = np.array([40 * a, 40 * a, 40 * a + 40.0])
    (F, y), (F64, y64) = (_run(p, x, v, L, tile) for p in (hip.GH_MIXED, hip.GH_FP64))
    rms = np.sqrt(np.mean(F64 ** 2))
    assert np.max(np.abs(F - F64)) <= 1e-5 * rms
    assert np.max(np.abs(y - y64)) <= 1e-7
