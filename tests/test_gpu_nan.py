"""A coordinate that is not a number shows in the forces of the atom and of the
neighbours its list holds, in the free-cluster passes of every potential."""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")


@pytest.mark.parametrize("prec", [hip.GH_FP64, hip.GH_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("pot", ["au", "agcu", "lj", "plj", "slj", "wca"])
@pytest.mark.parametrize("n", [100, 1200])
def test_nan_position_shows_in_the_forces(prec, pot, n):
    a = {"au": 4.078, "agcu": 3.87}.get(pot, 1.68)
    x = cm.fcc(7, a)[:n] + np.random.default_rng(n).normal(0.0, 0.01 * a, (n, 3))
    t = (np.arange(n) % 2).astype(np.int32) if pot not in ("au", "lj") else np.zeros(n, np.int32)
    e, s = np.array([[1.0, 0.9], [0.9, 0.8]]), np.array([[1.0, 0.97], [0.97, 0.94]])
    with hip.Context(0, prec) as c:
        c.set_box(None)
        c.set_atoms(x, t)
        c.set_skin(0.5)
        if pot == "au":
            c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        elif pot == "agcu":
            c.set_smatb(2, *cm.matrices(cm.agcu_params("Ag"), 2))
        elif pot == "lj":
            c.set_lj(1.0, 1.0, 2.5)
        elif pot == "plj":
            c.set_plj(e, s, 2.5)
        elif pot == "slj":
            c.set_slj(e, s, 1.6 * s)
        else:
            c.set_wca(e, 1.2 * s)  # the nearest shell within the cut
        F, _, et = c.compute()
        assert np.all(np.isfinite(F)) and np.isfinite(et)
        k = n // 2
        y = x.copy()
        y[k, 1] = np.nan
        c.set_positions(y)
        F, ea, et = c.compute()
        near = np.linalg.norm(x - x[k], axis=1) < 0.8 * a  # the nearest shell, itself included
        assert near.sum() > 5
        assert np.all(np.isnan(F[near]).any(1)) and np.all(np.isnan(ea[near])) and np.isnan(et)
        c.set_positions(x)
        assert np.all(np.isfinite(c.compute()[0]))
