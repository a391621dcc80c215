"""What a context reports and keeps from one system to the next."""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")


@pytest.mark.parametrize("pot", ["au", "lj"])
def test_longest_row_of_atoms_without_neighbours(pot):
    x = cm.fcc(4, 4.078 if pot == "au" else 1.68)
    lone = np.array([[0.0, 0.0, 0.0], [500.0, 0.0, 0.0]])
    with hip.Context(0, hip.GH_FP64) as c:
        c.set_box(None)
        if pot == "au":
            c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        else:
            c.set_lj(1.0, 1.0, 2.5)
        for y in (x, lone, x, lone[:1]):
            c.set_atoms(y)
            c.compute()
            nn, _ = c.neighbors(cap=256)
            assert c.stats()["maxnn"] == nn.max()
            assert (nn.max() == 0) == (len(y) < 3)


@pytest.mark.parametrize("n", [100, 2000])
@pytest.mark.parametrize("why", ["type", "position"])
def test_refused_atoms_leave_the_context_as_it_was(n, why):
    rng = np.random.default_rng(n)
    x = np.mod(cm.fcc(6, 4.078) + rng.normal(0.0, 0.05, (864, 3)), 6 * 4.078)
    v = rng.normal(0.0, 1.0, x.shape)
    with hip.Context(0, hip.GH_FP64) as c:
        c.set_box([6 * 4.078] * 3, (1, 1, 1))
        c.set_atoms(x)
        c.set_masses([cm.MASS_AU])
        c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        c.set_velocities(v)
        F, e, et = c.compute()
        y, t = rng.uniform(0.0, 20.0, (n, 3)), np.zeros(n, np.int32)
        if why == "type":
            t[n - 1] = 8
        else:
            y[n - 1, 2] = 100.0
        with pytest.raises(hip.GhError):
            c.set_atoms(y, t)
        for a, b in zip(c.state(), (x, v, F, e)):
            assert np.array_equal(a, b)
        assert c.compute()[2] == et


def test_autotune_without_candidates_keeps_the_automatic_choice():
    # cells so full that no brick of four of them fits the LDS: nothing to time
    a = (4.0 / 0.8442) ** (1.0 / 3.0)
    x = cm.fcc(11, a)
    with hip.Context(0, hip.GH_MIXED) as c:
        c.set_box([11 * a] * 3, (1, 1, 1))
        c.set_atoms(x)
        c.set_masses([1.0])
        c.set_lj(1.0, 1.0, 4.2)
        c.set_skin(0.4)
        F, _, _ = c.compute()
        before = c.stats()
        assert before["list_mode"] == 1 and before["chunks"] > 1
        c.autotune(reps=1)
        assert c.stats()["chunks"] == before["chunks"]
        assert cm.force_err(c.compute()[0], F) <= 1e-5
