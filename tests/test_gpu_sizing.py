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
