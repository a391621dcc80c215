"""Small mixed boxes take several workgroups per brick by themselves (as many as
leave each a compute unit): forces, energies and a trajectory are those of one
workgroup per brick, bit for bit, and an explicit shape keeps one.

Sizes: few bricks (split in four), the last brick counts that still split, boxes
with more bricks than half the compute units (one), slabs with empty bricks.
"""
import os

import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


@pytest.mark.parametrize("pot,n,pbc,gap", [
    ("au", 6, (1, 1, 1), 0.0), ("au", 20, (1, 1, 1), 0.0), ("au", 20, (1, 1, 0), 60.0),
    ("au", 26, (1, 1, 1), 0.0), ("agcu", 12, (1, 1, 1), 0.0), ("agcu", 22, (0, 1, 1), 15.0),
    ("lj", 20, (1, 1, 1), 0.0), ("lj", 28, (1, 1, 1), 0.0),
])
def test_default_split(pot, n, pbc, gap):
    a = {"au": 4.078, "agcu": 3.87}.get(pot, (4.0 / 0.8442) ** (1.0 / 3.0))
    x = cm.fcc(n, a)
    rng = np.random.default_rng(n)
    x += rng.normal(0.0, 0.02 * a, x.shape)
    v = rng.normal(0.0, 2.0, x.shape)
    t = (np.arange(len(x)) % 2 if pot == "agcu" else np.zeros(len(x))).astype(np.int32)
    L = n * a + gap * (1 - np.array(pbc))
    res, split = [], []
    for env in ("", "1"):
        if env:
            os.environ["GEMS_HIP_CHUNKS"] = env
        try:
            c = hip.Context(0, hip.GH_MIXED)
        finally:
            os.environ.pop("GEMS_HIP_CHUNKS", None)
        with c:
            c.set_box(L, pbc)
            c.set_atoms(x, t)
            if pot == "lj":
                c.set_masses([1.0])
                c.set_lj(1.0, 1.0, 2.5)
                c.set_skin(0.3)
            else:
                c.set_masses([cm.MASS_AU] if pot == "au" else cm.agcu_masses("Ag"))
                nt = 1 if pot == "au" else 2
                c.set_smatb(nt, *cm.matrices(cm.au_params() if pot == "au" else cm.agcu_params("Ag"), nt))
                c.set_skin(1.0)
            F, e, et = c.compute()
            split.append(c.stats()["chunks"])
            c.set_velocities(v)
            c.integrator_vv(5e-5 if pot == "lj" else 0.002)
            res.append([F, e, np.array([et]), c.run(40, 20), *c.state()])
            if not env:
                c.set_tile(np.array([2, 2, 2]))
                c.compute()
                assert c.stats()["chunks"] == 1
    assert split[1] == 1 and 1 <= split[0] <= 4
    if n < 20:
        assert split[0] == 4
    for p, q in zip(*res):
        assert np.array_equal(p, q)
