"""The O(N^2) list mode at the edges of its wavefronts: atom counts around the
64 candidates of a step and the changes of rows per wavefront (1, 4, 8), rows
longer than one round of 64 entries, against brute force and the oracle.

Bars as in test_gpu_parity.py: neighbour sets exact, FP64 forces within 1e-10
of rms, mixed within 1e-5.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


@pytest.mark.parametrize("n,spacing", [(1, 1.1), (2, 1.1), (63, 0.8), (64, 0.8), (65, 1.1),
                                       (1024, 0.9), (1025, 0.9), (8193, 1.1)])
def test_free_cluster_rows_and_forces(n, spacing):
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = spacing * g + np.random.default_rng(n).normal(0.0, 0.03, (n, 3))
    rl = 2.5 + 0.3
    rows = []
    for i in range(n):
        u = x - x[i]
        rows.append(set(np.nonzero((u * u).sum(1) <= rl * rl)[0]) - {i})
    box = O.make_box(None)
    nn, lst, _ = O.neighbours(x, box, rl)
    Fo, eo, epo = O.lj_force(x, box, 1.0, 1.0, 2.5, nn, lst)
    for prec, tol in ((hip.GH_FP64, 1e-10), (hip.GH_MIXED, 1e-5)):
        with hip.Context(0, prec) as c:
            c.set_box(None)
            c.set_atoms(x)
            c.set_masses([1.0])
            c.set_lj(1.0, 1.0, 2.5)
            c.set_skin(0.3)
            F, e, et = c.compute()
            gnn, gidx = c.neighbors(cap=512)
            assert c.stats()["list_mode"] == 0
        for i in range(n):
            assert set(gidx[i, :gnn[i]]) == rows[i], i
        if n == 1:
            assert np.all(F == 0.0) and et == 0.0
            continue
        assert cm.force_err(F, Fo) <= tol
        assert np.max(np.abs(e - eo)) <= tol * np.max(np.abs(eo))
