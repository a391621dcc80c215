"""Langevin steps of large mixed batches by a workgroup per system, staged in LDS
(144 times the largest system's atoms and more in all), against the passes over all
atoms.

The energies of the last step are those gh_batch_compute, over all atoms, finds
for the same positions (rows rebuilt: sums in another order, 1e-12 relative).
One to eight types, systems below and above a workgroup's 256 atoms a round, and
systems with atoms 64 A and more from their first one, which are not staged.
The first systems alone take the passes over all atoms: 12 steps, FP32 pair
terms that may round the other way after a different FP64 sum, bar 1e-6 A as for
the mixed trajectories of test_gpu_rows.py.
"""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


def _batch(clusters, types, nt):
    off = np.cumsum([0] + [len(c) for c in clusters]).astype(np.int32)
    b = hip.Batch(0, hip.GH_MIXED)
    b.set_systems(off, np.concatenate(clusters), np.concatenate(types))
    A, xi, p, q, r0, rci, rce = cm.matrices(cm.agcu_params("Ag"), 2)
    k = np.arange(nt) % 2
    b.set_smatb(nt, *[np.ascontiguousarray(np.asarray(m).reshape(2, 2)[np.ix_(k, k)])
                      for m in (A, xi, p, q, r0, rci, rce)])
    b.set_masses(np.asarray(cm.agcu_masses("Ag"))[k])
    b.set_skin(0.8)
    b.set_temperatures(np.full(len(clusters), 500.0))
    return b, off


@pytest.mark.parametrize("nt", [1, 2, 8])
def test_staged_systems(nt):
    rng = np.random.default_rng(nt)
    a, clusters, types = 3.87, [], []
    m = 0
    while m < 200000:
        n = int(rng.integers(13, 900))
        c = int(np.ceil((n / 4) ** (1 / 3))) + 2
        x = cm.fcc(c, a) - 0.5 * c * a
        x = x[np.argsort((x * x).sum(1))[:n]] + rng.normal(0.0, 0.04, (n, 3))
        if len(clusters) % 50 == 3:  # two pieces 70 A apart
            x[n // 2:, len(clusters) % 3] += 70.0
        clusters.append(x)
        types.append((rng.permutation(n) % nt).astype(np.int32))
        m += n
    b, off = _batch(clusters, types, nt)
    with b:
        x0 = b.state()[0]
        ep, _ = b.langevin(12, 0.002, 1.0, 5)
        x = b.state()[0]
        _, ec = b.compute()
        assert np.max(np.abs(np.asarray(ep) - np.asarray(ec))) <= 1e-12 * np.max(np.abs(ec))
    assert np.max(np.abs(x - x0)) > 1e-3
    # the random stream is keyed by the atom's number, which the first systems keep
    few = 60
    b, off = _batch(clusters[:few], types[:few], nt)
    with b:
        b.langevin(12, 0.002, 1.0, 5)
        assert np.max(np.abs(b.state()[0] - x[:off[few]])) <= 1e-6
