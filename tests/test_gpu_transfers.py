"""State in and out in the caller's order, through pinned buffers (small) and
staged copies (from 16 MiB): what goes in comes out bit for bit after the
atoms were sorted into cells, forces of compute() and state() agree, and a call
that fails writes nothing.
"""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")


def _liquid(nx, drop):
    a = (4.0 / 0.8442) ** (1.0 / 3.0)
    rng = np.random.default_rng(nx)
    x = cm.fcc(nx, a) + rng.normal(0.0, 0.02, (4 * nx ** 3, 3))
    x = np.mod(x, nx * a)
    rng.shuffle(x, axis=0)  # the caller's order is not the cells'
    return x[:len(x) - drop], nx * a, rng


@pytest.mark.parametrize("nx,drop", [(7, 0), (18, 3), (28, 1), (60, 5)],
                         ids=["1372", "23325", "87807", "863995"])
def test_state_round_trip(nx, drop):
    x, L, rng = _liquid(nx, drop)
    v = rng.normal(0.0, 1.0, x.shape)
    with hip.Context(0, hip.GH_FP64) as c:
        c.set_box([L] * 3, (1, 1, 1))
        c.set_atoms(x)
        c.set_masses([1.0])
        c.set_lj(1.0, 1.0, 2.5)
        c.set_skin(0.3)
        c.set_velocities(v)
        F0, e0, et0 = c.compute()
        assert c.stats()["list_mode"] == 1
        xs, vs, Fs, es = c.state()
        assert np.array_equal(xs, x) and np.array_equal(vs, v)
        assert np.array_equal(Fs, F0) and np.array_equal(es, e0)
        assert et0 == pytest.approx(e0.sum(), rel=1e-12)
        # in again, moved, then back where they were
        c.set_positions(np.mod(x + 0.01, L))
        c.set_velocities(-v)
        F1, _, _ = c.compute()
        assert cm.force_err(F1, F0) < 1e-6  # a rigid shift, up to the rounding of x + 0.01
        xs, vs, _, _ = c.state()
        d = xs - np.mod(x + 0.01, L)
        assert np.max(np.abs(d - L * np.round(d / L))) < 1e-12 and np.array_equal(vs, -v)
        c.set_velocities(None)
        assert not c.state()[1].any()


def test_failed_compute_writes_nothing():
    x, L, _ = _liquid(7, 0)
    with hip.Context(0, hip.GH_FP64) as c:
        c.set_box([L, L, 3 * L], (1, 1, 0))
        c.set_atoms(x + [0.0, 0.0, L])
        c.set_masses([1.0])
        c.set_lj(1.0, 1.0, 2.5)
        c.set_skin(0.3)
        c.compute()
        y = x + [0.0, 0.0, L]
        y[5, 2] = 10 * L  # out of the grid
        c.set_positions(y)
        F, e = np.full(x.shape, 7.0), np.full(len(x), 7.0)
        rc = c.L.gh_compute(c.h, hip._p(F), hip._p(e), None)
        assert rc == -5
        assert np.all(F == 7.0) and np.all(e == 7.0)
