"""A run that stopped inside a step (an atom left the grid) and whose positions
the caller then corrects: the rest of that step, or a force call, uses the
corrected positions with neighbour lists of their own.

Forces against those of a new context at the same positions, whose atoms are
sorted alike: FP64 1e-10 of rms, mixed (fixed point about the bricks' centres)
1e-5, the bars of test_gpu_parity.py.
"""
import numpy as np
import pytest

from tests import common as cm

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")

A = 4.078


def _ctx(prec, x, L):
    c = hip.Context(0, prec)
    c.set_box(L, (1, 1, 0))
    c.set_atoms(x)
    c.set_masses([cm.MASS_AU])
    c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
    c.set_skin(1.0)
    return c


@pytest.mark.parametrize("prec,tol", [(hip.GH_FP64, 1e-10), (hip.GH_MIXED, 1e-5)],
                         ids=["fp64", "mixed"])
@pytest.mark.parametrize("after", [0, 6], ids=["first-step", "seventh-step"])
@pytest.mark.parametrize("then", ["run", "compute"])
def test_corrected_positions_after_a_stop(prec, tol, after, then):
    x = cm.fcc(8, A) + np.random.default_rng(4).normal(0.0, 0.05, (2048, 3))
    L = np.array([8 * A] * 3)
    for d in range(2):
        x[:, d] = np.mod(x[:, d], L[d])
    x[:, 2] = np.clip(x[:, 2], 0.0, L[2] - 1e-9)
    top = int(np.argmax(x[:, 2]))
    with _ctx(prec, x, L) as c:
        c.integrator_vv(0.002)
        if after:
            c.run(after)
        v = c.state()[1]
        v[top, 2] = 5000.0  # 10 A in the next step: past the guard cell
        c.set_velocities(v)
        with pytest.raises(hip.GhError) as err:
            c.run(3)
        assert err.value.code == -5 and c.stats()["steps"] == after
        y, v = c.state()[:2]
        assert y[top, 2] > L[2] + 5.0
        y[top] = x[top] - [0.0, 0.0, 0.05]
        c.set_positions(y)
        v[top] = 0.0
        c.set_velocities(v)
        if then == "run":
            c.run(1)
            assert c.stats()["steps"] == after + 1
            y2, _, F, _ = c.state()
        else:
            F = c.compute()[0]
            y2 = c.state()[0]
    d = y2 - y
    d -= np.array([L[0], L[1], 1e9]) * np.round(d / np.array([L[0], L[1], 1e9]))
    assert np.max(np.abs(d)) < 1e-12
    with _ctx(prec, y2, L) as c:
        F0 = c.compute()[0]
    assert cm.force_err(F, F0) <= tol


def test_new_atoms_after_a_stop_start_a_step_of_their_own():
    x = cm.fcc(8, A) + np.random.default_rng(4).normal(0.0, 0.05, (2048, 3))
    L = np.array([8 * A] * 3)
    x = np.clip(x, 0.0, L - 1e-9)
    v = np.random.default_rng(5).normal(0.0, 1.0, x.shape)
    rows = []
    for stop in (True, False):
        with _ctx(hip.GH_FP64, x, L) as c:
            c.integrator_vv(0.002)
            if stop:
                w = v.copy()
                w[int(np.argmax(x[:, 2])), 2] = 5000.0
                c.set_velocities(w)
                with pytest.raises(hip.GhError):
                    c.run(3)
                c.set_atoms(x)
            c.set_velocities(v)
            rows.append((c.run(4, 1),) + c.state()[:2])
    for a, b in zip(*rows):
        assert np.array_equal(a, b)
