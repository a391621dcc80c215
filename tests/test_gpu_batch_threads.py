"""Mixed Langevin batches by a workgroup per system at the edges of its rules: a
few tiny systems, systems at one and a half times a workgroup's threads (one
lane per atom from there on, four below), both kinds in one batch, the largest
system whose staging still fits, each through row builds.

Against the passes over all atoms, which the same systems take beside a large
one at the end (the random stream is keyed by the atom's number): 25 steps, FP32
pair terms that may round the other way after a different FP64 sum, bar 1e-6 A
as for the mixed trajectories of test_gpu_rows.py.  The energies reported are
those gh_batch_compute finds at the final positions: 1e-12 relative.
"""
import numpy as np
import pytest

from gems_amd import clusters as CL

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")


def _systems(sizes, seed=1):
    rng, form, xs = np.random.default_rng(seed), {}, []
    for n in sizes:
        if n not in form:
            form[n] = CL.fcc_sphere(n, CL.AGCU["r0"] * np.sqrt(2.0), rng.uniform(-0.4, 0.4, 3))
        xs.append(form[n] + rng.normal(0.0, 0.05, (n, 3)))
    x = np.concatenate(xs)
    return np.cumsum([0] + list(sizes)).astype(np.int32), x, (rng.random(len(x)) < 0.5).astype(np.int32)


def _batch(off, x, t, nt, prec=hip.GH_MIXED):
    b = hip.Batch(0, prec)
    b.set_systems(off, x, t if nt == 2 else None)
    m = CL.agcu_params()
    b.set_smatb(nt, *(m if nt == 2 else [q[:1, :1] for q in m]))
    b.set_masses([CL.MASS_AG, CL.MASS_CU][:nt])
    b.set_skin(0.1)
    b.set_temperatures(np.full(len(off) - 1, 900.0))
    return b


@pytest.mark.parametrize("nt", [1, 2])
@pytest.mark.parametrize("sizes,large", [
    ([13], 100), ([1, 2, 32, 31, 17, 16], 100), ([32] * 300, 400),
    ([191, 192, 193] * 360, 2000), ([150, 250, 60] * 400, 2000), ([800, 767, 768] * 100, 2400),
    ([3799] * 144, 0),
], ids=["one", "tiny", "32", "192-of-128", "both", "768-of-512", "3799"])
def test_workgroup_per_system(sizes, large, nt):
    if large == 0 and nt == 2:
        pytest.skip("the tables of two types leave less room for the staging")
    sizes = sorted(sizes, key=lambda n: (n * 7919) % 101)  # in no order of size
    off, x, t = _systems(sizes)
    with _batch(off, x, t, nt) as b:
        ep, _ = b.langevin(25, 0.002, 1.0, 5)
        y = b.state()[0]
        ec = b.compute()[1]
        many = np.diff(off) > 1  # (a lone atom has no density)
        assert np.allclose(ep[many], ec[many], rtol=1e-12, atol=0)
        assert np.max(np.abs(y - x)) > 0.05  # half the skin: rows were built
    if large:
        off2, x2, t2 = _systems([large], seed=2)
        off2 = np.concatenate([off, [off[-1] + large]]).astype(np.int32)
        with _batch(off2, np.concatenate([x, x2]), np.concatenate([t, t2]), nt) as b:
            b.langevin(25, 0.002, 1.0, 5)
            z = b.state()[0][:len(x)]
        a = np.repeat(many, np.diff(off))
        assert np.max(np.abs(z[a] - y[a])) <= 1e-6


@pytest.mark.parametrize("n", [3799, 3800])
def test_largest_staged_system_quenches(n):
    # mixed FIRE with the largest staging and beyond it, against FP64: three steps
    # of at most 0.6 fs from forces within 1e-5
    off, x, t = _systems([n, 13])
    out = []
    for prec in (hip.GH_MIXED, hip.GH_FP64):
        with _batch(off, x, t, 1, prec) as b:
            r = b.fire(max_iter=3, fswitch=1e-9)
            out.append(b.state()[0])
            assert np.all(r["iters"] == 3)
    assert np.max(np.abs(out[0] - out[1])) < 1e-7
    assert np.max(np.abs(out[1] - x)) > 1e-5


@pytest.mark.parametrize("prec,bar", [(hip.GH_FP64, 1e-11), (hip.GH_MIXED, 1e-6)],
                         ids=["fp64", "mixed"])
@pytest.mark.parametrize("nt", [1, 2])
@pytest.mark.parametrize("edge,others", [((383, 384, 385), [384] * 557), ((767, 768, 769), [768] * 297),
                                         ((1535, 1536, 1537), [1000] * 300)],
                         ids=["384-of-256", "768-of-512", "1536-of-1024"])
def test_quench_with_one_lane_and_four(edge, others, nt, prec, bar):
    # the same quench alone (1,024 threads) and among many: FP64 forces sum the same
    # pairs in another order, 2^-53 of a few eV/A over 30 steps as in
    # test_gpu_fire_threads.py; mixed as above
    off, x, t = _systems(list(edge))
    off2, x2, t2 = _systems(others, seed=2)
    out = []
    for o, y, ty in ((off, x, t), (np.concatenate([off, off[-1] + off2[1:]]).astype(np.int32),
                                   np.concatenate([x, x2]), np.concatenate([t, t2]))):
        with _batch(o, y, ty, nt, prec) as b:
            r = b.fire(max_iter=30)
            out.append((b.state()[0][:len(x)], r["epot"][:3], r["fmax"][:3]))
    assert np.max(np.abs(out[0][0] - x)) > 0.01
    assert np.max(np.abs(out[0][0] - out[1][0])) <= bar
    assert np.allclose(out[0][1], out[1][1], rtol=bar, atol=0)
