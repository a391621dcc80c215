"""The FP64 pair terms at the places where their forms change: two atoms at
distances from a third of r0 through the inner bound rci and the cut rce (and
the neighbouring doubles of both), on the tiled and the O(N^2) path, against
the oracle.

Bar: the exponents reach p (1 - r/r0) ~ 7, so a few ulp of them are ~4e-15 of
each of the two terms of the force; the bar is 1e-13 of the larger term (plus
the same share of 1e-6 eV/A where both vanish at the cut).
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests import common as cm

pytestmark = pytest.mark.gpu

hip = pytest.importorskip("gems_amd.hip")


def _distances(rci, rce, r0):
    up, dn = np.nextafter(rci, 9), np.nextafter(rci, 0)
    return [r0 / 3, 0.6 * r0, 0.99 * r0, r0, 1.2 * r0, dn, rci, up, 0.5 * (rci + rce),
            0.999 * rce, np.nextafter(rce, 0)]


@pytest.mark.parametrize("boxed", [True, False], ids=["tiled", "n2"])
def test_smatb_pair_terms_where_the_form_changes(boxed):
    row = cm.au_params()[0]
    A, xi, p, q, r0, rci, rce = row[2:]
    s = O.smatb_params(cm.au_params(), 1)
    L = 40.0
    box = O.make_box([L] * 3, [1, 1, 1]) if boxed else O.make_box(None)
    for r in _distances(rci, rce, r0):
        x = np.array([[10.0, 11.0, 12.0], [10.0 + r, 11.0, 12.0]])
        nn, lst, _ = O.neighbours(x, box, rce + 1.0)
        Fo, eo, _, _ = O.smatb_force(x, np.zeros(2, np.int32), box, s, nn, lst)
        with hip.Context(0, hip.GH_FP64) as c:
            c.set_box([L] * 3 if boxed else None, (1, 1, 1))
            c.set_atoms(x)
            c.set_masses([cm.MASS_AU])
            c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
            c.set_skin(1.0)
            F, e, _ = c.compute()
            assert c.stats()["list_mode"] == (1 if boxed else 0)
        rr = x[1, 0] - x[0, 0]
        term = 2 * A * p / r0 * np.exp(-p * (rr / r0 - 1)) + \
            2 * xi * q / r0 * np.exp(-q * (rr / r0 - 1)) + 1e-6
        assert np.max(np.abs(F - Fo)) <= 1e-13 * term * cm.EV_UI, r
        assert np.max(np.abs(e - eo)) <= 1e-13 * term * r0 * cm.EV_UI, r


@pytest.mark.parametrize("boxed", [True, False], ids=["tiled", "n2"])
def test_atoms_on_one_site_and_a_lone_atom(boxed):
    """Two atoms on one site: energies finite (the exponentials at r = 0),
    forces undefined; the third atom, within the cut of both, keeps a finite
    energy; the energies that diverge at r = 0 are not finite."""
    x = np.array([[10.0, 10.0, 10.0], [10.0, 10.0, 10.0], [13.0, 10.0, 10.0]])
    with hip.Context(0, hip.GH_FP64) as c:
        c.set_box([40.0] * 3 if boxed else None, (1, 1, 1))
        c.set_atoms(x)
        c.set_masses([cm.MASS_AU])
        c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
        c.set_skin(1.0)
        F, e, et = c.compute()
        assert np.all(np.isfinite(e)) and np.isfinite(et)
        assert np.all(np.isnan(F[:2, 0])) and np.all(np.isfinite(F[2]))
        c.set_lj(1.0, 2.5, 6.0)
        F, e, _ = c.compute()
        assert not np.any(np.isfinite(e[:2])) and np.isfinite(e[2])
