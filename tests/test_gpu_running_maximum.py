"""The displacement maximum that the rebuild rule reads is a running one between
builds, also where the grid's first brick (whose workgroup carries it from step
to step) holds no atom.

A cold slab above vacuum, one atom pushed so that it swings out and back within
the skin: after the run the device's maximum must be the largest displacement of
any step, which the same run observed at every step gives (trajectories agree
within 1e-6 A: mixed pair terms, a few hundred femtoseconds from rest).
"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from tests import common as cm
from tests.conftest import REPO

pytestmark = pytest.mark.gpu
hip = pytest.importorskip("gems_amd.hip")

OFFSETS = """
#include <cstddef>
#include <cstdio>
#include "gh_internal.h"
int main() {
  std::printf("%zu %zu %zu %zu", offsetof(gh_ctx, status), offsetof(gh_ctx, step),
              sizeof(GhLine), (size_t)GH_DISP_SLOTS);
}
"""


@pytest.fixture(scope="module")
def maximum(tmp_path_factory):
    """The running maximum (A) of a context, read from its device status."""
    d = tmp_path_factory.mktemp("offsets")
    (d / "o.cpp").write_text(OFFSETS)
    subprocess.run(["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(REPO, "gems_amd", "csrc"), "-o", str(d / "o"),
                    str(d / "o.cpp")], check=True)
    at_status, at_step, line, slots = map(int, subprocess.run(
        [str(d / "o")], capture_output=True, text=True, check=True).stdout.split())
    rt = C.CDLL("libamdhip64.so")

    def read(c):
        status = C.c_void_p.from_address(c.h.value + at_status)
        step = C.c_longlong.from_address(c.h.value + at_step).value
        buf = (C.c_char * (2 * slots * line))()
        assert rt.hipMemcpy(buf, status, len(buf), 2) == 0
        words = np.frombuffer(buf, np.float64).reshape(2, slots, line // 8)[step & 1, :, 0]
        return np.sqrt(words.max())

    return read


@pytest.mark.parametrize("pot", ["au", "agcu"])
@pytest.mark.parametrize("low", [False, True], ids=["full-first-brick", "empty-first-brick"])
def test_maximum_runs_over_the_steps(maximum, pot, low):
    a = {"au": 4.078, "agcu": 3.87}[pot]
    x = cm.fcc(10, a, 10, 8)
    Lz = 30 * a
    x[:, 2] += Lz - 9 * a if low else 0.5 * a
    t = (np.arange(len(x)) % 2).astype(np.int32) if pot == "agcu" else None
    k = int(np.argmin(np.linalg.norm(x - [5 * a, 5 * a, x[:, 2].mean()], axis=1)))
    v = np.zeros_like(x)
    v[k, 0] = 6.0
    got, steps, largest = None, 120, 0.0

    def moved(c):
        d = c.state()[0] - x
        d[:, :2] -= 10 * a * np.round(d[:, :2] / (10 * a))
        return np.linalg.norm(d, axis=1).max()

    for each in (0, 1):
        with hip.Context(0, hip.GH_MIXED) as c:
            c.set_box([10 * a, 10 * a, Lz], (1, 1, 0))
            c.set_atoms(x, t)
            if pot == "au":
                c.set_masses([cm.MASS_AU])
                c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
            else:
                c.set_masses(cm.agcu_masses("Ag"))
                c.set_smatb(2, *cm.matrices(cm.agcu_params("Ag"), 2))
            c.set_skin(0.8)
            c.set_velocities(v)
            c.integrator_vv(0.004)
            c.compute()
            if each == 0:
                c.run(steps)
                assert c.stats()["nupd"] == 1
                got = maximum(c)
                last = moved(c)
            else:
                for _ in range(steps):
                    c.run(1)
                    largest = max(largest, moved(c))
    assert last < largest - 0.01  # it swung back
    assert abs(got - largest) < 1e-6
