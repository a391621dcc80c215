"""A context works on its own device whatever device is current in the thread:
every call that allocates, launches or copies, with another device current, on
a runtime of two devices (fake_hip.c: no hardware, kernels not run).  Atom
counts on both sides of the 2 MiB up to which transfers use pinned buffers.
"""
import os
import subprocess
import sys

from tests.conftest import REPO

DRIVER = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # found before the real runtime
import numpy as np
from gems_amd import hip
from tests import common as cm

bad = []
def calls(who, items):
    for name, f in items:
        fake.hipSetDevice(1)
        fake.fake_faults()
        f()
        if fake.fake_faults():
            bad.append((who, name))

for n in (100, 100000):
    x = np.random.default_rng(1).uniform(0.0, 100.0, (n, 3))
    for box in (None, [100.0] * 3):
        with hip.Context(0, hip.GH_FP64) as a, hip.Context(1, hip.GH_FP64) as b:
            def setup(c):
                c.set_box(box)
                c.set_atoms(x)
                c.set_masses([1.0])
                c.set_smatb(1, *cm.matrices(cm.au_params(), 1))
            calls("ctx %d %s" % (n, box), [
                ("setup", lambda: setup(a)),
                ("compute", a.compute),
                ("state", a.state),
                ("set_positions", lambda: a.set_positions(x)),
                ("set_velocities", lambda: a.set_velocities(x)),
                ("set_accelerations", lambda: a.set_accelerations(x)),
                ("zero velocities", lambda: a.set_velocities(None)),
                ("set_gdist", lambda: a.set_gdist(300.0)),
                ("neighbors", lambda: a.neighbors(8)),
                ("energies", a.energies),
                ("stats", a.stats),
                ("run", lambda: (a.integrator_vv(0.001), a.run(1))),
                ("smatb", lambda: a.set_smatb(1, *cm.matrices(cm.au_params(), 1))),
                ("lj", lambda: a.set_lj(1.0, 1.0, 2.5)),
                ("energies again", a.energies),
                ("lbfgs", lambda: a.lbfgs(max_iter=1)),
            ])
for prec in (hip.GH_FP64, hip.GH_MIXED):
    with hip.Batch(0, prec) as a, hip.Batch(1, prec) as b:
        x = np.random.default_rng(2).uniform(0.0, 10.0, (60, 3))
        lad = np.arange(4).reshape(2, 2)
        calls("batch", [
            ("systems", lambda: a.set_systems([0, 10, 25, 30, 60], x)),
            ("smatb", lambda: a.set_smatb(1, *cm.matrices(cm.au_params(), 1))),
            ("velocities", lambda: a.set_velocities(x)),
            ("temperatures", lambda: a.set_temperatures(np.full(4, 300.0))),
            ("compute", a.compute),
            ("langevin", lambda: a.langevin(3, 0.001, 1.0, 1)),
            ("exchange", lambda: a.exchange(lad, 0, 1)),
            ("fire", lambda: a.fire(max_iter=2)),
            ("state", a.state),
        ])
print("calls on a wrong device:", bad)
sys.exit(1 if bad else 0)
"""


def test_calls_use_their_own_device(tmp_path):
    so = str(tmp_path / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so,
                    os.path.join(REPO, "tests", "fake_hip.c")], check=True)
    r = subprocess.run([sys.executable, "-c", DRIVER, so], cwd=REPO, capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
