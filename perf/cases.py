"""What this library is used for, as cases that can be timed and checked.

A case names one of the ways a program drives the library:

``static``    forces of one small free cluster from device arrays, nothing
              allocated (``gh_cluster_forces_static``: code under graph
              capture, serving loops)
``forces``    the host integrates, minimises or samples: new positions in,
              forces, per-atom energies and the total out
              (``Context.set_positions`` + ``compute``: GEMS's interaction
              plugin at each ``interact()``)
``md``        velocity Verlet on the device between two outputs: state in, a
              chunk of steps with its energy rows, state out
              (``Context.run``: GEMS's ``dinamica`` loop)
``langevin``  the same with the Ermak integrator and the device's random
              stream
``re``        a replica-exchange interval of many free clusters at once and
              the exchange that follows it (``Batch.langevin``, ``exchange``)
``fire``      a quench of many clusters with a budget of iterations
              (``Batch.fire``)

Systems: ``au`` (SMA-TB gold), ``agcu`` (SMA-TB silver-copper, two types),
``lj`` (the unshifted Lennard-Jones liquid) and ``plj`` (the shifted form, two
types); periodic crystals with vacancies (so that atom counts are odd), slabs
with two free faces, and free clusters.
"""
import ctypes as C
import math

import numpy as np
import torch

from gems_amd import hip

# units (src/Constants.F90): energies in ui = amu A^2 / ps^2
UI_EV = 1.0e2 * 1.0e2 * 1.6605402e-27 / 1.60219e-19
KB_UI = 8.617385e-05 / UI_EV
TAU = 0.01018047  # ps: sqrt(m sigma^2 / eps) of the Lennard-Jones cases

AG = (0.1028, 1.178, 10.928, 3.139, 2.889)
CU = (0.0855, 1.224, 10.960, 2.278, 2.556)
AGCU = (0.0980, 1.2274, 10.700, 2.805, 2.7224)
AU_LAT, ALLOY_LAT, LJ_LAT = 4.078, 3.87, (4.0 / 0.8442) ** (1.0 / 3.0)
M_AU, M_AG, M_CU = (float(np.float32(m)) for m in (196.97, 107.87, 63.55))


def _smatb(system):
    """nt and the seven nt x nt parameter tables (A, xi, p, q, r0, rci, rce)."""
    if system == "au":
        row = (0.2061, 1.790, 10.229, 4.036, 2.884, AU_LAT, AU_LAT * math.sqrt(1.5))
        return 1, [np.full((1, 1), v) for v in row]
    out = [np.zeros((2, 2)) for _ in range(7)]
    for i, j, row in ((0, 0, AG), (1, 1, CU), (0, 1, AGCU), (1, 0, AGCU)):
        for k, v in enumerate(row + (row[4] * math.sqrt(2.0), row[4] * math.sqrt(3.0))):
            out[k][i, j] = v
    return 2, out


PLJ_EPS = np.array([[1.0, 0.8], [0.8, 0.6]])
PLJ_SIG = np.array([[1.0, 0.95], [0.95, 0.9]])
PLJ_RC, LJ_RC = 2.5, 2.5
MASS = {"au": [M_AU], "agcu": [M_AG, M_CU], "lj": [1.0], "plj": [1.0, 0.5]}
LAT = {"au": AU_LAT, "agcu": ALLOY_LAT, "lj": LJ_LAT, "plj": LJ_LAT}
SKIN = {"au": 1.0, "agcu": 1.0, "lj": 0.3, "plj": 0.3}
JITTER = {"au": 0.05, "agcu": 0.05, "lj": 0.05, "plj": 0.05}
# temperature (K): solids at room temperature and above, the liquids at T* = 1.0
TEMP = {"au": 300.0, "agcu": 600.0, "lj": 1.0 / 8.617385e-05, "plj": 1.0 / 8.617385e-05}
DT = {"au": 0.002, "agcu": 0.002, "lj": 0.005 * TAU, "plj": 0.005 * TAU}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _bulk(kind, system, cells, precision, vac=0, steps=0, each=0, slab=False, tile=""):
    return dict(kind=kind, system=system, nx=cells[0], ny=cells[1], nz=cells[2], vac=vac,
                precision=precision, steps=steps, each=each, slab=slab, tile=tile)


def listed():
    return [
        # one small alloy cluster in a serving loop: launches and latency
        dict(name="static_agcu_201", kind="static", system="agcu", n=201, precision="fp64"),
        # GEMS's own minimiser or sampler on a free cluster: one call per trial
        dict(name="forces_cluster_561", kind="forces", system="agcu", n=561, precision="fp64"),
        # GEMS integrates on the host: each step sends positions and takes forces
        dict(_bulk("forces", "au", (20, 20, 20), "fp64"), name="forces_au_32k"),
        # the same for a large alloy in mixed precision, with 37 vacancies
        dict(_bulk("forces", "agcu", (48, 48, 48), "mixed", vac=37), name="forces_alloy_442k"),
        # Langevin dynamics of one free cluster
        dict(name="langevin_cluster_201", kind="langevin", system="agcu", n=201,
             precision="fp64", steps=100, each=50),
        # Langevin dynamics of a small periodic crystal (the bulk example's 4000 atoms)
        dict(_bulk("langevin", "au", (10, 10, 10), "fp64", steps=100, each=50),
             name="langevin_au_4000"),
        # the Lennard-Jones liquid at 4000 atoms: a rebuild every dozen steps
        dict(_bulk("md", "lj", (10, 10, 10), "fp64", steps=200, each=100), name="md_lj_4000"),
        # 32,000 gold atoms between two energy rows
        dict(_bulk("md", "au", (20, 20, 20), "fp64", steps=200, each=100), name="md_au_32k"),
        # the headline: a million gold atoms in mixed precision, shape kept from a tuning run
        dict(_bulk("md", "au", (63, 63, 63), "mixed", steps=500, each=100, tile="4,3,3"),
             name="md_au_1m_mixed"),
        # a large liquid in FP64: list builds count as much as forces
        dict(_bulk("md", "lj", (64, 64, 64), "fp64", vac=5, steps=100, each=100, tile="3,2,2"),
             name="md_lj_1m"),
        # replica exchange: 16 geometries x 8 rungs, one interval and its exchange
        dict(name="re_128_mixed", kind="re", geoms=16, rungs=8, nmin=38, nmax=2000,
             precision="mixed", steps=50),
        # quench of a batch of gold clusters
        dict(name="fire_1024_mixed", kind="fire", nsys=1024, nmin=13, nmax=309,
             precision="mixed", steps=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["static", "forces", "forces", "md", "md", "md", "langevin", "re", "fire"])
    precision = rng.choice(["fp64", "fp64", "mixed"])
    if kind == "static":
        return dict(kind=kind, system=rng.choice(["au", "agcu"]), n=_log(rng, 13, 2048),
                    precision=precision)
    if kind == "re":
        return dict(kind=kind, geoms=rng.randint(2, 16), rungs=rng.randint(2, 8), nmin=38,
                    nmax=rng.choice([150, 600, 2000]), precision=precision,
                    steps=rng.randint(20, 50))
    if kind == "fire":
        return dict(kind=kind, nsys=_log(rng, 32, 1024), nmin=13, nmax=rng.choice([55, 147, 309]),
                    precision=precision, steps=rng.randint(30, 100))
    steps = 0 if kind == "forces" else rng.randint(50, 200)
    each = 0 if kind == "forces" else max(1, steps // rng.choice([1, 2, 5]))
    if rng.random() < 0.3:  # a free cluster
        return dict(kind=kind, system=rng.choice(["au", "agcu"]), n=_log(rng, 13, 2000),
                    precision="fp64" if kind == "langevin" else precision, steps=steps, each=each)
    system = rng.choice(["au", "au", "agcu", "lj", "plj"])
    n = _log(rng, 864, 600000 if kind != "langevin" else 60000)
    m = max(6, int(round((n / 4.0) ** (1.0 / 3.0))))
    cells = [max(6, m + rng.randint(-1, 1)) for _ in range(3)]
    return _bulk(kind, system, cells, "fp64" if kind == "langevin" else precision,
                 vac=rng.randint(0, 50), steps=steps, each=each,
                 slab=system in ("au", "agcu") and m >= 8 and rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _rng(seed):
    return np.random.default_rng([20260101, int(seed)])


def _fcc_sphere(n, a, center):
    """The n fcc sites nearest a centre point, about it."""
    m = int(math.ceil((3.0 * n / (16.0 * math.pi)) ** (1.0 / 3.0))) + 2
    r = np.arange(-m, m + 1, dtype=np.float64)
    g = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0, 0.5, 0.5], [0.5, 0, 0.5]])
    p = (g[:, None, :] + base[None, :, :]).reshape(-1, 3) * a - center
    return p[np.argsort((p * p).sum(1), kind="stable")[:n]]


def _cluster(rng, system, n, jitter):
    a = {"au": AU_LAT, "agcu": AGCU[4] * math.sqrt(2.0)}[system]
    x = _fcc_sphere(n, a, rng.uniform(-0.5, 0.5, 3) * a) + rng.normal(0.0, jitter, (n, 3))
    t = np.zeros(n, np.int32)
    if system == "agcu":
        t[n // 2:] = 1
        rng.shuffle(x, axis=0)
    return x, t


def _velocities(rng, system, t, T):
    m = np.asarray(MASS[system])[t]
    v = rng.normal(0.0, 1.0, (len(t), 3)) * np.sqrt(KB_UI * T / m)[:, None]
    return v - (m[:, None] * v).sum(0) / m.sum()


def _inputs(case, seed):
    """(box or None, pbc, x, types, v) of one system."""
    rng, s = _rng(seed), case["system"]
    if "n" in case:
        x, t = _cluster(rng, s, case["n"], 0.05)
        return None, (0, 0, 0), x, t, _velocities(rng, s, t, TEMP[s])
    a = LAT[s]
    cells = np.array([case["nx"], case["ny"], case["nz"]])
    g = np.stack(np.meshgrid(*[np.arange(c, dtype=np.float64) for c in cells[::-1]],
                             indexing="ij"), -1)[..., ::-1].reshape(-1, 3)
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0, 0.5, 0.5], [0.5, 0, 0.5]])
    x = ((g[:, None, :] + base[None, :, :]).reshape(-1, 3)) * a
    L = cells * a
    pbc = (1, 1, 1)
    if case["slab"]:  # two free faces normal to z, a third of the box vacuum
        L = L * np.array([1.0, 1.0, 1.5])
        x[:, 2] += cells[2] * a * 0.25
        pbc = (1, 1, 0)
    x += rng.normal(0.0, JITTER[s], x.shape)
    if case["vac"]:
        keep = np.ones(len(x), bool)
        keep[rng.choice(len(x), case["vac"], replace=False)] = False
        x = x[keep]
    for d in range(3):
        if pbc[d]:
            x[:, d] = np.mod(x[:, d], L[d])
    t = np.zeros(len(x), np.int32)
    if len(MASS[s]) == 2:
        t[rng.random(len(x)) < 0.5] = 1
    return L, pbc, np.ascontiguousarray(x), t, _velocities(rng, s, t, TEMP[s])


def _re_inputs(case, seed):
    rng = _rng(seed)
    G, R = case["geoms"], case["rungs"]
    sizes = np.round(np.geomspace(case["nmax"], case["nmin"], G)).astype(int)
    xs, ts, vs, off = [], [], [], [0]
    T = 300.0 * 3.0 ** (np.arange(R) / max(R - 1, 1))
    for n in sizes:
        x, t = _cluster(rng, "agcu", int(n), 0.05)
        for r in range(R):
            xs.append(x)
            ts.append(t)
            vs.append(_velocities(rng, "agcu", t, T[r]))
            off.append(off[-1] + int(n))
    lad = np.arange(G * R, dtype=np.int32).reshape(G, R)
    return np.array(off, np.int32), np.concatenate(xs), np.concatenate(ts), np.concatenate(vs), \
        np.tile(T, G), lad


def _fire_inputs(case, seed):
    rng = _rng(seed)
    # sizes over the whole range in no order, the same for every seed
    sizes = np.random.default_rng(7).integers(case["nmin"], case["nmax"] + 1, case["nsys"])
    xs = [_cluster(rng, "au", int(n), 0.1)[0] for n in sizes]
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32), np.concatenate(xs)


class _State:
    pass


def _context(case, seed):
    L, pbc, x, t, v = _inputs(case, seed)
    s = case["system"]
    c = hip.Context(0, hip.GH_MIXED if case["precision"] == "mixed" else hip.GH_FP64)
    c.set_box(L, pbc)
    c.set_atoms(x, t)
    c.set_masses(MASS[s])
    if s == "lj":
        c.set_lj(1.0, 1.0, LJ_RC)
    elif s == "plj":
        c.set_plj(PLJ_EPS, PLJ_SIG, PLJ_RC)
    else:
        nt, tables = _smatb(s)
        c.set_smatb(nt, *tables)
    c.set_skin(SKIN[s])
    if case.get("tile"):
        c.set_tile([int(k) for k in case["tile"].split(",")])
    return c, x, v


def prepare(case, seed):
    """The context or batch with its atoms and potential set, and the host
    arrays the next call sends; device arrays and parameter tables for
    ``static``."""
    S = _State()
    S.kind, S.case = case["kind"], case
    prec = hip.GH_MIXED if case["precision"] == "mixed" else hip.GH_FP64
    if S.kind == "static":
        _, _, x, t, _ = _inputs(case, seed)
        n, nt, tables = len(x), *_smatb(case["system"])
        S.x = torch.from_numpy(np.ascontiguousarray(x).reshape(-1)).cuda()
        S.t = torch.from_numpy(t).cuda()
        S.F = torch.empty(3 * n, dtype=torch.float64, device="cuda")
        S.e = torch.empty(n, dtype=torch.float64, device="cuda")
        S.ep = torch.empty(1, dtype=torch.float64, device="cuda")
        S.st = torch.empty(1, dtype=torch.int32, device="cuda")
        S.tables = [np.ascontiguousarray(m, np.float64) for m in tables]
        dp = C.POINTER(C.c_double)
        S.lib = hip.load()
        S.args = [0, prec, n, nt, C.c_void_p(S.x.data_ptr()), C.c_void_p(S.t.data_ptr()),
                  *[m.ctypes.data_as(dp) for m in S.tables], 1.0, C.c_void_p(S.F.data_ptr()),
                  C.c_void_p(S.e.data_ptr()), C.c_void_p(S.ep.data_ptr()),
                  C.c_void_p(S.st.data_ptr())]
    elif S.kind == "re":
        off, x, t, S.v, T, S.lad = _re_inputs(case, seed)
        S.b = hip.Batch(0, prec)
        S.b.set_systems(off, x, t)
        S.b.set_smatb(*_flat(_smatb("agcu")))
        S.b.set_masses(MASS["agcu"])
        S.b.set_velocities(S.v)
        S.b.set_temperatures(T)
        S.round = 0
    elif S.kind == "fire":
        S.off, S.x = _fire_inputs(case, seed)
        S.b = hip.Batch(0, prec)
        S.b.set_smatb(*_flat(_smatb("au")))
        S.b.set_masses(MASS["au"])
    else:
        S.c, S.x, S.v = _context(case, seed)
        if S.kind == "md":
            S.c.integrator_vv(DT[case["system"]])
        elif S.kind == "langevin":
            S.c.integrator_ermak(DT[case["system"]], TEMP[case["system"]], 1.0,
                                 rng=hip.GH_RNG_PHILOX, seed=int(seed))
    return S


def _flat(p):
    return (p[0], *p[1])


def run(S):
    if S.kind == "static":
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        rc = S.lib.gh_cluster_forces_static(*S.args, stream)
        if rc:
            raise RuntimeError("gh_cluster_forces_static: %d" % rc)
        return {"F": S.F, "e": S.e, "epot": S.ep, "status": S.st}
    if S.kind == "forces":
        S.c.set_positions(S.x)
        F, e, et = S.c.compute()
        return {"F": F, "e": e, "etot": et}
    if S.kind == "re":
        ep, ek = S.b.langevin(S.case["steps"], 0.002, 1.0, 11 + S.round)
        acc = S.b.exchange(S.lad, S.round & 1, 1000 + S.round)
        S.round += 1
        x, v = S.b.state()
        return {"epot": ep, "ekin": ek, "accepted": acc, "ladders": S.lad.copy(), "x": x, "v": v}
    if S.kind == "fire":  # new starts every quench
        S.b.set_systems(S.off, S.x)
        r = S.b.fire(max_iter=S.case["steps"])
        r["x"] = S.b.state()[0]
        return r
    # a chunk of dinamica: GEMS's state in, steps and their rows, the state out
    S.c.set_positions(S.x)
    S.c.set_velocities(S.v)
    S.c.set_accelerations(None)
    rows = S.c.run(S.case["steps"], each=S.case["each"])
    x, v, F, e = S.c.state()
    return {"rows": rows, "x": x, "v": v, "F": F, "e": e}


# pairs within the cut per atom (both directions), per system
_PAIRS = {"au": 42.0, "agcu": 50.0, "lj": 55.0, "plj": 55.0}


def work(case):
    """Positions, types and velocities in and out once per step (an MD step
    reads and writes x and v and reads the type; a force call reads x and type
    and writes F and e); the pair terms' arithmetic."""
    k = case["kind"]
    if k in ("re", "fire"):
        if k == "re":
            lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
            mean = (case["nmax"] - case["nmin"]) / (hi - lo) if hi > lo else case["nmax"]
            n = case["geoms"] * case["rungs"] * mean
        else:
            n = case["nsys"] * 0.5 * (case["nmin"] + case["nmax"])
        return {"bytes": n * 100.0 * case["steps"], "flops": n * 35.0 * 2 * 40.0 * case["steps"]}
    n = case["n"] if "n" in case else 4 * case["nx"] * case["ny"] * case["nz"] - case["vac"]
    pairs = _PAIRS[case["system"]] * (0.75 if "n" in case else 1.0)
    flops = pairs * (80.0 if case["system"] in ("au", "agcu") else 30.0)
    if k in ("static", "forces"):
        return {"bytes": n * 60.0, "flops": n * flops}
    return {"bytes": n * 100.0 * case["steps"], "flops": n * flops * case["steps"]}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------
class _Pairs:
    """Neighbours of every atom within `reach` as a padded table (torch)."""

    def __init__(self, x, L, pbc, reach):
        n, dev = len(x), x.device
        self.x0 = x.clone()
        if L is None:  # free cluster: every other atom
            j = torch.arange(n, device=dev).repeat(n, 1)
            self.nbr = j[~torch.eye(n, dtype=torch.bool, device=dev)].reshape(n, n - 1)
            self.ok = torch.ones_like(self.nbr, dtype=torch.bool)
            return
        nc = [max(1, int(L[d] / reach)) for d in range(3)]
        c = []
        for d in range(3):
            k = torch.floor(x[:, d] / L[d] * nc[d]).long()
            c.append(torch.remainder(k, nc[d]) if pbc[d] else k.clamp(0, nc[d] - 1))
        cell = (c[2] * nc[1] + c[1]) * nc[0] + c[0]
        ncell = nc[0] * nc[1] * nc[2]
        order = torch.argsort(cell, stable=True)
        count = torch.bincount(cell, minlength=ncell)
        start = torch.cumsum(count, 0) - count
        most = int(count.max())
        table = torch.full((ncell, most), -1, dtype=torch.long, device=dev)
        sc = cell[order]
        table[sc, torch.arange(n, device=dev) - start[sc]] = order
        offs = []
        for d in range(3):  # cells of each axis, none twice
            offs.append(sorted({o % nc[d] for o in (-1, 0, 1)}) if pbc[d] else [-1, 0, 1])
        ii, jj = [], []
        lim = reach * reach
        chunk = max(1, 30_000_000 // most)
        for oz in offs[2]:
            for oy in offs[1]:
                for ox in offs[0]:
                    k = [c[0] + ox, c[1] + oy, c[2] + oz]
                    good = torch.ones(n, dtype=torch.bool, device=dev)
                    for d in range(3):
                        if pbc[d]:
                            k[d] = torch.remainder(k[d], nc[d])
                        else:
                            good &= (k[d] >= 0) & (k[d] < nc[d])
                            k[d] = k[d].clamp(0, nc[d] - 1)
                    other = (k[2] * nc[1] + k[1]) * nc[0] + k[0]
                    for a in range(0, n, chunk):
                        b = min(n, a + chunk)
                        j = table[other[a:b]]
                        mine = torch.arange(a, b, device=dev)[:, None]
                        keep = (j >= 0) & (j != mine) & good[a:b, None]
                        r2 = 0.0
                        for d in range(3):
                            u = x[:, d][j.clamp(min=0)] - x[a:b, d][:, None]
                            if pbc[d]:
                                u = u - L[d] * torch.round(u / L[d])
                            r2 = r2 + u * u
                        keep &= r2 < lim
                        w = keep.nonzero()
                        ii.append((w[:, 0] + a).int())
                        jj.append(j[keep].int())
        i, j = torch.cat(ii), torch.cat(jj)
        i, by = torch.sort(i, stable=True)
        i, j = i.long(), j[by].long()
        num = torch.bincount(i, minlength=n)
        first = torch.cumsum(num, 0) - num
        width = max(1, int(num.max()))
        self.nbr = torch.zeros((n, width), dtype=torch.long, device=dev)
        self.ok = torch.zeros((n, width), dtype=torch.bool, device=dev)
        slot = torch.arange(len(i), device=dev) - first[i]
        self.nbr[i, slot] = j
        self.ok[i, slot] = True


class _Exact:
    """Forces (ui/A) and per-atom energies (ui) of one system in 64 bits."""

    def __init__(self, system, L, pbc, t):
        self.s, self.L, self.pbc = system, L, pbc
        self.t = torch.as_tensor(t, dtype=torch.long, device="cuda")
        if system in ("au", "agcu"):
            self.nt, tabs = _smatb(system)
            A, xi, p, q, r0, rci, rce = (torch.as_tensor(m, device="cuda") for m in tabs)
            dc = rce - rci
            ab = -1.0 / dc ** 3

            def tail(amp, k):  # quintic matched to the exponential at rci
                bb, cb = -k / dc ** 2, -k * k / dc
                return (amp * (12 * ab - 6 * bb + cb) / (2 * dc ** 2),
                        amp * (15 * ab - 7 * bb + cb) / dc, amp * (20 * ab - 8 * bb + cb) / 2)

            self.P = [A, xi, p, q, r0, rci, rce, *tail(xi * torch.exp(-q * (rci / r0 - 1)), q / r0),
                      *tail(A * torch.exp(-p * (rci / r0 - 1)), p / r0)]
            self.rcut = float(rce.max())
        elif system == "lj":
            self.rcut = LJ_RC
        else:
            self.P = [torch.as_tensor(PLJ_EPS, device="cuda"),
                      torch.as_tensor(PLJ_SIG, device="cuda")]
            self.rcut = PLJ_RC
        self.margin, self.pairs = (1.2 if system in ("au", "agcu") else 0.45), None

    def _geometry(self, x, a, b):
        j, ok = self.pairs.nbr[a:b], self.pairs.ok[a:b]
        u, r2 = [], 0.0
        for d in range(3):
            w = x[:, d][j] - x[a:b, d][:, None]
            if self.L is not None and self.pbc[d]:
                w = w - self.L[d] * torch.round(w / self.L[d])
            u.append(w)
            r2 = r2 + w * w
        return j, u, torch.sqrt(torch.where(ok & (r2 <= self.rcut ** 2), r2, 1e6))

    def _par(self, k, a, b, j):
        if len(MASS[self.s]) == 1:
            return self.P[k].reshape(-1)[0]
        return self.P[k][self.t[a:b][:, None], self.t[j]]

    def __call__(self, x):
        if self.pairs is None or (self.L is not None and float(
                ((x - self.pairs.x0) ** 2).sum(1).max()) > (0.5 * self.margin) ** 2):
            self.pairs = _Pairs(x, self.L, self.pbc, self.rcut + self.margin)
        n = len(x)
        F, e = torch.empty_like(x), torch.empty(n, dtype=x.dtype, device=x.device)
        size = max(1, 40_000_000 // self.pairs.nbr.shape[1])
        parts = [(a, min(n, a + size)) for a in range(0, n, size)]
        if self.s in ("au", "agcu"):
            rho = torch.empty_like(e)
            for a, b in parts:
                j, u, r = self._geometry(x, a, b)
                g = lambda k: self._par(k, a, b, j)  # noqa: E731
                d = r - g(6)
                inner = g(1) ** 2 * torch.exp(-2 * g(3) * (r / g(4) - 1))
                outer = (d ** 3 * (g(9) + d * (g(8) + d * g(7)))) ** 2
                rho[a:b] = torch.where(r <= g(6), torch.where(r < g(5), inner, outer), 0.0).sum(1)
            eb = 1 / torch.sqrt(rho)
            for a, b in parts:
                j, u, r = self._geometry(x, a, b)
                g = lambda k: self._par(k, a, b, j)  # noqa: E731
                d, z = r - g(6), eb[a:b][:, None] + eb[j]
                rep = g(0) * torch.exp(-g(2) * (r / g(4) - 1))
                f = 2 * rep * g(2) / g(4) - \
                    g(1) ** 2 * g(3) / g(4) * torch.exp(-2 * g(3) * (r / g(4) - 1)) * z
                rt = d ** 3 * (g(12) + d * (g(11) + d * g(10)))
                ft = d ** 3 * (g(9) + d * (g(8) + d * g(7))) * \
                    d ** 2 * (3 * g(9) + d * (4 * g(8) + d * 5 * g(7))) * z - \
                    2 * d ** 2 * (3 * g(12) + d * (4 * g(11) + d * 5 * g(10)))
                near, cut = r <= g(5), r <= g(6)
                f = torch.where(cut, torch.where(near, f, ft), 0.0) / r
                e[a:b] = torch.where(cut, torch.where(near, rep, rt), 0.0).sum(1) - \
                    torch.sqrt(rho[a:b])
                for k in range(3):
                    F[a:b, k] = -(f * u[k]).sum(1)
        else:
            for a, b in parts:
                j, u, r = self._geometry(x, a, b)
                eps, sig = (1.0, 1.0) if self.s == "lj" else \
                    (self._par(0, a, b, j), self._par(1, a, b, j))
                s6 = (sig / r) ** 6
                p, f = 4 * eps * (s6 * s6 - s6), eps * (48 * s6 - 24) * s6 / r
                if self.s == "plj":  # value and slope terms at the cut, as plj_set forms them
                    c6 = (sig / PLJ_RC) ** 6
                    slope = 24 * eps * (2 * c6 * c6 - c6) / PLJ_RC
                    p, f = p - 4 * eps * (c6 * c6 - c6) - slope * (r - PLJ_RC), f + slope
                cut = r <= self.rcut
                e[a:b] = 0.5 * torch.where(cut, p, 0.0).sum(1)
                f = torch.where(cut, f, 0.0) / r
                for k in range(3):
                    F[a:b, k] = -(f * u[k]).sum(1)
        return F / UI_EV, e / UI_EV


def _energy_row(e, v, m):
    cm = (m[:, None] * v).sum(0) / m.sum()
    ek = 0.5 * (m[:, None] * (v - cm) ** 2).sum()
    return [float(e.sum()) * UI_EV, float(ek) * UI_EV, float(e.sum() + ek) * UI_EV]


def _exact_fire(case, seed):
    """FIRE (Bitzek et al. 2006) of every cluster at once, padded, in FP64."""
    off, x0 = _fire_inputs(case, seed)
    S, n = len(off) - 1, np.diff(off)
    most = int(n.max())
    x = torch.zeros((S, most, 3), dtype=torch.float64, device="cuda")
    live = torch.arange(most, device="cuda")[None, :] < torch.as_tensor(n, device="cuda")[:, None]
    x[live] = torch.as_tensor(x0, device="cuda")
    x[~live] = 1e4 * (1 + torch.arange(int((~live).sum()), device="cuda",
                                       dtype=torch.float64))[:, None]
    E = _Exact("au", None, (0, 0, 0), np.zeros(1))
    A, xi, p, q, r0, rci, rce, b1, b2, b3, r1, r2, r3 = (float(k) for k in E.P)
    diag = torch.eye(most, dtype=torch.bool, device="cuda")[None]

    def forces(x):
        F, e = torch.empty_like(x), torch.empty((S, most), dtype=x.dtype, device="cuda")
        step = max(1, 20_000_000 // (most * most))
        for a in range(0, S, step):
            y = x[a:a + step]
            u = y[:, None, :, :] - y[:, :, None, :]
            r = torch.sqrt(torch.where(diag, 1e6, (u * u).sum(-1)))
            cut, near, d = r <= rce, r <= rci, r - rce
            t = torch.where(r < rci, xi * xi * torch.exp(-2 * q * (r / r0 - 1)),
                            (d ** 3 * (b3 + d * (b2 + d * b1))) ** 2)
            rho = torch.where(cut, t, 0.0).sum(-1)
            eb = 1 / torch.sqrt(torch.where(rho > 0, rho, 1.0))
            z = eb[:, :, None] + eb[:, None, :]
            rep = A * torch.exp(-p * (r / r0 - 1))
            f = 2 * rep * p / r0 - xi * xi * q / r0 * torch.exp(-2 * q * (r / r0 - 1)) * z
            ft = d ** 3 * (b3 + d * (b2 + d * b1)) * d ** 2 * (3 * b3 + d * (4 * b2 + d * 5 * b1)) \
                * z - 2 * d ** 2 * (3 * r3 + d * (4 * r2 + d * 5 * r1))
            rt = d ** 3 * (r3 + d * (r2 + d * r1))
            f = torch.where(cut, torch.where(near, f, ft), 0.0) / r
            e[a:a + step] = torch.where(cut, torch.where(near, rep, rt), 0.0).sum(-1) - \
                torch.sqrt(rho)
            F[a:a + step] = -(f[..., None] * u).sum(2)
        return F / UI_EV, e / UI_EV

    dt_max, a0, om = 0.005, 0.1, 1.0 / M_AU
    dt = torch.full((S, 1, 1), 0.1 * dt_max, dtype=torch.float64, device="cuda")
    al = torch.full_like(dt, a0)
    good = torch.zeros_like(dt)
    F, e = forces(x)
    v = torch.zeros_like(x)
    fmax = None
    for _ in range(case["steps"]):
        fmax = torch.sqrt((F * F).sum(-1).max(1).values) * UI_EV
        v = v + 0.5 * dt * F * om
        x = x + torch.where(live[..., None], dt * v, 0.0)
        F, e = forces(x)
        v = v + 0.5 * dt * F * om
        P = (F * v).sum((1, 2), keepdim=True)
        vv, ff = (v * v).sum((1, 2), keepdim=True), (F * F).sum((1, 2), keepdim=True)
        up = P > 0
        v = torch.where(up, (1 - al) * v + al * torch.sqrt(vv / ff) * F, 0.0)
        good = torch.where(up, good + 1, 0.0)
        grow = up & (good > 5)
        dt = torch.where(up, torch.where(grow, (dt * 1.1).clamp(max=dt_max), dt), 0.5 * dt)
        al = torch.where(up, torch.where(grow, al * 0.99, al), a0)
    return {"iters": None, "converged": None,
            "epot": torch.where(live, e, 0.0).sum(1) * UI_EV, "fmax": fmax, "x": x[live]}


def exact(case, seed):
    """None for the dynamics on the device's random stream, whose FP32 draws
    have no 64-bit value."""
    if case["kind"] in ("langevin", "re"):
        return None
    if case["kind"] == "fire":
        return _exact_fire(case, seed)
    L, pbc, x, t, v = _inputs(case, seed)
    E = _Exact(case["system"], L, pbc, t)
    x, v = torch.as_tensor(x, device="cuda"), torch.as_tensor(v, device="cuda")
    F, e = E(x)
    if case["kind"] == "static":
        return {"F": F.reshape(-1), "e": e, "epot": e.sum().reshape(1), "status": None}
    if case["kind"] == "forces":
        return {"F": F, "e": e, "etot": float(e.sum())}
    m = torch.as_tensor(np.asarray(MASS[case["system"]])[t], device="cuda")
    dt, om, rows = DT[case["system"]], (1.0 / m)[:, None], []
    for k in range(1, case["steps"] + 1):
        x = x + dt * v + 0.5 * dt * dt * F * om
        v = v + 0.5 * dt * F * om
        F, e = E(x)
        v = v + 0.5 * dt * F * om
        if k % case["each"] == 0:
            rows.append(_energy_row(e, v, m))
    for d in range(3):  # reported inside the box
        if L is not None and pbc[d]:
            x[:, d] = torch.remainder(x[:, d], L[d])
    return {"rows": np.array(rows), "x": x, "v": v, "F": F, "e": e}
