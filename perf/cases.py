"""Performance cases of the many-body energy and gradient path, through its public entry points.

Each case is a dict of plain values; listed() gives the ones that are timed, draw() more of the same
ranges.  prepare() makes what a program holds before a step (coordinates, an engine with its topology,
box and cutoffs), run() is one step, work() what the step cannot do without, and exact() the step's
results from the monomial tables in plain 64-bit torch (pure-water systems and the differentiable n-mers).

Cutoffs are 9 A (2B) and 7 A (3B) throughout, as in the benchmark and the reference systems.
"""
import ctypes
import functools
import json
import math
import os
import tempfile

import numpy as np
import torch

import mbx_amd
from mbx_amd import autograd, engine

CUT2, CUT3, CUT4 = 9.0, 7.0, 6.0
DENSITY = 0.03343  # waters per cubic Angstrom at 1 g/cm^3
SPACING = 3.3      # lattice spacing of the CH4 / H2O boxes, Angstrom
IONS = ("f-", "cl-", "br-", "i-", "li+", "na+", "k+", "rb+", "cs+")


def listed():
    return [
        # a water hexamer in the gas phase: one step of a geometry optimisation driven from host arrays;
        # launches and latency are all there is
        dict(name="cluster_6", kind="cluster", waters=6, fourbody=False),
        # a small cluster with the 4B term, as in benchmark calculations of water clusters
        dict(name="cluster_40_4b", kind="cluster", waters=40, fourbody=True),
        # the classic 256-water periodic box: a Monte Carlo move (energies only) and an MD step
        dict(name="box_256_energy", kind="box", waters=256, grads=False),
        dict(name="box_256", kind="box", waters=256, grads=True),
        # the benchmark's box, an MD step with everything resident on the device
        dict(name="box_2048", kind="box", waters=2048, grads=True),
        # a large liquid simulation cell (19 x 19 x 19 lattice)
        dict(name="box_6859", kind="box", waters=6859, grads=True),
        # a program linked against the C entry points: 1B + 2B + 3B, host arrays in and out, an odd size
        dict(name="drop_in_617", kind="drop_in", waters=617),
        # many gas-phase clusters of different sizes in one context: nucleation, data-set generation
        dict(name="clusters_256x", kind="clusters", systems=256, smallest=12, largest=256),
        # path-integral MD of methane in water: the beads of one ring-polymer step as a batch
        dict(name="beads_32", kind="mixture", beads=32, ch4=57, h2o=513),
        # a methane-rich mixture, one classical MD step
        dict(name="mixture_570", kind="mixture", beads=1, ch4=342, h2o=228),
        # a solution: ions of nine kinds and dissolved CO2 in a water box
        dict(name="solution_256", kind="solution", waters=231, ions=17, co2=8),
        # one fitting step: energies and forces of dimers and trimers, loss, backward to the
        # coordinates, the linear and the nonlinear parameters
        dict(name="fit_4096", kind="fit", dimers=4096, trimers=4096, backward=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cluster", "cluster", "box", "box", "box", "drop_in", "clusters", "mixture", "mixture",
                       "solution", "fit", "fit"])
    if kind == "cluster":
        four = rng.random() < 0.4
        return dict(kind=kind, waters=_log(rng, 4 if four else 2, 48 if four else 400), fourbody=four)
    if kind == "box":
        return dict(kind=kind, waters=_log(rng, 250, 6800), grads=rng.random() < 0.75)
    if kind == "drop_in":
        return dict(kind=kind, waters=_log(rng, 250, 4000))
    if kind == "clusters":
        lo = _log(rng, 3, 24)
        return dict(kind=kind, systems=_log(rng, 8, 250), smallest=lo, largest=_log(rng, 2 * lo, 256))
    if kind == "mixture":
        n = rng.randrange(330, 700)
        ch4 = int(n * rng.uniform(0.05, 0.6))
        return dict(kind=kind, beads=_log(rng, 1, 24) if ch4 < 0.2 * n else rng.randrange(1, 4), ch4=ch4, h2o=n - ch4)
    if kind == "solution":
        return dict(kind=kind, waters=rng.randrange(230, 420), ions=rng.randrange(1, 25), co2=rng.randrange(0, 12))
    return dict(kind=kind, dimers=_log(rng, 50, 4096), trimers=_log(rng, 50, 4096), backward=rng.random() < 0.7)


# ---- inputs --------------------------------------------------------------------------------------


def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], axis=-1).reshape(n, 3, 3)


def _waters(rng, oxygens):
    """(n, 3, 3): O, H, H at the given oxygen positions, perturbed geometries, random orientations."""
    n = len(oxygens)
    half = np.radians(104.52 + rng.uniform(-3.0, 3.0, n)) / 2
    body = np.zeros((n, 3, 3))
    for h, sign in ((1, 1.0), (2, -1.0)):
        r = 0.9572 + rng.uniform(-0.02, 0.02, n)
        body[:, h, 0] = r * np.cos(half)
        body[:, h, 1] = sign * r * np.sin(half)
    return np.einsum("nij,naj->nai", _rotations(rng, n), body) + oxygens[:, None, :]


def _lattice(rng, n, edge, jitter=0.3):
    """n jittered sites of the smallest cubic lattice that holds them, in a cube of the given edge."""
    m = math.ceil(round(n ** (1 / 3), 9))
    i = np.sort(rng.permutation(m ** 3)[:n])
    site = np.stack([i % m, i // m % m, i // (m * m)], axis=1)
    return (site + 0.5) * (edge / m) + rng.uniform(-jitter, jitter, (n, 3))


def _droplet(rng, n):
    """n waters: the jittered lattice sites nearest to a random centre."""
    a = DENSITY ** (-1 / 3)
    m = math.ceil((3 * n / (4 * math.pi)) ** (1 / 3)) + 2
    site = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * a
    site = site + rng.uniform(-0.5, 0.5, 3) * a
    near = np.argsort((site ** 2).sum(1), kind="stable")[:n]
    return _waters(rng, site[near] + rng.uniform(-0.3, 0.3, (n, 3)))


def _edge(waters):
    return (waters / DENSITY) ** (1 / 3)


def _cube(edge):
    return np.diag([edge] * 3).reshape(-1)


def _methanes(rng, centers):
    tet = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]]) / math.sqrt(3.0) * 1.09
    h = np.einsum("nij,aj->nai", _rotations(rng, len(centers)), tet) + centers[:, None, :]
    return np.concatenate([centers[:, None, :], h], axis=1)


def _cluster_sizes(case):
    k = (np.arange(case["systems"]) + 0.5) / case["systems"]
    return np.round(case["smallest"] * (case["largest"] / case["smallest"]) ** k).astype(int)


def _mixture(rng, ch4, h2o):
    n = ch4 + h2o
    edge = SPACING * math.ceil(round(n ** (1 / 3), 9))
    sites = rng.permutation(_lattice(rng, n, edge, 0.2))
    return np.concatenate([_methanes(rng, sites[:ch4]).reshape(-1), _waters(rng, sites[ch4:]).reshape(-1)]), edge


def _solution(rng, case):
    """The ions (each kind in turn), then CO2, then waters on the sites of a water lattice."""
    n = case["ions"] + case["co2"] + case["waters"]
    edge = _edge(n)
    sites = rng.permutation(_lattice(rng, n, edge))
    ions, co2, water = np.split(sites, [case["ions"], case["ions"] + case["co2"]])
    axis = _rotations(rng, len(co2))[:, :, 0] * 1.16
    xyz = np.concatenate([ions.reshape(-1), np.stack([co2, co2 + axis, co2 - axis], axis=1).reshape(-1),
                          _waters(rng, water).reshape(-1)])
    kinds = ([engine.KIND_OF[IONS[i % len(IONS)]] for i in range(case["ions"])] + [engine.CO2] * case["co2"]
             + [engine.H2O] * case["waters"])
    return xyz, kinds, edge


def _nmers(rng, n, order):
    """n water dimers (O-O 2.4 .. 9 A) or trimers (each O-O 2.5 .. 7 A) in random orientations."""
    o = np.zeros((n, order, 3))
    if order == 2:
        o[:, 1] = _rotations(rng, n)[:, 0] * rng.uniform(2.4, 9.0, (n, 1))
    else:
        d = rng.uniform(2.5, 7.0, (8 * n + 64, 3))
        d = d[2 * d.max(1) < d.sum(1)][:n]
        cosa = (d[:, 0] ** 2 + d[:, 1] ** 2 - d[:, 2] ** 2) / (2 * d[:, 0] * d[:, 1])
        o[:, 1, 0] = d[:, 0]
        o[:, 2, 0], o[:, 2, 1] = d[:, 1] * cosa, d[:, 1] * np.sqrt(1 - cosa ** 2)
        o = np.einsum("nij,naj->nai", _rotations(rng, n), o)
    return _waters(rng, o.reshape(-1, 3)).reshape(n, 9 * order)


def _inputs(case, seed):
    """Coordinates (flat, Angstrom) and the box edge (None in the gas phase) of the engine's kinds."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "cluster":
        return _droplet(rng, case["waters"]).reshape(-1), None
    if kind in ("box", "drop_in"):
        edge = _edge(case["waters"])
        return _waters(rng, _lattice(rng, case["waters"], edge)).reshape(-1), edge
    if kind == "clusters":
        return np.concatenate([_droplet(rng, n).reshape(-1) for n in _cluster_sizes(case)]), None
    if kind == "mixture":
        xyz, edge = _mixture(rng, case["ch4"], case["h2o"])
        return (xyz + rng.normal(0.0, 0.05, (case["beads"], len(xyz)))).reshape(-1), edge
    raise ValueError(kind)


def _fit_inputs(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for order, n in ((2, case["dimers"]), (3, case["trimers"])):
        out.append((_nmers(rng, n, order), rng.normal(0.0, 1.0, n), rng.normal(0.0, 5.0, (n, 9 * order))))
    return out


# ---- the step --------------------------------------------------------------------------------------


class _DeviceArray:
    """A device buffer of an engine, for torch.as_tensor; keeps the engine."""

    def __init__(self, eng, ptr, n):
        self.engine = eng
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2)


def _engine(kinds, edge, offsets=None):
    e = engine.Engine()
    e.set_topology(kinds)
    e.set_box(None if edge is None else _cube(edge))
    e.set_cutoffs(CUT2, CUT3)
    if offsets is not None:
        e.set_batch(offsets)
    e.set_graph(True)
    return e


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fit":
        sets = []
        for family, (x, e, f) in zip(("mbpol_2b", "mbpol_3b"), _fit_inputs(case, seed)):
            coef, theta = autograd.defaults(family)
            x, e, f = (torch.from_numpy(v).cuda() for v in (x, e, f))
            sets.append((family, x.requires_grad_(case["backward"]), coef.requires_grad_(case["backward"]),
                         theta.requires_grad_(case["backward"]), e, f))
        return dict(kind=kind, sets=sets, backward=case["backward"])
    if kind == "solution":
        rng = np.random.default_rng(seed)
        xyz, kinds, edge = _solution(rng, case)
        return dict(kind=kind, engine=_engine(kinds, edge), xyz=xyz, terms=engine.TERM_2B | engine.TERM_3B)
    xyz, edge = _inputs(case, seed)
    if kind == "drop_in":
        return _drop_in(case["waters"], xyz, edge)
    if kind == "cluster":
        e = _engine([engine.H2O] * case["waters"], None)
        terms = engine.TERM_2B | engine.TERM_3B
        if case["fourbody"]:
            e.set_cutoff4b(CUT4)
            terms |= engine.TERM_4B
        return dict(kind=kind, engine=e, xyz=xyz, terms=terms)
    if kind == "box":
        e = _engine([engine.H2O] * case["waters"], edge)
    elif kind == "clusters":
        sizes = _cluster_sizes(case)
        e = _engine([engine.H2O] * int(sizes.sum()), None, np.concatenate([[0], np.cumsum(sizes)]))
    else:
        one = [engine.CH4] * case["ch4"] + [engine.H2O] * case["h2o"]
        b = case["beads"]
        e = _engine(one * b, edge, np.arange(b + 1) * len(one) if b > 1 else None)
    grad, totals = e.device_outputs()
    return dict(kind=kind, engine=e, xyz=torch.from_numpy(xyz).cuda(), grads=case.get("grads", True),
                gradient=torch.as_tensor(_DeviceArray(e, grad, len(xyz)), device="cuda"),
                totals=torch.as_tensor(_DeviceArray(e, totals, 21), device="cuda"))


def _drop_in(n, xyz, edge):
    """The C entry points' global system (one per process), set up as a reference caller does."""
    L = engine.lib()
    dp, ip, cpp = (ctypes.POINTER(t) for t in (ctypes.c_double, ctypes.c_int, ctypes.c_char_p))
    L.initialize_system_py_.argtypes = [dp, ip, cpp, cpp, ip, ctypes.c_char_p]
    L.get_energy_g_.argtypes = [dp, ip, dp, dp]
    with tempfile.TemporaryDirectory() as tmp:
        path = os.path.join(tmp, "mbx.json")
        with open(path, "w") as f:
            json.dump({"MBX": {"box": list(_cube(edge)), "twobody_cutoff": CUT2, "threebody_cutoff": CUT3}}, f)
        L.initialize_system_py_(xyz.ctypes.data_as(dp), (ctypes.c_int * n)(*[3] * n),
                                (ctypes.c_char_p * (3 * n))(*[b"O", b"H", b"H"] * n),
                                (ctypes.c_char_p * n)(*[b"h2o"] * n), ctypes.byref(ctypes.c_int(n)), path.encode())
    return dict(kind="drop_in", call=L.get_energy_g_, dp=dp, xyz=xyz, atoms=ctypes.c_int(3 * n))


def run(state):
    kind = state["kind"]
    if kind == "fit":
        out = []
        for family, x, coef, theta, e_ref, f_ref in state["sets"]:
            e, f = autograd.energy_forces(x, coef, theta, family)
            if state["backward"]:
                loss = autograd.energy_force_loss(e, f, e_ref, f_ref)
                out.append((e, f, loss) + torch.autograd.grad(loss, (x, coef, theta)))
            else:
                out.append((e, f))
        return out
    if kind == "drop_in":
        e, g = ctypes.c_double(), np.zeros(len(state["xyz"]))
        state["call"](state["xyz"].ctypes.data_as(state["dp"]), ctypes.byref(state["atoms"]), ctypes.byref(e),
                      g.ctypes.data_as(state["dp"]))
        return e.value, g
    eng = state["engine"]
    if kind in ("cluster", "solution"):
        eng.set_coords(state["xyz"])
        eng.compute(state["terms"])
        e2, e3, g, v = eng.results()
        return eng.term_energies() if state["terms"] & engine.TERM_4B else (e2, e3), g, v
    eng.set_coords_device(state["xyz"].data_ptr())
    eng.compute(do_grads=state["grads"])
    if eng.nconf > 1:
        return eng.batch_results(), state["gradient"]
    eng.synchronize()
    return (state["totals"], state["gradient"]) if state["grads"] else state["totals"][::7]


# ---- what a step cannot do without ---------------------------------------------------------------

# FP64 operations (fused multiply-adds as two) per n-mer for value and gradient when the polynomial is
# evaluated in coordinates adapted to the molecules' permutation symmetry, and evaluated n-mers per
# molecule in the bulk liquid at the holders' switching distances
_FLOPS = dict(dimer=15e3, trimer=36e3, ch4h2o=12e3, ch4ch4=82e3, ch4h2o2=26e3, tetramer=45e3)


def _bulk(n):
    """Evaluated (dimers, trimers) of n waters in one droplet: the bulk's 19 and 81 a water less the surface's share."""
    inner = max(0.0, 1.0 - 1.6 / max(n, 2) ** (1 / 3))
    return min(19 * n * (0.3 + 0.7 * inner), n * (n - 1) / 2), min(81 * n * inner, n * (n - 1) * (n - 2) / 6)


def work(case):
    kind = case["kind"]
    if kind == "fit":
        k = 4.0 if case["backward"] else 1.0
        n2, n3 = case["dimers"], case["trimers"]
        return dict(bytes=8.0 * (n2 * 18 + n3 * 27) * (4 if case["backward"] else 2) + 8.0 * 2 * 2336,
                    flops=k * (n2 * _FLOPS["dimer"] + n3 * _FLOPS["trimer"]))
    if kind == "mixture":
        c, w, b = case["ch4"], case["h2o"], case["beads"]
        d = 1.0 / SPACING ** 3
        x = c / (c + w)
        n9, n65, n6 = (4 / 3 * math.pi * r ** 3 * d for r in (9.0, 6.5, 6.0))
        flops = (c * (1 - x) * n9 * _FLOPS["ch4h2o"] + c * x * n9 / 2 * _FLOPS["ch4ch4"]
                 + w * (1 - x) * n65 / 2 * _FLOPS["dimer"] + w * 60 * (1 - x) ** 2 * _FLOPS["trimer"]
                 + c * 1.2 * (n6 * (1 - x)) ** 2 / 2 * _FLOPS["ch4h2o2"])
        return dict(bytes=48.0 * b * (5 * c + 3 * w), flops=b * flops)
    if kind == "solution":
        n = case["waters"]
        return dict(bytes=48.0 * (3 * n + case["ions"] + 3 * case["co2"]),
                    flops=n * (19 * _FLOPS["dimer"] + 81 * _FLOPS["trimer"]) + case["ions"] * 250 * 40e3)
    if kind == "clusters":
        sizes = _cluster_sizes(case)
        pairs = [_bulk(int(n)) for n in sizes]
        atoms = 3 * int(sizes.sum())
        n2, n3 = sum(p[0] for p in pairs), sum(p[1] for p in pairs)
    else:
        n = case["waters"]
        atoms = 3 * n
        n2, n3 = _bulk(n) if kind == "cluster" else (19 * n, 81 * n)
    share = 1.0 if case.get("grads", True) else 0.5
    flops = share * (n2 * _FLOPS["dimer"] + n3 * _FLOPS["trimer"])
    if case.get("fourbody"):
        flops += 8 * n3 * _FLOPS["tetramer"]
    return dict(bytes=(48.0 if share == 1.0 else 24.0) * atoms + 168, flops=flops)


# ---- the same in plain 64-bit torch -----------------------------------------------------------------

# Sites of a dimer: O H H, O H H, then each water's two out-of-plane sites; of a trimer: O H H three times.
# (rate, form, site, site); forms: 0 exp(k(1-r)), 1 exp(k(4-r))/r, 2 exp(k(4-r)).
_VARS2 = ([(0, 0, 1, 2), (0, 0, 4, 5)] + [(1, 0, o, o + h) for o in (0, 3) for h in (1, 2)]
          + [(2, 1, a, b) for a in (1, 2) for b in (4, 5)]
          + [(3, 1, 0, 4), (3, 1, 0, 5), (3, 1, 3, 1), (3, 1, 3, 2), (4, 1, 0, 3)]
          + [(5, 2, a, b) for a in (6, 7) for b in (4, 5)] + [(5, 2, a, b) for a in (8, 9) for b in (1, 2)]
          + [(6, 2, 0, 8), (6, 2, 0, 9), (6, 2, 3, 6), (6, 2, 3, 7)] + [(7, 2, a, b) for a in (6, 7) for b in (8, 9)])
# (set, site, site): exp(-k_set (r - d_set))
_VARS3 = ([(0, o + 1, o + 2) for o in (0, 3, 6)] + [(1, o, o + h) for o in (0, 3, 6) for h in (1, 2)]
          + [(2, a, b) for a in (1, 2) for b in (4, 5, 7, 8)] + [(2, a, b) for a in (4, 5) for b in (7, 8)]
          + [(3, o, h + i) for o in (0, 3, 6) for h in (0, 3, 6) if h != o for i in (1, 2)]
          + [(4, 0, 3), (4, 0, 6), (4, 3, 6)])
_THETA2 = (-6.480884773303821e-01, 1.674518993682975e+00, 1.148231864355956e+00, 1.205989761123099e+00,
           1.395357065790959e+00, 7.347036852042255e-01, 7.998249864422826e-01, 7.960663960630585e-01,
           -9.721486914088159e-02, 9.859272078406150e-02)
_THETA3 = (-2.254303257872797e+00, -2.564771901404151e-01, 4.247920544074333e-01, 8.128985941165371e-01,
           3.749457984616480e-02, 1.690594510379166e+00, -2.999999868517452e+00, 3.499031358429095e+00,
           4.854042963514281e+00, 4.816312044947604e-08)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


@functools.lru_cache(maxsize=None)
def _table(name):
    """(coefficients, each monomial's coefficient index, its four factors; factor nvars is 1)."""
    path = os.path.join(os.path.dirname(os.path.abspath(mbx_amd.__file__)), "tables", name + ".tbl")
    with open(path) as f:
        lines = [t for t in (ln.split("#")[0].split() for ln in f) if t]
    at = [t[0] for t in lines].index("coef") + 1
    nv, nc = int(lines[0][1]), int(lines[1][1])
    coef = torch.tensor([float(t[0]) for t in lines[at:at + nc]], dtype=torch.float64, device=_device())
    rows = lines[at + nc + 1:]
    k = torch.tensor([int(t[0]) for t in rows], device=_device())
    idx = torch.tensor([[int(v) for v in t[2:]] + [nv] * (4 - int(t[1])) for t in rows], device=_device())
    return coef, k, idx.T.contiguous()


def _variables(order, w, theta):
    """(nvars, n) variables of the n-mers w (n, 3 * order, 3)."""
    if order == 3:
        a, b = (torch.tensor(v, device=w.device) for v in zip(*[(p, q) for _, p, q in _VARS3]))
        s = torch.tensor([v[0] for v in _VARS3], device=w.device)
        r = (w[:, a] - w[:, b]).square().sum(-1).sqrt()
        return torch.exp(-theta[s] * (r - theta[5 + s])).T
    sites = [w]
    for o in (0, 3):
        p, q = w[:, o + 1] - w[:, o], w[:, o + 2] - w[:, o]
        mid, out = w[:, o] + 0.5 * theta[8] * (p + q), theta[9] * torch.linalg.cross(p, q)
        sites += [(mid + out)[:, None], (mid - out)[:, None]]
    w = torch.cat(sites, dim=1)
    k, form, a, b = (torch.tensor(v, device=w.device) for v in zip(*_VARS2))
    r = (w[:, a] - w[:, b]).square().sum(-1).sqrt()
    e = torch.exp(theta[k] * (torch.where(form == 0, 1.0, 4.0).to(r.dtype) - r))
    return torch.where(form == 1, e / r, e).T


def _switch(order, w):
    def f(r, inner, outer):
        s = 0.5 * (1 + torch.cos((r - inner) * (math.pi / (outer - inner))))
        return torch.where(r <= inner, torch.ones_like(r), torch.where(r > outer, torch.zeros_like(r), s))

    def dist(i, j):
        return (w[:, i] - w[:, j]).square().sum(-1).sqrt()

    if order == 2:
        return f(dist(0, 3), 4.5, 6.5)
    ab, ac, bc = (f(dist(i, j), 0.0, 4.5) for i, j in ((0, 3), (0, 6), (3, 6)))
    return ab * ac + ab * bc + ac * bc


def _polynomial(name, x):
    """Value and gradient (the variables are positive, so x_j dP/dx_j counts x_j's factors)."""
    coef, k, idx = _table(name)
    nv = len(x)
    weight = torch.zeros(nv + 1, idx.shape[1], dtype=x.dtype, device=x.device)
    for row in idx:
        weight.scatter_add_(0, row[None], coef[k][None])
    weight[nv] = coef[k]
    value, grad = [], []
    for c in x.split(2048, dim=1):
        one = torch.cat([c, torch.ones_like(c[:1])])
        s = weight @ (one[idx[0]] * one[idx[1]] * one[idx[2]] * one[idx[3]])
        value.append(s[nv])
        grad.append(s[:nv] / c)
    return torch.cat(value), torch.cat(grad, dim=1)


def _lists(o, edge):
    """Dimers within 6.5 A and trimers with two of the three pairs within 4.5 A (the others have a zero switch)."""
    def close(cut):
        out = []
        for i in range(0, len(o), 1024):
            d = o[i:i + 1024, None] - o[None]
            if edge is not None:
                d -= edge * np.floor(d / edge + 0.5)
            p, q = np.nonzero((d * d).sum(-1) <= cut * cut)
            out.append(np.stack([p + i, q], axis=1))
        out = np.concatenate(out)
        return out[out[:, 0] != out[:, 1]]

    d = close(6.5)
    near = close(4.5)
    count = np.bincount(near[:, 0], minlength=len(o)) if len(near) else np.zeros(len(o), int)
    width = int(count.max()) if len(o) else 0
    nb = np.full((len(o), max(width, 1)), -1)
    nb[near[:, 0], np.concatenate([np.arange(c) for c in count]) if len(near) else []] = near[:, 1]
    u, v = np.triu_indices(nb.shape[1], 1)
    t = np.stack([np.repeat(np.arange(len(o)), len(u)), nb[:, u].reshape(-1), nb[:, v].reshape(-1)], axis=1)
    t = np.unique(np.sort(t[(t >= 0).all(1)], axis=1), axis=0)
    return d[d[:, 0] < d[:, 1]], t


def _water_system(xyz, edge):
    """{order: (energy, virial xx xy xz yy yz zz)} and the gradient of one water system."""
    w = torch.from_numpy(xyz.reshape(-1, 3, 3)).to(_device())
    grad = torch.zeros_like(w)
    terms = {}
    for order, nmers in zip((2, 3), _lists(xyz.reshape(-1, 3, 3)[:, 0], edge)):
        energy, virial = 0.0, torch.zeros(3, 3, dtype=w.dtype, device=w.device)
        theta = torch.tensor(_THETA2 if order == 2 else _THETA3, dtype=w.dtype, device=w.device)
        for part in torch.from_numpy(nmers).to(w.device).split(65536):
            if not len(part):
                continue
            m = w[part]  # (n, order, 3 atoms, 3)
            if edge is not None:
                m = m - edge * torch.floor((m[:, :, :1] - m[:, :1, :1]) / edge + 0.5)
            a = m.reshape(len(part), 3 * order, 3).clone().requires_grad_()
            x, s = _variables(order, a, theta), _switch(order, a)
            p, g = _polynomial("mbpol_%db" % order, x.detach())
            (f,) = torch.autograd.grad((s.detach() * (g * x).sum(0) + s * p).sum(), a)
            energy += float((s * p).sum().detach())
            virial -= torch.einsum("nai,naj->ij", a.detach(), f)
            grad.index_add_(0, part.reshape(-1), f.reshape(-1, 3, 3))
        v = virial.cpu().numpy()
        terms[order] = (energy, np.array([v[0, 0], v[0, 1], v[0, 2], v[1, 1], v[1, 2], v[2, 2]]))
    return terms, grad.cpu().numpy().reshape(-1)


def _mirror(v):
    return v[..., [0, 1, 2, 1, 3, 4, 2, 4, 5]]


def _exact_fit(case, seed):
    out = []
    for order, (x, e_ref, f_ref) in zip((2, 3), _fit_inputs(case, seed)):
        coef, k, idx = _table("mbpol_%db" % order)
        coef = coef.clone().requires_grad_()
        theta = torch.tensor(_THETA2 if order == 2 else _THETA3, dtype=torch.float64, device=_device()).requires_grad_()
        parts, n = [], len(x)
        for lo in range(0, n, 512):
            w, er, fr = (torch.from_numpy(v[lo:lo + 512]).to(_device()) for v in (x, e_ref, f_ref))
            w.requires_grad_()
            m = w.reshape(-1, 3 * order, 3)
            one = _variables(order, m, theta)
            one = torch.cat([one, torch.ones_like(one[:1])])
            basis = one[idx[0]] * one[idx[1]] * one[idx[2]] * one[idx[3]]
            e = _switch(order, m) * (coef[k] @ basis)
            (g,) = torch.autograd.grad(e.sum(), w, create_graph=case["backward"])
            row = [e.detach(), -g.detach()]
            if case["backward"]:
                loss = (e - er).square().sum() / n + (-g - fr).square().sum() / (n * 9 * order)
                row += [loss.detach()] + list(torch.autograd.grad(loss, (w, coef, theta)))
            parts.append(row)
        cat = [torch.cat([p[i] for p in parts]) for i in (0, 1)]
        if case["backward"]:
            cat += [sum(p[2] for p in parts), torch.cat([p[3] for p in parts]), sum(p[4] for p in parts),
                    sum(p[5] for p in parts)]
        out.append(tuple(cat))
    return out


def exact(case, seed):
    """run()'s results from the tables alone; None where the system holds other families than water's 2B and 3B."""
    kind = case["kind"]
    if kind == "fit":
        return _exact_fit(case, seed)
    if kind in ("drop_in", "mixture", "solution") or case.get("fourbody"):
        return None
    xyz, edge = _inputs(case, seed)
    if kind == "clusters":
        e2, e3, v, g, at = [], [], [], [], 0
        for n in _cluster_sizes(case):
            t, gr = _water_system(xyz[at:at + 9 * n], None)
            at += 9 * n
            e2.append(t[2][0])
            e3.append(t[3][0])
            v.append(_mirror(t[2][1] + t[3][1]))
            g.append(gr)
        return (np.array(e2), np.array(e3), np.array(v)), np.concatenate(g)
    t, g = _water_system(xyz, edge)
    if kind == "cluster":
        return (t[2][0], t[3][0]), g, _mirror(t[2][1] + t[3][1])
    if not case["grads"]:
        return np.array([t[2][0], t[3][0], 0.0])
    return np.concatenate([[t[2][0]], t[2][1], [t[3][0]], t[3][1], np.zeros(7)]), g
