"""Performance cases: the work users of this library have it do, through its
public Python entry points (``libecp_amd.native``).

Molecules come from the library's own seeded workload recipes
(``libecp_amd.workloads``); another seed is another geometry, basis and ECP
of the same sizes.

Kinds of call
  matrix     ``get_integrals``: host arrays in, the ECP matrix out
  gradient   a handle of order 1 for a new geometry, contracted with a density
  energy     a resident batch evaluated and contracted with densities in HBM
  matrices   a batch of new molecules: creation, evaluation, every matrix
  serving    a burst of requests to a resident server, every matrix

Recipes
  small      4 atoms, one ECP centre, s..d basis
  molecule   20 % ECP atoms, s..f basis (atom count given)
  cluster    50 atoms, 10 ECP centres, s..f basis
  high_l     s..g basis on every atom, 40 % ECP atoms with L = 5
"""
from __future__ import annotations

import math

import numpy as np
import torch

from libecp_amd import native, workloads


def listed():
    return [
        # one call on a tiny molecule: launch and call latency
        {"name": "small_matrix", "kind": "matrix", "recipe": "small", "atoms": 4},
        # an ordinary molecule of an odd size, one call per geometry
        {"name": "molecule_matrix", "kind": "matrix", "recipe": "molecule", "atoms": 17},
        # the 50-atom cluster, one call per geometry (drop-in use)
        {"name": "cluster_matrix", "kind": "matrix", "recipe": "cluster", "atoms": 50},
        # the largest molecule of the request stream
        {"name": "large_matrix", "kind": "matrix", "recipe": "molecule", "atoms": 120},
        # high angular momenta, wide exponents, contractions of four
        {"name": "high_l_matrix", "kind": "matrix", "recipe": "high_l", "atoms": 20},
        # a step of a geometry optimisation: the forces of one density
        {"name": "cluster_gradient", "kind": "gradient", "recipe": "cluster", "atoms": 50},
        # the same for a tiny molecule
        {"name": "small_gradient", "kind": "gradient", "recipe": "small", "atoms": 4},
        # resident evaluation, the steady-state throughput of one cluster
        {"name": "cluster_energy", "kind": "energy", "recipe": "cluster", "atoms": 50, "molecules": 1},
        # the same with g shells
        {"name": "high_l_energy", "kind": "energy", "recipe": "high_l", "atoms": 20, "molecules": 1},
        # many uneven molecules in one resident job (3 to 40 atoms)
        {"name": "batch_energy", "kind": "energy", "recipe": "molecule", "atoms": 40, "molecules": 256},
        # a data set of new molecules, matrices to the host
        {"name": "batch_matrices", "kind": "matrices", "recipe": "molecule", "atoms": 40, "molecules": 48},
        # a burst of requests of 5 to 120 atoms
        {"name": "serving_burst", "kind": "serving", "recipe": "molecule", "atoms": 120, "molecules": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matrix", "matrix", "gradient", "energy", "energy", "matrices", "serving"])
    if kind == "matrix":
        recipe = rng.choice(["molecule", "molecule", "cluster", "high_l"])
        atoms = {"molecule": lambda: _log_int(rng, 3, 120), "cluster": lambda: rng.randint(11, 60),
                 "high_l": lambda: rng.randint(4, 20)}[recipe]()
        return {"kind": kind, "recipe": recipe, "atoms": atoms}
    if kind == "gradient":
        recipe = rng.choice(["molecule", "cluster"])
        return {"kind": kind, "recipe": recipe, "atoms": rng.randint(11, 50) if recipe == "cluster" else
                _log_int(rng, 3, 60)}
    if kind == "energy":
        recipe = rng.choice(["cluster", "high_l", "molecule"])
        if recipe == "molecule":
            return {"kind": kind, "recipe": recipe, "atoms": rng.randint(12, 40), "molecules": _log_int(rng, 2, 256)}
        return {"kind": kind, "recipe": recipe, "molecules": 1,
                "atoms": rng.randint(11, 60) if recipe == "cluster" else rng.randint(4, 20)}
    if kind == "matrices":
        return {"kind": kind, "recipe": "molecule", "atoms": rng.randint(8, 40), "molecules": _log_int(rng, 2, 48)}
    return {"kind": kind, "recipe": "molecule", "atoms": rng.randint(20, 120), "molecules": _log_int(rng, 4, 64)}


# ---------------------------------------------------------------------------
# inputs

def _molecules(case, seed):
    recipe, atoms = case["recipe"], case["atoms"]
    rng = np.random.default_rng(seed)
    if recipe == "small":
        return [workloads.plain_small(seed)]
    if recipe == "cluster":
        if atoms == 50:
            return [workloads.medium_cluster(seed)]
        return [workloads.medium_cluster(seed, nat=atoms, n_ecp=max(1, atoms // 5),
                                         box=30.0 * (atoms / 50.0) ** (1.0 / 3.0))]
    if recipe == "high_l":
        if atoms == 20:
            return [workloads.high_l(seed)]
        return [workloads.high_l(seed, nat=atoms, n_ecp=max(1, (2 * atoms) // 5),
                                 box=15.0 * (atoms / 20.0) ** (1.0 / 3.0))]
    if "molecules" not in case:
        return [workloads.batch_molecule(rng, atoms)]
    # uneven sizes: uniform from 3 atoms (5 in a request stream) to the
    # largest, the same for every seed
    low = 5 if case["kind"] == "serving" else 3
    sizes = np.random.default_rng(case["molecules"]).integers(low, atoms + 1, size=case["molecules"])
    return [workloads.batch_molecule(rng, int(n)) for n in sizes]


def _density(rng, nao):
    """A closed-shell density 2 C C^T of nao / 4 random orbitals."""
    C = rng.normal(size=(nao, max(1, nao // 4))) / math.sqrt(nao)
    return 2.0 * (C @ C.T)


def prepare(case, seed):
    kind = case["kind"]
    mols = _molecules(case, seed)
    state = {"kind": kind, "mols": mols}
    if kind == "gradient":
        state["density"] = _density(np.random.default_rng(seed + 1), mols[0].nao)
    elif kind == "energy":
        rng = np.random.default_rng(seed + 1)
        P = np.concatenate([_density(rng, m.nao).ravel() for m in mols])
        state["batch"] = native.Batch(mols)
        state["density"] = torch.from_numpy(P).cuda()
        state["energies"] = torch.zeros(len(mols), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        # resident use: the first evaluation, the graph of the following ones,
        # and the kernel times a program logs once (which also clears the HIP
        # error that capturing the graph can leave on the thread)
        state["batch"].execute(2)
        state["batch"].profile()
    elif kind == "serving":
        state["server"] = native.Server(slots=4, hbm_budget=8 << 30)
    return state


def run(state):
    kind, mols = state["kind"], state["mols"]
    if kind == "matrix":
        rc, V = native.get_integrals(mols[0])
        return {"rc": rc, "matrix": V}
    if kind == "gradient":
        h = native.Handle(mols[0], n=1)
        rc, g = h.contract(state["density"])
        h.close()
        return {"rc": rc, "gradient": g}
    if kind == "energy":
        b = state["batch"]
        b.execute(1)
        codes, _ = b.contract_device(state["density"].data_ptr(), state["energies"].data_ptr())
        return {"codes": codes, "energies": state["energies"]}
    if kind == "matrices":
        b = native.Batch(mols)
        b.execute(1)
        b.fetch()
        out = [b.matrix(i) for i in range(len(mols))]
        b.close()
        return _packed(out)
    s = state["server"]
    tickets = {s.submit(m): i for i, m in enumerate(mols)}
    out = [None] * len(mols)
    for _ in mols:
        t = s.next()
        out[tickets[t]] = s.result(t)[:2]
    return _packed(out)


def _packed(results):
    """Every molecule's return code and its matrix, one after the other."""
    return {"codes": np.asarray([rc for rc, _ in results]), "matrices": np.concatenate([V.ravel() for _, V in results])}


# ---------------------------------------------------------------------------
# what a pass cannot do without

POINTS = 11  # radial points of an integral that converges at the fifth level


def _pair_work(m):
    """(FLOPs per surviving triplet summed, triplets): every surviving
    (centre, shell, shell) needs, per primitive pair, the type-1 integrand
    (exponential, Bessel functions, n_Q products) on POINTS points, and its
    assembly; the type-2 radial entries on POINTS points each."""
    h = native.Handle(m)
    keys = h.screened_triplets()
    h.close()
    if len(keys) == 0:
        return 0.0, 0
    first = np.concatenate([[0], np.cumsum(m.shellsBS)[:-1]])
    sa, sb = first[keys[:, 1]] + keys[:, 2], first[keys[:, 3]] + keys[:, 4]
    la, lb = m.lBS[sa].astype(np.float64), m.lBS[sb].astype(np.float64)
    pairs = m.KBS[sa].astype(np.float64) * m.KBS[sb]
    lab = la + lb
    nq = np.floor((lab + 2) ** 2 / 4.0)
    top = np.asarray([0 if n == 0 else n - 1 for n in m.shellsECP])
    L = top[keys[:, 0]].astype(np.float64)
    dim = (la + 1) * (la + 2) * (la + 3) / 6 * (lb + 1) * (lb + 2) * (lb + 3) / 6
    t1 = pairs * (POINTS * (31 * lab + 74 + 4 * nq) + 36 * (lab + 1) ** 2)
    t2 = L * dim * (4 * POINTS + 8)
    return float((t1 + t2).sum()), len(keys)


def work(case):
    mols = _molecules(case, 0)
    flops = 0.0
    bytes_in = bytes_out = 0
    for m in mols:
        f, _ = _pair_work(m)
        # a first derivative has a raised and a lowered block of either side
        flops += f * (4.0 if case["kind"] == "gradient" else 1.0)
        bytes_in += 8 * (m.geometry.size + 2 * m.aBS.size + 3 * m.aECP.size) + 8 * (m.lBS.size + m.lECP.size)
        if case["kind"] in ("gradient", "energy"):
            bytes_in += 8 * m.nao * m.nao
            bytes_out += 24 * m.nat
        else:
            bytes_out += 8 * m.nao * m.nao
    return {"bytes": bytes_in + bytes_out, "flops": flops}


# ---------------------------------------------------------------------------
# exact values: product quadrature about every ECP centre in 64 bits

def _components(l):
    return [(l - i, i - j, j) for i in range(l + 1) for j in range(i + 1)]


def _harmonics(lmax, ct, ph):
    """Orthonormal real spherical harmonics, [(lmax + 1)^2, points]."""
    st = torch.sqrt(torch.clamp(1.0 - ct * ct, min=0.0))
    P = {(0, 0): torch.ones_like(ct)}
    for l in range(1, lmax + 1):
        P[l, l] = (2 * l - 1) * st * P[l - 1, l - 1]
        P[l, l - 1] = (2 * l - 1) * ct * P[l - 1, l - 1]
        for m in range(l - 1):
            P[l, m] = ((2 * l - 1) * ct * P[l - 1, m] - (l + m - 1) * P[l - 2, m]) / (l - m)
    rows = []
    for l in range(lmax + 1):
        for m in range(-l, l + 1):
            a = abs(m)
            n = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - a) / math.factorial(l + a))
            f = n * P[l, a]
            if m:
                f = math.sqrt(2.0) * f * (torch.cos(a * ph) if m > 0 else torch.sin(a * ph))
            rows.append(f)
    return torch.stack(rows)


class _Basis:
    """Values of every AO."""

    def __init__(self, m, dev):
        atom, shell_atom, ao_shell, ao_e, prim_shell = [], [], [], [], []
        s = p = 0
        for A in range(m.nat):
            for _ in range(int(m.shellsBS[A])):
                shell_atom.append(A)
                prim_shell += [s] * int(m.KBS[s])
                for e in _components(int(m.lBS[s])):
                    ao_shell.append(s)
                    ao_e.append(e)
                    atom.append(A)
                s += 1
        t = lambda x: torch.as_tensor(np.asarray(x), device=dev)
        self.atom, self.ao_shell, self.e = t(atom), t(ao_shell), t(ao_e)
        self.a, self.d = t(m.aBS), t(m.dBS)
        self.prim_atom = t(np.asarray(shell_atom)[prim_shell])
        S = np.zeros((s, len(prim_shell)))
        S[prim_shell, np.arange(len(prim_shell))] = 1.0
        self.S = t(S)
        self.R = t(m.geometry.reshape(-1, 3))
        self.lmax = int(m.lBS.max())

    def __call__(self, pts):
        x = pts.T[None, :, :] - self.R[:, :, None]          # [atoms, 3, points]
        g = self.d[:, None] * torch.exp(-self.a[:, None] * (x * x).sum(1)[self.prim_atom])
        rad = (self.S @ g)[self.ao_shell]
        pw = [torch.ones_like(x)]
        for _ in range(self.lmax):
            pw.append(pw[-1] * x)
        pw = torch.stack(pw)                                # [power, atoms, 3, points]
        e = self.e
        return rad * pw[e[:, 0], self.atom, 0] * pw[e[:, 1], self.atom, 1] * pw[e[:, 2], self.atom, 2]


def _exact_molecule(m):
    """The full symmetric ECP matrix."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    B = _Basis(m, dev)
    nao = m.nao
    V = torch.zeros((nao, nao), dtype=torch.float64, device=dev)
    amax = float(m.aBS.max())
    xg, wg = np.polynomial.legendre.leggauss(16)
    s = p = 0
    for A in range(m.nat):
        n = int(m.shellsECP[A])
        if n == 0:
            continue
        chan = []
        for _ in range(n):
            k = int(m.KECP[s])
            chan.append((int(m.lECP[s]), m.nECP[p:p + k], m.dECP[p:p + k], m.aECP[p:p + k]))
            s += 1
            p += k
        L = max(c[0] for c in chan)
        amin = min(float(c[3].min()) for c in chan)
        panels = max(8, int(math.ceil(math.sqrt(42.0 / amin) / 0.25)))
        h = math.sqrt(42.0 / amin) / panels
        rr = (np.arange(panels)[:, None] * h + 0.5 * h * (xg + 1.0)).ravel()
        ww = np.tile(0.5 * h * wg, panels)
        for r, w in zip(rr, ww):
            u = {}
            for l, nn, dd, aa in chan:
                u[l] = u.get(l, 0.0) + w * float((dd * r ** nn * np.exp(-aa * r * r)).sum())
            # an angular function exp(z cos) needs Legendre degrees up to
            # about sqrt(2 z ln(1 / eps)); z = 4 amax r^2 at most
            deg = r * math.sqrt(8.0 * amax * max(2.0, 36.0 - amin * r * r))
            N = int(deg / 2) + L + B.lmax + 8
            c, wc = np.polynomial.legendre.leggauss(N) if N <= 24 else _leggauss(N)
            ct = torch.as_tensor(c, device=dev).repeat_interleave(2 * N)
            ph = (torch.arange(2 * N, device=dev, dtype=torch.float64) * (math.pi / N)).repeat(N)
            wo = torch.as_tensor(wc, device=dev).repeat_interleave(2 * N) * (math.pi / N)
            st = torch.sqrt(1.0 - ct * ct)
            pts = B.R[A] + r * torch.stack([st * torch.cos(ph), st * torch.sin(ph), ct], dim=1)
            Y = _harmonics(max(L - 1, 0), ct, ph)
            for j in range(0, pts.shape[0], 1 << 17):
                q = slice(j, j + (1 << 17))
                part = B(pts[q])
                S = (part * wo[q]) @ Y[:, q].T if j == 0 else S + (part * wo[q]) @ Y[:, q].T
                V += u.get(L, 0.0) * ((part * wo[q]) @ part.T)
            ul = torch.as_tensor([u.get(l, 0.0) for l in range(L) for _ in range(2 * l + 1)], dtype=torch.float64,
                                 device=dev)
            if L > 0:
                S = S[:, :L * L]
                V += (S * ul) @ S.T
    return V.cpu().numpy()


_rules = {}


def _leggauss(n):
    """Gauss-Legendre nodes and weights by Newton's iteration, kept by order."""
    if n not in _rules:
        x = np.cos(math.pi * (np.arange(1, n + 1) - 0.25) / (n + 0.5))
        for _ in range(8):
            p0, p1 = np.ones_like(x), x
            for k in range(2, n + 1):
                p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
            dp = n * (x * p1 - p0) / (x * x - 1.0)
            x = x - p1 / dp
        _rules[n] = (x, 2.0 / ((1.0 - x * x) * dp * dp))
    return _rules[n]


def exact(case, seed):
    """The exact integrals, for the recipe whose integrals the library's
    adaptive quadratures resolve.  In the others (and in derivatives) some
    integrals of tight primitives far from the centre are what the
    quadrature's rules give at its tolerance, and not the exact value
    (differences up to 0.4): they have no value but the algorithm's own."""
    if case["recipe"] != "small" or case["kind"] != "matrix":
        return None
    return {"rc": None, "matrix": np.triu(_exact_molecule(_molecules(case, seed)[0]))}
