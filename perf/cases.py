"""Workloads of the engine, as a user's program calls them: single H.v products, ground states, T = 0 and
finite-temperature Green's functions, real-time propagation, batched impurity solves and bath-fit gradients.

A case is a dict of plain values; ``kind`` names the call and the rest are its sizes.  Impurity baths, interactions and
start vectors are drawn from the seed; impurities sit at ``eps_imp = -U/2`` (``mu = 0``), lattices at ``mu = U/2``.
"""

import math

import numpy as np
import torch

import cmpy_amd as ed
from cmpy_amd.batch import AndersonBatch, anderson_gf, matsubara, random_batch


def listed():
    return [
        # one H.v on the 4x4 periodic Hubbard sector (8,8), rows padded to whole 128-byte lines: the largest vectors
        # (1.3 GB), what a caller's own eigensolver or propagator spends its time on
        dict(name="hv_square16", kind="hv", lattice="square", sites=16, n_up=8, n_dn=8, nvec=1, padded=True),
        # the same product for an impurity with 13 bath levels, every hybridisation different (no uniform hopping),
        # on contiguous vectors
        dict(name="hv_siam14", kind="hv", lattice="siam", sites=14, n_up=7, n_dn=7, nvec=1, padded=False),
        # a 13-site chain away from half filling: odd row lengths, vectors that fit the last-level cache
        dict(name="hv_chain13", kind="hv", lattice="chain", sites=13, n_up=6, n_dn=5, nvec=1, padded=False),
        # the smallest whole call: a new 1+5-site impurity model, its ground state and G(i w_n), as a parameter sweep
        # or a fit makes it for every point
        dict(name="solve_siam6", kind="solve", lattice="siam", sites=6, n_up=3, n_dn=3, nsteps=200, nw=128, beta=50.0,
             fresh=True),
        # an ordinary impurity solve, 1+7 sites (4,900 states), the model and its operators kept
        dict(name="solve_siam8", kind="solve", lattice="siam", sites=8, n_up=4, n_dn=4, nsteps=200, nw=512, beta=100.0,
             fresh=False),
        # ground state and 200-step fractions of the 12-site chain (853,776 states)
        dict(name="solve_chain12", kind="solve", lattice="chain", sites=12, n_up=6, n_dn=6, nsteps=200, nw=1024,
             beta=50.0, fresh=False),
        # the ground-state vector of a 1+9-site impurity (63,504 states), fully reorthogonalised by default
        dict(name="ground_siam10", kind="ground", lattice="siam", sites=10, n_up=5, n_dn=5),
        # grand-canonical finite-temperature G and occupations of a 1+6-site impurity: 64 dense sectors up to 1,225
        dict(name="spectrum_siam7", kind="spectrum", sites=7, nz=1000, beta=20.0),
        # greater and lesser real-time G of the 10-site chain on 1000 times, and its transform to 1000 frequencies
        dict(name="realtime_chain10", kind="realtime", lattice="chain", sites=10, n_up=5, n_dn=5, nt=1000, tmax=20.0,
             nz=1000),
        # one iteration's impurity solves of an 8-point DMFT sweep: new baths, ground states, G(i w_n)
        dict(name="batch_dmft", kind="batch", models=8, nb_min=5, nb_max=5, nw=128, beta=50.0),
        # a batch of uneven impurities (400 to 63,504 states), G on 256 frequencies
        dict(name="batch_mixed", kind="batch", models=48, nb_min=5, nb_max=9, nw=256, beta=50.0),
        # loss and gradient of a bath fit, 64 impurities of 1+7 sites
        dict(name="bathfit_64", kind="fit", models=64, nb=7, nw=512, beta=100.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "solve", "solve", "ground", "spectrum", "realtime", "batch", "fit"])
    if kind == "hv":
        lattice = rng.choice(["chain", "siam", "square"])
        sites = rng.choice([8, 9, 12, 15, 16]) if lattice == "square" else rng.randint(6, 16)
        n_up = sites // 2 + rng.choice([-2, -1, 0, 1])
        n_dn = sites // 2 + rng.choice([-3, -2, -1, 0, 1])
        return dict(kind="hv", lattice=lattice, sites=sites, n_up=n_up, n_dn=n_dn,
                    nvec=rng.choice([1, 1, 1, 2, 4]) if sites < 13 else 1, padded=rng.random() < 0.5)
    if kind in ("solve", "ground"):
        lattice = rng.choice(["chain", "siam"])
        sites = rng.randint(5, 12 if lattice == "chain" else 11)
        n_up = (sites + 1) // 2 - rng.choice([0, 0, 1])
        n_dn = sites // 2
        c = dict(kind=kind, lattice=lattice, sites=sites, n_up=n_up, n_dn=n_dn)
        if kind == "solve":
            c.update(nsteps=rng.randint(100, 200), nw=_log_int(rng, 33, 1024), beta=round(rng.uniform(20.0, 100.0), 2),
                     fresh=rng.random() < 0.3)
        return c
    if kind == "spectrum":
        return dict(kind=kind, sites=rng.randint(3, 7), nz=_log_int(rng, 50, 1000),
                    beta=round(math.exp(rng.uniform(math.log(2.0), math.log(50.0))), 3))
    if kind == "realtime":
        lattice = rng.choice(["chain", "siam"])
        sites = rng.randint(5, 10)
        return dict(kind=kind, lattice=lattice, sites=sites, n_up=(sites + 1) // 2, n_dn=sites // 2,
                    nt=_log_int(rng, 100, 1500), tmax=round(rng.uniform(5.0, 20.0), 2), nz=_log_int(rng, 50, 1000))
    if kind == "batch":
        nb_min = rng.randint(3, 5)
        return dict(kind=kind, models=_log_int(rng, 4, 48), nb_min=nb_min, nb_max=rng.randint(nb_min, 9),
                    nw=_log_int(rng, 33, 512), beta=round(rng.uniform(20.0, 100.0), 2))
    return dict(kind="fit", models=_log_int(rng, 4, 64), nb=rng.randint(3, 7), nw=_log_int(rng, 33, 512),
                beta=round(rng.uniform(20.0, 100.0), 2))


# -- models ----------------------------------------------------------------------------------------------------------


def _params(case, seed):
    """(bonds, hops, eps, u per site, fermionic signs) of the case's model."""
    rng = np.random.default_rng([seed, 11])
    ns = case["sites"]
    lattice = case.get("lattice", "siam")
    if lattice == "siam":
        u = rng.uniform(2.0, 6.0)
        eps = np.append(-u / 2, rng.uniform(-2.0, 2.0, ns - 1))
        return [(0, k) for k in range(1, ns)], rng.uniform(0.2, 1.0, ns - 1), eps, np.append(u, np.zeros(ns - 1)), False
    u = rng.uniform(2.0, 8.0)
    if lattice == "square":
        nx = {8: 4, 9: 3, 12: 4, 15: 5, 16: 4}[ns]
        bonds = ed.square_neighbors(nx, ns // nx)
    else:
        bonds = ed.chain_neighbors(ns)
    return bonds, np.ones(len(bonds)), np.full(ns, -u / 2), np.full(ns, u), True


def _model(par):
    bonds, hops, eps, u, fermionic = par
    if fermionic:
        return ed.HubbardModel(len(eps), bonds, inter=float(u[0]), eps=0.0, hop=1.0, mu=float(u[0]) / 2)
    return ed.SingleImpurityAndersonModel(float(u[0]), float(eps[0]), eps[1:], hops, mu=0.0)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _padded(n):
    """Row stride of whole 128-byte lines."""
    return (n + 15) // 16 * 16


def _vectors(case, seed):
    nu, nd = math.comb(case["sites"], case["n_up"]), math.comb(case["sites"], case["n_dn"])
    x = torch.rand((case["nvec"], nu, nd), dtype=torch.float64, device="cuda", generator=_generator(seed)) - 0.5
    return x / torch.linalg.vector_norm(x[0])


def _fit_params(case, seed):
    rng = np.random.default_rng([seed, 13])
    m, nb = case["models"], case["nb"]
    u = rng.uniform(2.0, 4.0, m)
    return u, rng.uniform(-2.0, 2.0, (m, nb)), rng.uniform(0.2, 1.0, (m, nb)), rng.uniform(-0.1, 0.1, (m, nb))


# -- the calls -------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "batch":
        p = random_batch(case["models"], seed, nb_range=(case["nb_min"], case["nb_max"]))
        s.update(batch=AndersonBatch(**p), eps=p["eps_bath"], v=p["v"], wn=matsubara(case["beta"], case["nw"]))
    elif kind == "fit":
        u, eps, v, shift = _fit_params(case, seed)
        wn = matsubara(case["beta"], case["nw"])
        delta = (v[:, None, :] ** 2 / (1j * wn[None, :, None] - eps[:, None, :] - shift[:, None, :])).sum(axis=2)
        s.update(batch=AndersonBatch(u=u, eps_imp=-u / 2, eps_bath=list(eps), v=list(v), mu=0.0, keep_basis=True),
                 eps=torch.from_numpy(eps), v=torch.from_numpy(v), wn=wn,
                 target=torch.from_numpy(1.0 / (1j * wn[None, :] - delta)))
    else:
        par = _params(case, seed)
        s.update(par=par, model=_model(par))
        if kind == "hv":
            op = s["op"] = s["model"].hamilton_operator(n_up=case["n_up"], n_dn=case["n_dn"])
            x = _vectors(case, seed)
            if case["padded"]:
                ld = s["ld"] = _padded(op.num_dn)
                s["x"] = torch.zeros((case["nvec"], op.num_up, ld), dtype=torch.float64, device="cuda")
                s["x"][:, :, :op.num_dn] = x
            else:
                s["x"] = x.view(case["nvec"], -1)
            s["y"] = torch.empty_like(s["x"])
        elif kind == "spectrum":
            s["z"] = np.linspace(-8.0, 8.0, case["nz"]) + 0.1j
        else:
            n_up, n_dn = case["n_up"], case["n_dn"]
            if kind == "solve":
                s["z"] = 1j * matsubara(case["beta"], case["nw"])
            if kind == "realtime":
                s["gs"] = ed.groundstate(s["model"], n_up, n_dn, tol=1e-12, device=True)
                s["omegas"] = np.linspace(-8.0, 8.0, case["nz"])
            if kind == "ground":
                s["v0"] = _start(case, seed)
            if not case.get("fresh"):  # a program that solves a model repeatedly has its operators
                for d in (-1, 0, 1) if kind != "ground" else (0,):
                    if 0 <= n_up + d <= case["sites"]:
                        s["model"].hamilton_operator(n_up=n_up + d, n_dn=n_dn)
    return s


def _start(case, seed):
    d = math.comb(case["sites"], case["n_up"]) * math.comb(case["sites"], case["n_dn"])
    return torch.rand(d, dtype=torch.float64, device="cuda", generator=_generator(seed)) - 0.5


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "hv":
        if case["padded"]:
            return state["op"].matvec_device_ld(state["x"], state["ld"], out=state["y"])
        return state["op"].matvec_device(state["x"], out=state["y"])
    if kind == "solve":
        model = _model(state["par"]) if case["fresh"] else state["model"]
        r = ed.greens_cf(model, state["z"], case["n_up"], case["n_dn"], nsteps=case["nsteps"])
        return {"e0": r.e0, "gf": r.gf, "norm2_p": r.norm2_p, "norm2_h": r.norm2_h}
    if kind == "ground":
        r = ed.groundstate(state["model"], case["n_up"], case["n_dn"], v0=state["v0"], device=True)
        return {"e0": r.energy, "psi": r.state}
    if kind == "spectrum":
        r = ed.gf_lehmann(state["model"], state["z"], case["beta"])
        return {"gf": r.gf, "occ": r.occ, "occ_double": r.occ_double}
    if kind == "realtime":
        t, greater = ed.gf_greater(state["model"], state["gs"], 0.0, case["tmax"], case["nt"])
        _, lesser = ed.gf_lesser(state["model"], state["gs"], 0.0, case["tmax"], case["nt"])
        _, gz = ed.fourier_t2z(t, greater - lesser, state["omegas"])
        return {"greater": greater, "lesser": lesser, "gz": gz}
    if kind == "batch":
        state["batch"].set_bath(state["eps"], state["v"])
        r = state["batch"].solve(state["wn"])
        return {"e0": r.e0, "g": r.g}
    eps, v = state["eps"].clone().requires_grad_(), state["v"].clone().requires_grad_()
    g = anderson_gf(eps, v, state["batch"], state["wn"])
    loss = (g - state["target"]).abs().pow(2).sum()
    loss.backward()
    return {"g": g.detach(), "loss": loss.detach(), "grad_eps": eps.grad, "grad_v": v.grad}


# -- work ------------------------------------------------------------------------------------------------------------


def _sector_work(case, dn=0):
    """(states, hop terms per state) of the case's sector (n_up + dn, n_dn)."""
    ns, nu, nd = case["sites"], case["n_up"] + dn, case["n_dn"]
    if not 0 <= nu <= ns:
        return 0, 0.0
    bonds = len(_params(case, 0)[0])
    per = sum(2.0 * bonds * n * (ns - n) / (ns * (ns - 1)) for n in (nu, nd))
    return math.comb(ns, nu) * math.comb(ns, nd), per


def work(case):
    """Bytes and operations one pass cannot do without: an H.v reads and writes a vector once, a Lanczos step reads two
    and writes one (about 100 steps to a ground state), a dense eigenproblem takes 6 n^3 operations, a pole or pair term
    10 per frequency."""
    kind = case["kind"]
    if kind == "hv":
        d, per = _sector_work(case)
        return {"bytes": 16.0 * d * case["nvec"], "flops": 2.0 * (per + 1) * d * case["nvec"]}
    if kind in ("solve", "ground", "realtime"):
        d, per = _sector_work(case)
        gs = 0 if kind == "realtime" else 100
        b, f = 24.0 * d * gs, (2.0 * per + 10) * d * gs
        if kind != "ground":
            m = case["nsteps"] if kind == "solve" else 12 * case["tmax"]
            for dn in (1, -1):
                d, per = _sector_work(case, dn)
                b, f = b + 24.0 * d * min(m, d), f + (2.0 * per + 10) * d * min(m, d)
        if kind == "solve":
            f += 10.0 * 2 * case["nsteps"] * case["nw"]
        elif kind == "realtime":
            f += case["nt"] * (40.0 * 2 * 12 * case["tmax"] + 60.0 * case["nz"])
        return {"bytes": b, "flops": f}
    if kind == "spectrum":
        ns, b, f = case["sites"], 0.0, 0.0
        for nu in range(ns + 1):
            for nd in range(ns + 1):
                d = math.comb(ns, nu) * math.comb(ns, nd)
                b, f = b + 8.0 * d * d, f + 6.0 * d ** 3
                if nu < ns:
                    m = math.comb(ns, nu + 1) * math.comb(ns, nd)
                    f += 2.0 * d * m * m + 10.0 * d * m * case["nz"]
        return {"bytes": b, "flops": f}
    if kind == "batch":
        sizes = range(case["nb_min"], case["nb_max"] + 1)
        share, steps = case["models"] / len(sizes), 200
    else:
        sizes, share, steps = [case["nb"]], case["models"], 400
    d = sum(math.comb(n + 1, (n + 1) // 2) ** 2 * share for n in sizes)
    hops = sum(sizes) / len(sizes)
    f = (2.0 * hops + 10) * d * steps + 10.0 * steps * case["models"] * case["nw"]
    if kind == "fit":
        f += 2.0 * 2 * 150 ** 2 * (d + 2.0 * case["nw"] * case["models"])
    return {"bytes": 24.0 * d * steps, "flops": f}


# -- reference values in 64 bits, plain torch and numpy --------------------------------------------------------------


class _Sector:
    """H of one sector from its definition: states in ascending order, up index slowest."""

    def __init__(self, par, n_up, n_dn, dev="cuda"):
        bonds, hops, eps, u, fermionic = par
        ns = len(eps)
        self.n, self.dev = ns, dev
        self.up, self.dn = (self._states(ns, n) for n in (n_up, n_dn))
        both = self.up[:, None] & self.dn[None, :]
        diag = sum(eps[i] * (((self.up >> i) & 1)[:, None] + ((self.dn >> i) & 1)[None, :]) + u[i] * ((both >> i) & 1)
                   for i in range(ns))
        self.diag = torch.as_tensor(diag, device=dev)
        self.shape = diag.shape
        self.hops = [[self._hop(st, i, j, t, fermionic) for (i, j), t in zip(bonds, hops)] for st in (self.up, self.dn)]

    @staticmethod
    def _states(ns, n):
        s = np.arange(1 << ns, dtype=np.int64)
        return s[sum((s >> i) & 1 for i in range(ns)) == n] if ns else s[:1]

    def _hop(self, st, i, j, t, fermionic):
        src = np.nonzero(((st >> i) ^ (st >> j)) & 1)[0]
        to = np.searchsorted(st, st[src] ^ (1 << i) ^ (1 << j))
        sign = np.ones(len(src))
        if fermionic:
            for k in range(i + 1, j):
                sign *= 1.0 - 2.0 * ((st[src] >> k) & 1)
        return [torch.as_tensor(a, device=self.dev) for a in (src, to, t * sign)]

    def __matmul__(self, x):
        x = x.view(self.shape)
        y = self.diag * x
        for src, to, val in self.hops[0]:  # the targets of one bond are all different
            y[to] += val[:, None] * x[src]
        for src, to, val in self.hops[1]:
            y[:, to] += val[None, :] * x[:, src]
        return y.view(-1)

    def ladder(self, other, psi):
        """c+ or c of site 0, spin up, from sector ``other`` into this one."""
        src = np.searchsorted(other.up, self.up ^ 1)
        ok = (src < len(other.up)) & (other.up[np.minimum(src, len(other.up) - 1)] == (self.up ^ 1))
        rows = torch.as_tensor(np.nonzero(ok)[0], device=self.dev)
        y = torch.zeros(self.shape, dtype=torch.float64, device=self.dev)
        y[rows] = psi.view(other.shape)[torch.as_tensor(src[ok], device=self.dev)]
        return y.view(-1)

    def dense(self):
        d = self.diag.numel()
        h = torch.diag(self.diag.reshape(-1)).view(self.shape + self.shape)
        iu = torch.arange(self.shape[0], device=self.dev)
        idn = torch.arange(self.shape[1], device=self.dev)
        for src, to, val in self.hops[0]:
            h[to[:, None], idn[None, :], src[:, None], idn[None, :]] += val[:, None]
        for src, to, val in self.hops[1]:
            h[iu[:, None], to[None, :], iu[:, None], src[None, :]] += val[None, :]
        return h.reshape(d, d)


def _lanczos(h, v, m, tol=None):
    """Lanczos with every vector orthogonalised twice against all before it; with ``tol`` until the lowest Ritz pair has
    that residual.  Returns (a, b, vectors as rows)."""
    V = torch.zeros((m, v.numel()), dtype=torch.float64, device=v.device)
    V[0] = v / torch.linalg.vector_norm(v)
    a, b = [], []
    for j in range(m):
        w = h @ V[j]
        a.append(float(V[j] @ w))
        for _ in range(2):
            w = w - (V[:j + 1] @ w) @ V[:j + 1]
        nrm = float(torch.linalg.vector_norm(w))
        if nrm < 1e-11 or j + 1 == m:
            break
        if tol is not None and j % 10 == 9:
            s = np.linalg.eigh(np.diag(a) + np.diag(b, 1) + np.diag(b, -1))[1][:, 0]
            if nrm * abs(s[-1]) < tol:
                break
        b.append(nrm)
        V[j + 1] = w / nrm
    return np.array(a), np.array(b[:len(a) - 1]), V


def _ground(h, v0):
    a, b, V = _lanczos(h, v0, min(h.diag.numel(), 400), tol=1e-13)
    w, s = np.linalg.eigh(np.diag(a) + np.diag(b, 1) + np.diag(b, -1))
    psi = torch.as_tensor(s[:, 0], device=v0.device) @ V[:len(a)]
    return w[0], psi * (torch.sign(psi @ v0) / torch.linalg.vector_norm(psi))


def _fraction(a, b, n2, z):
    t = np.zeros_like(z)
    for j in range(len(a) - 1, 0, -1):
        t = b[j - 1] ** 2 / (z - a[j] - t)
    return n2 / (z - a[0] - t)


def _parts(par, case, e0, psi, h):
    for sign in (1, -1):
        if 0 <= case["n_up"] + sign <= case["sites"]:
            hs = _Sector(par, case["n_up"] + sign, case["n_dn"])
            phi = hs.ladder(h, psi)
            yield sign, hs, phi, float(phi @ phi)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "fit":  # no closed form of the gradients short of a dense resolvent for every frequency and parameter
        return None
    par = _params(case, seed)
    if kind == "spectrum":
        return _exact_spectrum(case, par)
    h = _Sector(par, case["n_up"], case["n_dn"])
    if kind == "hv":
        x = _vectors(case, seed)
        y = torch.stack([(h @ v).view(h.shape) for v in x])
        if case["padded"]:
            return torch.nn.functional.pad(y, (0, _padded(h.shape[1]) - h.shape[1]))
        return y.view(case["nvec"], -1)
    v0 = _start(case, seed)
    e0, psi = _ground(h, v0)
    if kind == "ground":
        return {"e0": float(e0), "psi": psi}
    if kind == "solve":
        z = 1j * matsubara(case["beta"], case["nw"])
        g, norms = 0.0, {1: 0.0, -1: 0.0}
        for sign, hs, phi, n2 in _parts(par, case, e0, psi, h):
            a, b, _ = _lanczos(hs, phi, min(case["nsteps"], phi.numel()))
            g = g + sign * _fraction(a, b, n2, sign * z + e0)
            norms[sign] = n2
        return {"e0": float(e0), "gf": g, "norm2_p": norms[1], "norm2_h": norms[-1]}
    t = np.linspace(0.0, case["tmax"], case["nt"])
    out = {"greater": np.zeros(len(t), complex), "lesser": np.zeros(len(t), complex)}
    for sign, hs, phi, n2 in _parts(par, case, e0, psi, h):
        a, b, _ = _lanczos(hs, phi, min(int(12 * case["tmax"]) + 60, phi.numel()))
        th, s = np.linalg.eigh(np.diag(a) + np.diag(b, 1) + np.diag(b, -1))
        out["greater" if sign > 0 else "lesser"] = (
            -1j * sign * n2 * (np.exp(-1j * sign * (th[None, :] - e0) * t[:, None]) @ s[0] ** 2))
    g = out["greater"] - out["lesser"]
    z = np.linspace(-8.0, 8.0, case["nz"]) - 1j * np.log(1e-2) / t[-1]
    dt = t[1] - t[0]
    x = 1j * z * dt
    series = np.abs(x) < 0.5
    xs = np.where(series, x, 0.0)
    e1, e2 = (sum(c(n) * xs ** n for n in range(24)) for c in (lambda n: 1.0 / math.factorial(n + 1),
                                                              lambda n: (n + 1.0) / math.factorial(n + 2)))
    xl = np.where(series, 1.0, x)
    e1 = np.where(series, e1, (np.exp(xl) - 1) / xl)
    e2 = np.where(series, e2, (xl * np.exp(xl) - np.exp(xl) + 1) / xl ** 2)
    ph = np.exp(1j * z[:, None] * t[None, :-1])
    out["gz"] = dt * (e1 * (ph @ g[:-1]) + e2 * (ph @ np.diff(g)))
    return out


def _exact_spectrum(case, par):
    ns, beta = case["sites"], case["beta"]
    z = torch.as_tensor(np.linspace(-8.0, 8.0, case["nz"]) + 0.1j, device="cuda")
    sec = {(nu, nd): _Sector(par, nu, nd) for nu in range(ns + 1) for nd in range(ns + 1)}
    eig = {k: torch.linalg.eigh(s.dense()) for k, s in sec.items()}
    emin = min(float(w[0]) for w, _ in eig.values())
    part, occ, docc = 0.0, 0.0, 0.0
    g = torch.zeros(len(z), dtype=torch.complex128, device="cuda")
    for (nu, nd), s in sec.items():
        if nu == ns:
            continue
        s1, (w, v), (w1, v1) = sec[nu + 1, nd], eig[nu, nd], eig[nu + 1, nd]
        boltz = torch.exp(-beta * (w - emin))
        part += float(boltz.sum())
        rho = (v ** 2 @ boltz).view(s.shape)
        up = torch.as_tensor((s.up & 1) == 1, device="cuda")
        dn = torch.as_tensor((s.dn & 1) == 1, device="cuda")
        occ += float(rho[up].sum())
        docc += float(rho[up][:, dn].sum())
        cv = torch.stack([s1.ladder(s, v[:, k]) for k in range(v.shape[1])], dim=1)
        wt = (v1.T @ cv) ** 2 * (boltz[None, :] + torch.exp(-beta * (w1 - emin))[:, None])
        pole = w1[:, None] - w[None, :]
        keep = wt.reshape(-1) > 0
        wt, pole = wt.reshape(-1)[keep], pole.reshape(-1)[keep]
        for k in range(0, len(z), 20):
            g[k:k + 20] += (wt[None, :] / (z[k:k + 20, None] - pole[None, :])).sum(dim=1)
    return {"gf": (g / part).cpu().numpy(), "occ": occ / part, "occ_double": docc / part}


def _exact_batch(case, seed):
    if case["nb_max"] > 5 or case["models"] > 16:  # one dense eigenproblem a sector and model
        return None
    p = random_batch(case["models"], seed, nb_range=(case["nb_min"], case["nb_max"]))
    z = 1j * matsubara(case["beta"], case["nw"])
    e0s, gs = [], []
    for i in range(case["models"]):
        nb = len(p["v"][i])
        par = ([(0, k) for k in range(1, nb + 1)], p["v"][i], np.append(p["eps_imp"][i], p["eps_bath"][i]),
               np.append(p["u"][i], np.zeros(nb)), False)
        n = (nb + 1) // 2
        h = _Sector(par, n, n, "cpu")
        w, v = np.linalg.eigh(h.dense().numpy())
        psi = torch.from_numpy(np.ascontiguousarray(v[:, 0]))
        g = 0.0
        for sign in (1, -1):
            hs = _Sector(par, n + sign, n, "cpu")
            w1, v1 = np.linalg.eigh(hs.dense().numpy())
            ov = v1.T @ hs.ladder(h, psi).numpy()
            g = g + (ov ** 2 / (z[:, None] - sign * (w1 - w[0]))).sum(axis=1)
        e0s.append(w[0])
        gs.append(g)
    return {"e0": np.array(e0s), "g": np.array(gs)}
