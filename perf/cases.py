"""Work that a user of this package has it do, as cases that can be timed.

A case is a dict of plain values: what is asked for (``ask``), how many
molecules, how large they are and under which options.  Molecules are those
of ``dxtb_amd.workloads``: CHNO chains of ``lo``..``hi`` carbons and water
clusters of ``lo``..``hi`` waters (about three atoms and eight orbitals per
unit either way), ``water`` being the clusters' share.  The composition is
fixed by the case; every geometry is drawn from the seed.

``tol`` is the SCF threshold on the potential: 1e-10 where tight results are
served or differentiated further (the threshold of ``bench.py``), 0 for the
calculator's defaults.

``exact`` is an independent GFN1 single point in 64 bits (torch on the CPU,
dense eigensolves, gradient by automatic differentiation), for cases small
enough for it.
"""

from __future__ import annotations

import json
import math
from pathlib import Path

import numpy as np
import torch

import dxtb_amd
from dxtb_amd import workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.serving import RaggedServer, Request

MD_STEP = 0.01  # bohr, drift per trajectory step (one time step at room temperature)
MD_LENGTH = 4


def listed():
    return [
        # one ethane-sized molecule: the smallest call, all latency
        {"name": "energy_small", "ask": "energy", "count": 1, "lo": 2, "hi": 2, "water": 0.0, "tol": 0.0},
        # octane, the reference's own plain single point, with its forces
        {"name": "forces_octane", "ask": "forces", "count": 1, "lo": 8, "hi": 8, "water": 0.0, "tol": 0.0},
        # one drug- or oligomer-sized molecule of some hundred atoms
        {"name": "forces_chain", "ask": "forces", "count": 1, "lo": 39, "hi": 39, "water": 0.0, "tol": 1e-10},
        # molecular dynamics of a solvent cluster, warm starts along the trajectory
        {"name": "md_cluster", "ask": "md", "count": 1, "lo": 66, "hi": 66, "water": 1.0, "tol": 1e-10},
        # the largest single system: 600 waters, 1800 atoms, 4800 orbitals
        {"name": "forces_water600", "ask": "forces", "count": 1, "lo": 600, "hi": 600, "water": 1.0, "tol": 1e-10},
        # screening energies of a padded batch that fills the chip
        {"name": "energy_batch", "ask": "energy", "count": 256, "lo": 2, "hi": 20, "water": 0.0, "tol": 0.0},
        # forces of a large batch (data set labelling, parallel relaxations)
        {"name": "forces_batch", "ask": "forces", "count": 512, "lo": 5, "hi": 40, "water": 0.0, "tol": 1e-10},
        # alkyl radicals (bond dissociation): open shells take the eigensolver in every SCF step
        {"name": "forces_radicals", "ask": "radicals", "count": 64, "lo": 3, "hi": 17, "water": 0.0, "tol": 1e-10},
        # orbital energies of a batch (spectra, frontier levels)
        {"name": "orbitals_batch", "ask": "orbitals", "count": 64, "lo": 3, "hi": 15, "water": 0.3, "tol": 1e-10},
        # parameter gradients of a training batch
        {"name": "params_batch", "ask": "params", "count": 64, "lo": 2, "hi": 12, "water": 0.3, "tol": 1e-10},
        # a burst of requests of all sizes (5 to 200 atoms) to the serving loop
        {"name": "serve_burst", "ask": "serve", "count": 600, "lo": 1, "hi": 66, "water": 0.3, "tol": 1e-10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    ask = rng.choice(["energy", "forces", "forces", "single", "single", "md", "radicals", "orbitals", "params", "serve"])
    tol = rng.choice([0.0, 1e-10, 1e-10])
    water = rng.choice([0.0, 0.0, 1.0])
    if ask == "single":  # one molecule, up to some thousand orbitals
        u = _log_int(rng, 2, 260)
        return {"ask": "forces", "count": 1, "lo": u, "hi": u, "water": 1.0 if u > 66 else water, "tol": tol}
    if ask == "md":
        u = _log_int(rng, 5, 90)
        return {"ask": ask, "count": 1, "lo": u, "hi": u, "water": 1.0 if u > 66 else water, "tol": 1e-10}
    if ask == "serve":
        return {"ask": ask, "count": _log_int(rng, 40, 600), "lo": 1, "hi": rng.randint(20, 66), "water": 0.3, "tol": 1e-10}
    if ask in ("energy", "forces"):
        return {"ask": ask, "count": _log_int(rng, 6, 512), "lo": rng.randint(1, 6), "hi": rng.randint(9, 40),
                "water": water, "tol": tol}
    if ask == "radicals":
        return {"ask": ask, "count": _log_int(rng, 6, 160), "lo": rng.randint(2, 5), "hi": rng.randint(6, 19),
                "water": 0.0, "tol": 1e-10}
    return {"ask": ask, "count": _log_int(rng, 4, 96), "lo": rng.randint(1, 4), "hi": rng.randint(6, 16),
            "water": 0.3, "tol": 1e-10}


# --------------------------------------------------------------- the inputs
def _molecules(case, seed):
    """[(numbers, positions in bohr)]: composition from the case, geometry from the seed."""
    mix = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    noise = np.random.default_rng([seed, 77])
    out = []
    for _ in range(case["count"]):
        if case["ask"] == "serve":  # log-uniform sizes, as the request stream's
            u = int(round(math.exp(mix.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        else:
            u = int(mix.integers(case["lo"], case["hi"] + 1))
        if mix.random() < case["water"]:
            out.append(workloads.water_cluster(noise, u, order="compact" if case["count"] > 1 else "lex"))
        else:
            if case["ask"] == "radicals":  # an alkane less a hydrogen at the end of the chain
                z, p = (a[:-1] for a in workloads.chain(mix, u, p_n=0.0, p_o=0.0, sigma=0.0))
            else:
                z, p = workloads.chain(mix, u, sigma=0.0)
            out.append((z, p + noise.normal(0.0, 0.03 * 1.8897261246, size=p.shape)))
    return out


def _scf_options(case):
    return {"x_atol": case["tol"], "x_atol_max": case["tol"], "maxiter": 300} if case["tol"] else {}


def prepare(case, seed):
    mols = _molecules(case, seed)
    ask = case["ask"]
    if ask == "serve":
        return {"ask": ask, "server": RaggedServer("cuda:0", ScfOptions(**_scf_options(case))), "mols": mols}
    if case["count"] == 1:
        z, p = mols[0]
    else:
        z, p = workloads.pad(mols)
    opts = {**_scf_options(case), "exclude": ["disp"]}
    state = {"ask": ask}
    if ask == "md":
        opts["warm_start"] = True
        drift = np.random.default_rng([seed, 78]).normal(size=p.shape)
        state["trajectory"] = [torch.tensor(p + k * MD_STEP * drift, device="cuda:0") for k in range(MD_LENGTH)]
    else:
        state["positions"] = torch.tensor(p, device="cuda:0", requires_grad=ask in ("forces", "radicals"))
    state["calc"] = dxtb_amd.GFN1Calculator(torch.tensor(z, device="cuda:0"), opts=opts, dtype=torch.float64)
    state["spin"] = torch.ones(case["count"]) if ask == "radicals" else None
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    ask = state["ask"]
    if ask == "serve":
        server = state["server"]
        reqs = [Request(rid=i, numbers=z, positions=p) for i, (z, p) in enumerate(state["mols"])]
        server.feed(reqs)
        server.drain()
        return {"energy": np.array([r.energy for r in reqs]), "forces": np.concatenate([r.forces for r in reqs])}
    calc = state["calc"]
    if ask == "md":
        return [calc.forces_analytical(p) for p in state["trajectory"]]
    pos = state["positions"]
    if ask == "energy":
        return {"energy": calc.get_energy(pos)}
    if ask == "orbitals":
        return {"orbital_energies": calc.get_mo_energies(pos)}
    if ask == "params":
        g = calc.get_param_gradient(pos)
        h = g.pop("hamiltonian")
        out = {sym: torch.cat([v if v.ndim == 2 else v[:, None] for _, v in sorted(d.items())], dim=1)
               for sym, d in g.items()}
        out["shell"] = torch.stack([h["shell"][k] for k in sorted(h["shell"])], dim=1)
        return out
    energy = calc.get_energy(pos, 0, state["spin"])
    (g,) = torch.autograd.grad(energy.sum(), pos)
    return {"energy": energy.detach(), "forces": -g}


# -------------------------------------------------------- what a pass is about
_ORBITALS = {1: 2, 6: 4, 7: 4, 8: 4}
_VALENCE = {1: 1, 6: 4, 7: 5, 8: 6}
SCF_STEPS = 12  # potential evaluations that a self-consistent run of these molecules takes at least


def work(case):
    """Per geometry: a Cholesky reduction and one eigensolve of the start
    (n^3/3 + n^3, and 9 1/3 n^3), then SCF_STEPS potential updates, each at
    least a projection of the Fock matrix on occupied x virtual orbitals
    (2 k n^2 + 2 k (n - k) n), a rotation between them (4 k (n - k) n) and
    half a density product (k n^2); S, H0 and gamma once out and in, P and W
    likewise for gradients."""
    steps = MD_LENGTH if case["ask"] == "md" else 1
    bytes_, flops = 0.0, 0.0
    for z, _ in _molecules(case, 1):
        n = sum(_ORBITALS[int(a)] for a in z)
        k = sum(_VALENCE[int(a)] for a in z) / 2.0
        flops += n**3 * (4.0 / 3.0 + 28.0 / 3.0) + SCF_STEPS * (3.0 * k * n * n + 6.0 * k * (n - k) * n)
        mats = 2 + (0 if case["ask"] in ("energy", "orbitals") else 2)
        bytes_ += 2.0 * 8.0 * mats * n * n + 8.0 * (6 * len(z) + n)
    return {"bytes": steps * bytes_, "flops": steps * flops}


# ---------------------------------------------- GFN1 in plain torch, 64 bits
_BOHR, _EV, _KB = 0.52917721090380, 27.21138505, 3.166808578545117e-06
_RCOV = {1: 0.32, 6: 0.75, 7: 0.71, 8: 0.63}
_RAD = {1: 0.32, 6: 0.75, 7: 0.71, 8: 0.64}


def _parameters():
    here = Path(dxtb_amd.__file__).resolve().parent / "param"
    with open(here / "gfn1.json") as fh:
        par = json.load(fh)
    with np.load(here / "sto_ng.npz", allow_pickle=False) as d:
        sto = {k: d[k].astype(np.float64) for k in d.files}
    return par, sto


def _contraction(sto, ng, n, l, zeta):
    row = n - 1 + (0, 4)[l]
    c, a = sto[f"sto{ng}"][0, row].copy(), sto[f"sto{ng}"][1, row] * zeta**2
    return a, c * (2 * a / math.pi) ** 0.75 * (4 * a) ** (l / 2)


def _ss(a, c, b, d):
    return float((c[:, None] * d[None] * (math.pi / (a[:, None] + b[None])) ** 1.5).sum())


class _Model:
    """Shell and orbital tables of one molecule."""

    def __init__(self, z):
        par, sto = _parameters()
        els = {e["z"]: (s, e) for s, e in par["elements"].items()}
        self.z = [int(a) for a in z]
        sh = []
        for at, a in enumerate(self.z):
            _, e = els[a]
            for k, (n, l) in enumerate(e["shells"]):
                al, co = _contraction(sto, e["ngauss"][k], n, l, e["slater"][k])
                if not e["valence"][k]:  # orthogonal to the shell below
                    b, d = sh[-1]["al"], sh[-1]["co"]
                    al, co = np.concatenate([al, b]), np.concatenate([co, -_ss(b, d, al, co) * d])
                    co = co / math.sqrt(_ss(al, co, al, co))
                sh.append({"at": at, "l": l, "al": al, "co": co, "val": e["valence"][k], "ref": e["refocc"][k],
                           "level": e["levels"][k] / _EV, "kcn": e["kcn"][k] / _EV, "poly": e["shpoly"][k],
                           "hard": e["lgam"][k] * e["gam"]})
        t = lambda key: torch.tensor([s[key] for s in sh], dtype=torch.float64)
        self.al = torch.ones(len(sh), 8, dtype=torch.float64)
        self.co = torch.zeros(len(sh), 8, dtype=torch.float64)
        for i, s in enumerate(sh):
            self.al[i, : len(s["al"])] = torch.tensor(s["al"])
            self.co[i, : len(s["al"])] = torch.tensor(s["co"])
        self.at = torch.tensor([s["at"] for s in sh])
        self.level, self.kcn, self.poly, self.hard = t("level"), t("kcn"), t("poly"), t("hard")
        h = par["hamiltonian"]

        def scale(a, b):
            ka, kb = (h["shell"]["sp"[s["l"]] * 2] if s["val"] else h["kpol"] for s in (a, b))
            if not (a["val"] and b["val"]):
                return 0.5 * (ka + kb)
            (na, ea), (nb, eb) = els[self.z[a["at"]]], els[self.z[b["at"]]]
            pair = h["kpair"].get(f"{na}-{nb}", h["kpair"].get(f"{nb}-{na}", 1.0))
            return (ka if a["l"] == b["l"] else h["shell"]["sp"]) * pair * (1 + h["enscale"] * (ea["en"] - eb["en"]) ** 2)

        kinds = {}
        index = [kinds.setdefault((self.z[s["at"]], s["l"], s["val"]), (len(kinds), s)) for s in sh]
        small = torch.tensor([[scale(a, b) for _, b in kinds.values()] for _, a in kinds.values()], dtype=torch.float64)
        ids = torch.tensor([i for i, _ in index])
        self.K = small[ids][:, ids]
        # orbitals: shell and direction (p in the order y, z, x)
        axes = {0: [(0, 0, 0)], 1: [(0, 1, 0), (0, 0, 1), (1, 0, 0)]}
        orb = [(i, d) for i, s in enumerate(sh) for d in axes[s["l"]]]
        self.sh = torch.tensor([i for i, _ in orb])
        self.d = torch.tensor([d for _, d in orb], dtype=torch.float64)
        self.n0 = t("ref")[self.sh] / (2 * torch.tensor([s["l"] for s in sh])[self.sh] + 1)
        at = lambda key: torch.tensor([els[a][1][key] for a in self.z], dtype=torch.float64)
        self.gam3, self.zeff, self.arep, self.kexp = at("gam3"), at("zeff"), at("arep"), par["repulsion"]["kexp"]
        self.rcov = torch.tensor([4 / 3 * _RCOV[a] / _BOHR for a in self.z], dtype=torch.float64)
        self.rad = torch.tensor([_RAD[a] / _BOHR for a in self.z], dtype=torch.float64)

    def integrals(self, x):
        """S, H0, gamma (shells), repulsion energy at positions x."""
        nat = len(self.z)
        eye = torch.eye(nat, dtype=torch.float64)
        vec = x[:, None] - x[None]
        r = torch.sqrt((vec**2).sum(-1) + eye)  # the diagonal, 1, is masked below
        off = 1 - eye
        cn = (off * (r <= 25.0) / (1 + torch.exp(-16.0 * ((self.rcov[:, None] + self.rcov[None]) / r - 1)))).sum(1)
        rep = self.zeff[:, None] * self.zeff[None] * torch.exp(-torch.sqrt(self.arep[:, None] * self.arep[None]) * r**self.kexp) / r
        erep = 0.5 * (rep * off * (r <= 25.0)).sum()
        a, b = self.at[:, None], self.at[None]
        r2 = (vec**2).sum(-1)[a, b]
        avg = 2 / (1 / self.hard[:, None] + 1 / self.hard[None])
        gamma = 1 / torch.sqrt(r2 + 1 / avg**2)
        al, be = self.al[:, None, :, None], self.al[None, :, None, :]
        ip = 1 / (al + be)
        s00 = self.co[:, None, :, None] * self.co[None, :, None, :] * (math.pi * ip) ** 1.5 * torch.exp(-al * be * ip * r2[..., None, None])
        con = lambda w: (w * s00).sum((-1, -2))[self.sh][:, self.sh]
        rij = vec[self.at[self.sh]][:, self.at[self.sh]]
        ui, uj = (rij * self.d[:, None]).sum(-1), (rij * self.d[None]).sum(-1)
        dd = self.d @ self.d.T
        pi_, pj = self.d.sum(1)[:, None], self.d.sum(1)[None]
        si, sj = 1 - pi_, 1 - pj
        S = si * sj * con(1.0) + pi_ * sj * ui * con(-be * ip) + si * pj * uj * con(al * ip)
        S = S + pi_ * pj * (ui * uj * con(-al * be * ip * ip) + dd * con(0.5 * ip))
        same = (self.at[self.sh][:, None] == self.at[self.sh][None])
        S = torch.where(same, torch.eye(len(self.sh), dtype=torch.float64), S * (r[a, b] < 50.0)[self.sh][:, self.sh])
        h = self.level - self.kcn * cn[self.at]
        q = torch.sqrt(r / (self.rad[:, None] + self.rad[None]))[a, b]
        fac = 0.5 * (h[:, None] + h[None]) * self.K * (1 + self.poly[:, None] * q) * (1 + self.poly[None] * q)
        fac = fac[self.sh][:, self.sh]
        H0 = torch.where(same, torch.diag(h[self.sh]), S * fac)
        return S, H0, gamma, erep

    def reduce(self, v, index, size):
        return torch.zeros(size, dtype=torch.float64).index_add_(0, index, v)


def _fermi(e, nel, kt):
    f = lambda mu: 1 / (1 + torch.exp(torch.clamp((e - mu) / kt, -700, 700)))
    if nel == 0:
        return torch.zeros_like(e)
    lo, hi = float(e[0]) - 1, float(e[-1]) + 1
    mu = float(e[int(nel) - 1 : int(nel) + 1].mean())
    for _ in range(200):
        s = float(f(mu).sum()) - nel
        if abs(s) < 1e-12:
            break
        lo, hi = (mu, hi) if s < 0 else (lo, mu)
        mu = 0.5 * (lo + hi)
    return f(mu)


def _single_point(z, p, spin=0, gradient=True):
    """(energy, forces or None, orbital energies) of one molecule."""
    m = _Model(z)
    x = torch.tensor(p, dtype=torch.float64, requires_grad=gradient)
    S, H0, gamma, erep = m.integrals(x)
    Sd, Hd, Gd = S.detach(), H0.detach(), gamma.detach()
    L = torch.linalg.cholesky(Sd)
    nel = float(m.n0.sum())
    counts = [round((nel + spin) / 2), round((nel - spin) / 2)]
    kt = 300.0 * _KB
    nsh, nat = len(m.at), len(m.z)

    def evaluate(v):
        F = Hd - 0.5 * Sd * (v[m.sh][:, None] + v[m.sh][None])
        A = torch.linalg.solve_triangular(L, F, upper=False)
        A = torch.linalg.solve_triangular(L, A.T, upper=False)
        e, C = torch.linalg.eigh(0.5 * (A + A.T))
        C = torch.linalg.solve_triangular(L.T, C, upper=True)
        occ = [_fermi(e, c, kt) for c in counts]
        P = (C * (occ[0] + occ[1])) @ C.T
        q = m.n0 - (P * Sd).sum(1)
        qsh = m.reduce(q, m.sh, nsh)
        qat = m.reduce(qsh, m.at, nat)
        return Gd @ qsh + (m.gam3 * qat**2)[m.at], (e, C, occ, P, qsh, qat)

    v = torch.zeros(nsh, dtype=torch.float64)
    xs, fs = [], []
    for _ in range(200):
        out, _ = evaluate(v)
        f = out - v
        if float(f.abs().max()) < 1e-13:
            break
        xs, fs = (xs + [v])[-8:], (fs + [f])[-8:]
        if len(xs) > 1:
            dF = torch.stack([fs[-1] - g for g in fs[:-1]], 1)
            dX = torch.stack([xs[-1] - g for g in xs[:-1]], 1)
            th = torch.linalg.lstsq(dF, fs[-1][:, None], driver="gelsd").solution[:, 0]
            v = xs[-1] - dX @ th + 0.5 * (fs[-1] - dF @ th)
        else:
            v = v + 0.5 * f
    vout, (e, C, occ, P, qsh, qat) = evaluate(out)
    ts = sum((torch.xlogy(o, o) + torch.xlogy(1 - o, 1 - o)).sum() for o in occ)
    energy = (P * Hd).sum() + 0.5 * qsh @ Gd @ qsh + (m.gam3 * qat**3).sum() / 3 + kt * ts + erep.detach()
    if not gradient:
        return float(energy), None, e
    # the energy is stationary in the density: dE/dR at fixed P, W and charges
    W = (C * ((occ[0] + occ[1]) * e)) @ C.T
    fixed = (P * H0).sum() + 0.5 * qsh @ gamma @ qsh - (P * S * vout[m.sh][None]).sum() - (W * S).sum() + erep
    (g,) = torch.autograd.grad(fixed, x)
    return float(energy), -g, e


def exact(case, seed):
    mols = _molecules(case, seed)
    cost = sum((sum(_ORBITALS[int(a)] for a in z) / 100.0) ** 2.5 * 0.2 + 0.12 for z, _ in mols)
    if case["ask"] in ("params", "md") or cost > 20:
        return None
    threads = torch.get_num_threads()
    torch.set_num_threads(min(threads, 8))
    gradient = case["ask"] in ("forces", "radicals", "serve")
    try:
        res = [_single_point(z, p, 1 if case["ask"] == "radicals" else 0, gradient) for z, p in mols]
    finally:
        torch.set_num_threads(threads)
    energy = torch.tensor([r[0] for r in res], dtype=torch.float64)
    if case["ask"] == "orbitals":  # padding levels lie at zero, in order with the others
        n = max(len(r[2]) for r in res)
        levels = [torch.sort(torch.cat([r[2], torch.zeros(n - len(r[2]), dtype=torch.float64)])).values for r in res]
        return {"orbital_energies": torch.stack(levels) if case["count"] > 1 else levels[0]}
    if case["ask"] == "serve":
        return {"energy": energy, "forces": torch.cat([r[1] for r in res])}
    out = {"energy": energy if case["count"] > 1 else energy[0]}
    if gradient:
        nat = max(len(z) for z, _ in mols)
        forces = torch.zeros(len(mols), nat, 3, dtype=torch.float64)
        for b, (_, f, _) in enumerate(res):
            forces[b, : len(f)] = f
        out["forces"] = forces if case["count"] > 1 else forces[0]
    return out
