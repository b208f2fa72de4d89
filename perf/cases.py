"""The work that users of this framework have it do, as cases to be timed and checked.

Every case is one call of a public entry point on a batch that is already resident on the device:

* ``widom``  adsorption screening: Henry coefficient and heat of adsorption by test-particle
             insertion, in mixed precision (the default) or in Float64;
* ``grad``   the same with the derivatives with respect to force-field parameters and charges;
* ``moves``  many attempts of one Monte Carlo move type on loaded chains;
* ``gcmc``   grand-canonical cycles, the body of an adsorption isotherm;
* ``nvt``    canonical cycles with test insertions into the loaded configurations.

Frameworks are this repository's own: RUBTAK (the published benchmark system, 3x3x3, 3,078 atoms),
the hexagonal 13/13/15 A cell and the cubic 12.9 A cell of the benchmark's configurations at
densities that leave pores open, and random triclinic cells of the screening configuration. All
are replicated to widths of twice the 12 A cutoffs. Temperatures are those of adsorption work.

The ranges that `draw` spreads over: 1,000 to 1,000,000 insertions for one framework, 2 to 32
frameworks at 10,000 to 100,000 insertions each, 1,000 to 100,000 insertions in Float64, 1 to 512
chains of 20 to 2,000 attempts, guests CO2 (three charged sites) and CH4 (one uncharged site).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()
sys.path.insert(0, os.path.join(ROOT, "pureadsorb.jl_amd"))

import pureadsorb_amd as pa  # noqa: E402
from pureadsorb_amd import synth  # noqa: E402

CUTOFF, PRECISION = 12.0, 1.0e-6
GOLDEN = os.path.join(ROOT, "tests", "golden")


def listed():
    return [
        # a quick estimate for one porous framework: the smallest call, where launches and host work count
        dict(name="widom_quick", do="widom", fw="hex", atoms=40, nfw=1, guest="co2", n=5_000, T=298.15, prec="mixed"),
        # the published benchmark system at its published sample size
        dict(name="widom_rubtak", do="widom", fw="rubtak", atoms=114, nfw=1, guest="co2", n=1_000_000, T=298.15,
             prec="mixed"),
        # the benchmark's CO2 cell at a porous density, the usual production sample
        dict(name="widom_porous", do="widom", fw="hex", atoms=80, nfw=1, guest="co2", n=1_000_000, T=298.15,
             prec="mixed"),
        # screening: a batch of unlike frameworks in one call, odd sizes, many k-vectors each
        dict(name="widom_screen", do="widom", fw="mix", atoms=0, nfw=32, guest="co2", n=3_200_000, T=298.15,
             prec="mixed"),
        # an uncharged united-atom guest: Lennard-Jones only
        dict(name="widom_ch4", do="widom", fw="cubic", atoms=53, nfw=1, guest="ch4", n=100_000, T=298.15, prec="mixed"),
        # a Float64 reference value, as a study reports it beside the mixed-precision one
        dict(name="widom_f64", do="widom", fw="rubtak", atoms=114, nfw=1, guest="co2", n=100_000, T=298.15, prec="f64"),
        # force-field fitting: gradients over a training set of frameworks
        dict(name="grad_fit", do="grad", fw="mix", atoms=0, nfw=16, guest="co2", n=1_600_000, T=298.15, prec="mixed"),
        # one chain, the latency of a move
        dict(name="moves_one", do="moves", fw="rubtak", atoms=114, nfw=1, guest="co2", n=500, move=1, load=1500, T=298.15),
        # many chains, the throughput of moves
        dict(name="moves_many", do="moves", fw="rubtak", atoms=114, nfw=512, guest="co2", n=60, move=1, load=300, T=298.15),
        # an isotherm's body: 8 fugacities x 3 replicas on the move benchmark's cell
        dict(name="gcmc_isotherm", do="gcmc", fw="hex32", atoms=40, nfw=24, guest="co2", n=40, cycle=20, load=150, T=298.15),
        # canonical chains with test insertions after every cycle
        dict(name="nvt_insert", do="nvt", fw="rubtak", atoms=114, nfw=16, guest="co2", n=10, cycle=20, load=300, nw=256,
             T=298.15),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["widom", "widom", "screen", "f64", "grad", "moves", "gcmc", "nvt"])
    T = rng.uniform(273.0, 350.0)
    guest = "ch4" if rng.random() < 0.25 else "co2"
    if do in ("widom", "f64"):
        fw = rng.choice(["hex", "hex", "rubtak"])
        atoms = 114 if fw == "rubtak" else rng.randint(25, 80)
        guest = "co2" if fw == "rubtak" else guest
        n = _log(rng, 1_000, 1_000_000 if do == "widom" else 100_000)
        return dict(do="widom", fw=fw, atoms=atoms, nfw=1, guest=guest, n=n, T=T, prec="f64" if do == "f64" else "mixed")
    if do == "screen":
        nfw = rng.randint(2, 32)
        return dict(do="widom", fw="mix", atoms=0, nfw=nfw, guest=guest, n=nfw * _log(rng, 10_000, 100_000) + rng.randint(0, 99),
                    T=T, prec="mixed")
    if do == "grad":
        nfw = rng.randint(1, 16)
        return dict(do="grad", fw="mix", atoms=0, nfw=nfw, guest="co2", n=nfw * _log(rng, 10_000, 100_000), T=T, prec="mixed")
    fw = rng.choice(["hex32", "rubtak"])
    atoms = 114 if fw == "rubtak" else rng.randint(30, 50)
    if do == "moves":
        nfw = _log(rng, 1, 512)
        return dict(do="moves", fw=fw, atoms=atoms, nfw=nfw, guest="co2", n=max(20, min(2_000, _log(rng, 5_000, 30_000) // nfw)),
                    move=rng.choice([1, 2, 3]), load=_log(rng, 100, 400), T=T)
    if do == "gcmc":
        return dict(do="gcmc", fw=fw, atoms=atoms, nfw=rng.randint(3, 24), guest="co2", n=rng.randint(20, 40),
                    cycle=rng.randint(5, 20), load=_log(rng, 50, 150), T=T)
    return dict(do="nvt", fw=fw, atoms=atoms, nfw=rng.randint(1, 24), guest="co2", n=rng.randint(10, 20),
                cycle=rng.randint(5, 20), load=_log(rng, 100, 300), nw=_log(rng, 32, 256), T=T)


# ---- inputs ------------------------------------------------------------------------------------
def _frameworks(case, seed):
    fw, seed = case["fw"], int(seed)
    if fw == "rubtak":
        return [pa.replicate(pa.read_cif(os.path.join(GOLDEN, "RUBTAK.cif")), (3, 3, 3))]
    if fw == "cubic":
        return [pa.replicate(synth.synthetic_framework(12.9, 12.9, 12.9, 90, 90, 90, case["atoms"], seed), (2, 2, 2))]
    if fw in ("hex", "hex32"):
        cell = synth.synthetic_framework(13.0, 13.0, 15.0, 90, 90, 120, case["atoms"], seed, charge_sd=0.15)
        return [pa.replicate(cell, (3, 3, 3) if fw == "hex" else (3, 3, 2))]
    # cells and atom counts belong to the case, the atoms and their charges come from the seed
    out, r = [], np.random.RandomState(case["nfw"])
    for i in range(case["nfw"]):
        a, b, c = r.uniform(10.0, 30.0, 3)
        angles = r.uniform(70.0, 110.0, 3)
        volume = pa.volume(pa.cell_matrix(a, b, c, *angles))
        atoms = max(8, int(round(volume * math.exp(r.uniform(math.log(0.012), math.log(0.04))))))
        cell = synth.synthetic_framework(a, b, c, *angles, atoms, seed * 1000 + i, charge_sd=0.15)
        out.append(pa.replicate(cell, synth.replication_for_width(cell, 2 * CUTOFF)))
    return out


def _model(case, seed):
    """Frameworks, force field and guest of a case."""
    fws = _frameworks(case, seed)
    if case["fw"] == "rubtak":
        ff = pa.read_forcefield(os.path.join(GOLDEN, "trappe.yaml"))
        guest = pa.read_guest(os.path.join(GOLDEN, case["guest"] + ".yaml"), ff)
    else:
        ff = synth.synthetic_forcefield(CUTOFF, guest=case["guest"])
        guest = synth.co2_guest(ff) if case["guest"] == "co2" else synth.ch4_guest(ff)
    return fws, ff, guest


def prepare(case, seed):
    fws, ff, guest = _model(case, seed)
    chains = case["do"] in ("moves", "gcmc", "nvt")
    if chains:
        fws = fws * case["nfw"]
    batch = pa.FrameworkBatch(fws, ff, guest, pa.EwaldParams(CUTOFF, PRECISION), fullk=chains)
    s = dict(case=case, seed=int(seed), batch=batch, guest=guest, ff=ff)
    if chains:
        # chains loaded by insertions at high pressure, so that no guest overlaps anything
        s["state"] = pa.SystemState(batch, guest, [0] * batch.nsys, T=case["T"], seed=int(seed), capacities=[600] * batch.nsys)
        pa.mc_moves(s["state"], pa.MOVE_INSERTION, case["load"], T=case["T"], fugacity=1.0e6)
        # an isotherm's fugacities, 1 kPa to 1 MPa, three replicas each
        s["fugacity"] = np.array([1.0e3 * 10.0 ** (3.0 * ((i // 3) % 8) / 7.0) for i in range(batch.nsys)])
    return s


# ---- one pass ----------------------------------------------------------------------------------
def _fields(results, names, dtype):
    return {k: np.array([getattr(r, k) for r in results], dtype=dtype) for k in names}


WIDOM = ("mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "q_st_err", "ln_K_H")


def _widom_out(results, dtype):
    return {**_fields(results, WIDOM, dtype), **_fields(results, ("nsamples", "nblocks"), np.int64)}


def run(s):
    c = s["case"]
    if c["do"] == "widom":
        res = pa.widom(s["batch"], s["guest"], T=c["T"], ninsert=c["n"], seed=s["seed"], precision=c["prec"])
        # the mixed path sums Float32 energy terms, and its results are kept in that type
        return _widom_out(res, np.float64 if c["prec"] == "f64" else np.float32)
    if c["do"] == "grad":
        res = pa.widom_grad(s["batch"], s["guest"], T=c["T"], ninsert=c["n"], seed=s["seed"], precision=c["prec"])
        out = _widom_out([r.result for r in res], np.float32)
        for k in ("dlnkh_deps", "dlnkh_dsig", "dqst_deps", "dqst_dsig", "dlnkh_dq", "dqst_dq"):
            out[k] = np.concatenate([getattr(r, k) for r in res]).astype(np.float32)
        return out
    st, T = s["state"], c["T"]
    if c["do"] == "moves":
        tr = pa.mc_moves(st, c["move"], c["n"], T=T, step_trans=0.5, step_rot=0.5, trace=True)
        # every attempt's energy change, and which guest was tried and whether it moved
        return {"dU": np.ascontiguousarray(tr[..., 2]), "slot": tr[..., 1].astype(np.int64),
                "accepted": tr[..., 3].astype(np.int64)}
    if c["do"] == "gcmc":
        res = pa.run_gcmc(st, T=T, n_warmup=0, n_production=c["n"], n_audit=1000, step_trans=1.0, step_rot=0.5,
                          fugacity=s["fugacity"], min_cycle_length=c["cycle"], nblocks=5)
        return {**_fields(res, ("loading", "loading_err", "energy", "energy_err"), np.float64),
                **_fields(res, ("max_occupancy", "accepted", "attempted"), np.int64)}
    res = pa.run_nvt(s["batch"], st, s["guest"], s["ff"], T=T, n_warmup=0, n_production=c["n"], n_widom_per_cycle=c["nw"],
                     n_audit=1000, step_trans=0.3, step_rot=0.3, min_cycle_length=c["cycle"], widom_seed=s["seed"] + 1000,
                     nblocks=5)
    return _fields(res, ("energy", "energy_err", "mu_ex", "mu_ex_err", "K_H", "K_H_err", "q_st", "q_st_err", "acceptance"),
                   np.float64)


# ---- what a pass cannot do without -------------------------------------------------------------
def work(case):
    """Bytes: the tables read once and the results written once. Flops: per attempt, and per
    insertion that overlaps no atom (about 0.55 of them), the in-cutoff pairs at the mean density
    (61 each with charges, 16 without), 11 per k-vector and site and 4 per k-vector."""
    sphere = 4.0 / 3.0 * math.pi * CUTOFF**3
    if case["fw"] == "mix":
        cell, density, k = 8.0e3, 0.022, 450.0
    elif case["fw"] == "cubic":
        cell, density, k = 2146.7, case["atoms"] / 2146.7, 0.0
    elif case["fw"] == "rubtak":
        cell, density, k = 2276.2, 114 / 2276.2, 190.0
    else:
        cell, density, k = 2195.4, case["atoms"] / 2195.4, 184.0
    sites, per_pair = (3, 61.0) if case["guest"] == "co2" else (1, 16.0)
    k = k if sites == 3 else 0.0
    natoms = density * max(cell, 3.2e4)
    if case["do"] in ("widom", "grad"):
        n = case["n"]
        flops = 0.55 * n * (per_pair * sites * density * sphere + (11.0 * sites + 4.0) * k)
        nbytes = case["nfw"] * (32.0 * natoms + 48.0 * k) + 8.0 * n + (16.0 * natoms * case["nfw"] if case["do"] == "grad" else 0.0)
        return {"bytes": nbytes, "flops": flops}
    kfull = 4600.0 if case["fw"] == "rubtak" else 3300.0  # a guest's structure factor is nonzero at every k-vector
    attempts = case["nfw"] * case["n"] * case.get("cycle", 1)
    inserts = case["nfw"] * case["n"] * case.get("nw", 0)
    flops = (attempts + inserts) * (per_pair * sites * density * sphere + (11.0 * sites + 4.0) * kfull)
    return {"bytes": case["nfw"] * 2 * 16.0 * kfull + 32.0 * natoms + 32.0 * attempts + 8.0 * inserts, "flops": flops}


# ---- the same in 64 bits, in plain torch --------------------------------------------------------
KB = 1.38064852e-23 / 1.6021766208e-19  # eV/K
KE = 14.399645351950548  # eV A / e^2
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _i64(v):
    return v - (1 << 64) if v >= (1 << 63) else v


def _shift(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _mix(seed, index):
    """SplitMix64 of seed + index * golden on int64 tensors (wrapping)."""
    z = seed + index * _i64(0x9E3779B97F4A7C15)
    z = (z ^ _shift(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _shift(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _shift(z, 31)


def _uniforms(seed, cycle, move, count):
    """`count` uniforms of the counter-based stream (seed, cycle, move), broadcast: (..., count)."""
    key = _mix(_mix(seed, cycle), move)
    return torch.stack([_shift(_mix(key, torch.full_like(key, i)), 11).double() * 2.0**-53 for i in range(count)], -1)


def _quaternions(u):
    a, b = torch.sqrt(1 - u[..., 0]), torch.sqrt(u[..., 0])
    p, q = 2 * math.pi * u[..., 1], 2 * math.pi * u[..., 2]
    return torch.stack([a * torch.cos(p), b * torch.sin(q), b * torch.cos(q), a * torch.sin(p)], -1)


def _rotated(q, sites):
    """(..., sites, 3): the sites turned by unit quaternions (x, y, z, w)."""
    v, w = q[..., None, :3], q[..., None, 3:]
    s = sites.expand(q.shape[:-1] + sites.shape)
    v = v.expand_as(s)
    return s + 2 * torch.linalg.cross(v, torch.linalg.cross(v, s) + w * s)


class _Exact:
    """Insertion energies of one framework in Float64."""

    def __init__(self, fw, ff, guest, rows=3.0e7):
        t = lambda x: torch.tensor(np.asarray(x, dtype=np.float64), device=DEV)  # noqa: E731
        lo, hi, target = 0.0, 20.0, CUTOFF * PRECISION / 2
        for _ in range(200):
            mid = (lo + hi) / 2
            lo, hi = (mid, hi) if math.erfc(mid) > target else (lo, mid)
        self.alpha = alpha = (lo + hi) / 2 / CUTOFF
        self.A, self.inv = t(fw.cell), t(np.linalg.inv(fw.cell))
        self.V = V = abs(float(np.linalg.det(fw.cell)))
        self.frac, self.q = t(fw.frac), t(fw.charges)
        self.images = int(np.prod(fw.replication))
        self.atype = torch.tensor([ff.names.index(s + "_") for s in fw.symbols], device=DEV)
        self.gtype = torch.tensor([int(x) for x in guest.types], device=DEV)
        self.sites, self.gq = t(guest.sites), t(guest.charges)
        self.sigma, self.eps = t(np.diag(ff.sigma)), t(np.diag(ff.epsilon))
        self.cutoff, self.tail = float(ff.cutoff), bool(ff.tail)
        self.charged = bool(np.any(np.asarray(guest.charges) != 0))
        self.rows = rows
        # k = 2 pi A^-T n in the half space n1 >= 0; the framework couples to multiples of its replication
        B = 2 * math.pi * np.linalg.inv(fw.cell).T
        kmax = 2 * alpha * math.sqrt(-math.log(PRECISION / 2))
        m = [int(math.ceil(kmax * np.linalg.norm(fw.cell[:, d]) / (2 * math.pi))) for d in range(3)]
        n = np.stack(np.meshgrid(np.arange(0, m[0] + 1), np.arange(-m[1], m[1] + 1), np.arange(-m[2], m[2] + 1),
                                 indexing="ij"), -1).reshape(-1, 3)
        k = n @ B.T
        k2 = (k * k).sum(1)
        keep = (k2 > 0) & (np.sqrt(k2) <= kmax)
        n, k, k2 = n[keep], k[keep], k2[keep]
        pre = np.where(n[:, 0] == 0, 1.0, 2.0) * 2 * math.pi / V * np.exp(-k2 / (4 * alpha**2)) / k2
        self.offset_self = 0.0
        if self.charged:
            # the guest with itself, a mean over 64 fixed orientations
            o = torch.arange(1, 65, device=DEV)
            turned = _rotated(_quaternions(_uniforms(torch.full_like(o, 0x5E1F), torch.zeros_like(o), o, 3)), self.sites)
            ph = turned @ t(k).T
            re, im = (self.gq[:, None] * torch.cos(ph)).sum(1), (self.gq[:, None] * torch.sin(ph)).sum(1)
            self.offset_self = KE * float(((re**2 + im**2) @ t(pre)).mean()) - KE * alpha / math.sqrt(math.pi) * float((self.gq**2).sum())
            for i in range(len(guest.charges)):
                for j in range(i):
                    r = float(np.linalg.norm(np.asarray(guest.sites)[i] - np.asarray(guest.sites)[j]))
                    self.offset_self -= KE * float(guest.charges[i] * guest.charges[j]) * math.erf(alpha * r) / r
        c = np.all(n % np.array(fw.replication) == 0, 1)
        self.n, self.pre = t(n[c]), t(pre[c])

    def offset(self, sigma, eps, q):
        """What every insertion carries: tail correction, net charge and the guest with itself."""
        total = torch.as_tensor(self.offset_self, dtype=torch.float64, device=DEV)
        if self.tail:
            ntypes = len(sigma)
            host = torch.bincount(self.atype, minlength=ntypes).double()
            mine = torch.bincount(self.gtype, minlength=ntypes).double()
            s, e = (sigma[:, None] + sigma) / 2, self._mixed(eps, eps)
            x = s / self.cutoff
            total = total + 8 * math.pi / 3 / self.V * ((2 * host[:, None] * mine + mine[:, None] * mine) * e * s**3 * (x**9 / 3 - x**3)).sum()
        if self.charged:
            Qh, Qg = q.sum(), self.gq.sum()
            total = total - KE * math.pi / (2 * self.V * self.alpha**2) * ((Qh + Qg) ** 2 - Qh**2)
        return total

    @staticmethod
    def _mixed(a, b):
        p = a[:, None] * b
        return torch.where(p > 0, torch.sqrt(torch.where(p > 0, p, torch.ones_like(p))), torch.zeros_like(p))

    def sites_of(self, seed, system, j):
        chain = _mix(torch.full_like(j, _i64(seed & (2**64 - 1))), torch.full_like(j, system + 1))
        u = _uniforms(chain, j + 1, torch.zeros_like(j), 6)
        return u[:, None, :3] + _rotated(_quaternions(u[:, 3:]), self.sites) @ self.inv.T

    def energies(self, f, sigma, eps, q):
        """Energies (eV) of guests with fractional site coordinates f (m, sites, 3)."""
        E = self.offset(sigma, eps, q).expand(len(f))
        for a in range(f.shape[1]):
            d = [f[:, a, i, None] - self.frac[:, i] for i in range(3)]
            d = [x - torch.round(x) for x in d]
            r2 = sum((self.A[i, 0] * d[0] + self.A[i, 1] * d[1] + self.A[i, 2] * d[2]) ** 2 for i in range(3))
            s = (sigma[self.gtype[a]] + sigma[self.atype]) / 2
            e = self._mixed(eps[self.gtype[a], None], eps)[0][self.atype]
            x = (s * s / r2) ** 3
            E = E + torch.where(r2 < self.cutoff**2, 4 * e * (x * x - x), 0.0).sum(1)
            if self.charged:
                r = torch.sqrt(r2)
                E = E + KE * self.gq[a] * torch.where(r2 < CUTOFF**2, torch.erfc(self.alpha * r) / r, 0.0) @ q
        if self.charged:
            hp = 2 * math.pi * (self.n @ self.frac.T)
            Sr, Si = torch.cos(hp) @ q, torch.sin(hp) @ q
            for a in range(f.shape[1]):
                ph = 2 * math.pi * (f[:, a] @ self.n.T)
                E = E + 2 * KE * self.gq[a] * (torch.cos(ph) @ (self.pre * Sr) + torch.sin(ph) @ (self.pre * Si))
        return E

    def insertions(self, seed, system, count):
        out, step = [], max(1, int(self.rows / max(len(self.q), 1)))
        for j0 in range(0, count, step):
            j = torch.arange(j0, min(count, j0 + step), device=DEV)
            out.append(self.energies(self.sites_of(seed, system, j), self.sigma, self.eps, self.q))
        return torch.cat(out)


def _statistics(dU, V, T, nblocks=10):
    """The Widom estimators and their block errors from the insertion energies."""
    kT = KB * T
    lw = -dU / kT
    M = float(lw.max())
    M = M if math.isfinite(M) else 0.0
    w = torch.exp(lw - M)
    u = torch.where(w > 0, dU * w, torch.zeros_like(w))
    per = len(dU) // nblocks
    cut = [(k * per, len(dU) if k == nblocks - 1 else (k + 1) * per) for k in range(nblocks)]
    mW, mU = (np.array([float(x[a:b].mean()) for a, b in cut]) for x in (w, u))
    W, U = float(w.mean()), float(u.mean())
    vW, vU = ((mW - W) ** 2).sum() / (nblocks - 1), ((mU - U) ** 2).sum() / (nblocks - 1)
    cov = ((mW - W) * (mU - U)).sum() / (nblocks - 1)
    sem, ratio = math.sqrt(vW / nblocks), U / W
    var = ratio**2 * (vU / U**2 + vW / W**2 - 2 * cov / (U * W)) / nblocks if U else 0.0
    lnW = math.log(W) + M
    return dict(mu_ex=-kT * lnW, mu_ex_err=kT * sem / W, K_H=V * W * math.exp(M) / kT, K_H_err=V * sem * math.exp(M) / kT,
                q_st=kT - ratio, q_st_err=math.sqrt(max(var, 0.0)), ln_K_H=math.log(V) + lnW - math.log(kT))


def _counts(n, nsys):
    run = min(max((n // nsys) // 4, 1), 256)
    full, rest = divmod(n, run)
    out = [full // nsys * run + (run if s < full % nsys else 0) for s in range(nsys)]
    out[full % nsys] += rest
    return out


def _gradients(x, seed, system, dU, T):
    """d ln K_H and d q_st with respect to every type's epsilon and sigma and every atom's charge,
    by automatic differentiation over the insertions whose weight counts in Float64."""
    beta = 1 / (KB * T)
    lw = -beta * dU
    w = torch.exp(lw - lw.max())
    pick = torch.nonzero(w > math.exp(-40.0))[:, 0]
    W, R = float(w.sum()), float((w * dU)[pick].sum())
    leaf = [v.clone().requires_grad_(True) for v in (x.sigma, x.eps, x.q)]
    G, H = ([torch.zeros_like(v) for v in leaf] for _ in range(2))
    step = max(1, int(2.0e6 / max(len(x.q), 1)))
    for i in range(0, len(pick), step):
        at = pick[i:i + step]
        E = x.energies(x.sites_of(seed, system, at), *leaf)
        for acc, c in ((G, w[at]), (H, (w * dU)[at])):
            for a, g in zip(acc, torch.autograd.grad((c * E).sum(), leaf, retain_graph=True, allow_unused=True)):
                a += 0 if g is None else g
    for acc in (G, H):  # an atom moves with its replication images
        acc[2] = acc[2].reshape(x.images, -1).mean(0).repeat(x.images)
    dk = [-beta * g / W for g in G]
    dq = [-(g - beta * h) / W - beta * (R / W) * (g / W) for g, h in zip(G, H)]
    return dict(dlnkh_deps=dk[1], dlnkh_dsig=dk[0], dqst_deps=dq[1], dqst_dsig=dq[0], dlnkh_dq=dk[2], dqst_dq=dq[2])


def exact(case, seed):
    # a chain's outputs follow from hundreds of decisions in sequence, one after the other and with
    # every earlier one's rounding: there is no plain 64-bit value of them in 20 seconds
    if case["do"] not in ("widom", "grad"):
        return None
    fws, ff, guest = _model(case, seed)
    out, grads = {k: [] for k in WIDOM}, []
    counts = _counts(case["n"], len(fws))
    for s, fw in enumerate(fws):
        x = _Exact(fw, ff, guest)
        dU = x.insertions(int(seed), s, counts[s])
        for k, v in _statistics(dU, x.V, case["T"]).items():
            out[k].append(v)
        if case["do"] == "grad":
            grads.append(_gradients(x, int(seed), s, dU, case["T"]))
    got = {k: np.array(v, dtype=np.float64) for k, v in out.items()}
    got.update(nsamples=None, nblocks=None)
    for k in grads[0] if grads else ():
        got[k] = torch.cat([g[k] for g in grads]).cpu().numpy()
    return got
