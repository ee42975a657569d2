"""The work a user of the engine has it do, as measurable cases.

Every case goes through the package's public entry points: a stretch of molecular
dynamics followed by the download of the frame it ends in (`Engine.run` and
`Engine.download`, how trajectories are sampled), a single-point evaluation
(`Engine.upload` and `Engine.compute_forces`) or a force-matching loss with its
gradient (`md_gpu_amd.fit.fm_loss` and its backward pass).

The systems are the package's own generators (argon, Ar-Xe batches, molten NaCl,
flexible and rigid water) with thermal displacements; the launch settings are the ones
that the autotuner picks for these workloads, fixed here so that a run does not depend
on a tuning pass.  Stretches are short enough that a frame is still that of its inputs:
rounding grows along a trajectory, fastest where velocities come from constrained
positions (rigid water).  A case's `kind`:

  argon         plain Lennard-Jones, NVE velocity Verlet
  npt           the same under Berendsen temperature and pressure coupling
  arxe          many small replicas of uneven size in one launch
  nacl          ions: Wolf, reaction-field or damped Coulomb, or smooth PME
  water         flexible 3-site water, Nose-Hoover velocity Verlet
  water_rigid   rigid 3-site water (SETTLE), Wolf Coulomb or smooth PME
  forces        forces, energies and virial of given positions
  fm            force matching over frames of NaCl

`exact` restates the arithmetic in 64 bits with plain torch: a neighbor matrix, the pair
laws, the integrators, SHAKE for rigid molecules and smooth PME.
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from md_gpu_amd import systems as S

COUL = {"rf": S.COUL_RF, "wolf": S.COUL_WOLF, "damped": S.COUL_DAMPED, "pme": S.COUL_DAMPED}


def listed():
    """The cases; each comment says what the case stands for."""
    return [
        # the smallest call: a few steps of a few hundred atoms between two prints
        dict(name="argon256_10steps", kind="argon", size=4, steps=10, launch="lanes=16,persist=1"),
        # the classic argon benchmark, small enough for the one-launch kernel
        dict(name="argon864_100steps", kind="argon", size=6, steps=100, launch="lanes=16,persist=1"),
        # equilibration of a Lennard-Jones liquid at constant pressure, default launch settings
        dict(name="argon4000_npt_40steps", kind="npt", size=10, steps=40, launch=""),
        # a small parameter sweep: uneven replicas in one launch
        dict(name="arxe64_60steps", kind="arxe", size=64, nmax=8192, steps=60,
             launch="lanes=4,check_every=4,build_lanes=4,defer=0"),
        # the headline batch: 512 replicas, 1.3 million atoms
        dict(name="arxe512_60steps", kind="arxe", size=512, nmax=8192, steps=60,
             launch="lanes=4,check_every=4,build_lanes=4,defer=0"),
        # single-point forces and energies of the reference's example size (reaction field)
        dict(name="nacl4096_rf_forces", kind="forces", size=16, coulomb="rf", launch=""),
        # molten salt with Wolf electrostatics
        dict(name="nacl32768_wolf_30steps", kind="nacl", size=32, coulomb="wolf", steps=30,
             launch="lanes=8,check_every=8,build_lanes=8,refresh=1"),
        # the same salt with Ewald electrostatics
        dict(name="nacl32768_pme_30steps", kind="nacl", size=32, coulomb="pme", order=4, steps=30,
             launch="lanes=8,check_every=3,build_lanes=8,defer=0"),
        # a small rigid water box with Ewald electrostatics: launch-bound, ragged tiles
        dict(name="water6591_rigid_pme_6steps", kind="water_rigid", size=2197, coulomb="pme", order=4, steps=6,
             launch="lanes=8,check_every=2,build_lanes=8,defer=0"),
        # rigid water, production size, Ewald electrostatics
        dict(name="water196608_rigid_pme_4steps", kind="water_rigid", size=65536, coulomb="pme", order=4, steps=4,
             launch="lanes=8,check_every=1,build_lanes=8,defer=0"),
        # flexible water, production size
        dict(name="water196608_nvt_40steps", kind="water", size=65536, coulomb="wolf", steps=40,
             launch="lanes=8,check_every=4,build_lanes=8"),
        # one loss-and-gradient evaluation of a force-field fit
        dict(name="nacl4096x64_fm", kind="fm", size=16, frames=64, launch="lanes=8"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["argon", "argon", "npt", "arxe", "arxe", "forces", "nacl", "nacl", "nacl_pme", "water",
                       "water_rigid", "water_rigid", "fm"])
    lanes = rng.choice([4, 8, 16])
    check = rng.randint(1, 12)
    launch = "lanes=%d,check_every=%d,build_lanes=%d,cell_div=%d" % (lanes, check, rng.choice([4, 8]), rng.choice([1, 2, 2, 2, 3]))
    steps = rng.randint(5, 30)
    if kind == "argon":
        size = rng.randint(4, 16)
        persist = size <= 10 and rng.random() < 0.7
        return dict(kind=kind, size=size, steps=rng.randint(5, 100), launch="lanes=%d,persist=1" % lanes if persist else launch)
    if kind == "npt":
        return dict(kind=kind, size=rng.randint(5, 16), steps=steps, launch=launch)
    if kind == "arxe":
        return dict(kind=kind, size=int(round(_log(rng, 4, 400))), nmax=rng.choice([2048, 4096, 8192]), steps=rng.randint(5, 60),
                    launch=launch + ",defer=%d" % rng.randint(0, 1))
    if kind == "forces":
        return dict(kind=kind, size=2 * rng.randint(6, 16), coulomb=rng.choice(["rf", "wolf", "damped"]), launch=launch)
    if kind == "nacl":
        return dict(kind=kind, size=2 * rng.randint(6, 18), coulomb=rng.choice(["rf", "wolf", "wolf", "damped"]), steps=steps,
                    launch=launch + ",refresh=%d,defer=%d" % (rng.randint(0, 1), rng.randint(0, 1)))
    if kind == "nacl_pme":
        return dict(kind="nacl", size=2 * rng.randint(6, 18), coulomb="pme", order=rng.choice([4, 4, 6]), steps=steps,
                    launch="lanes=%d,check_every=%d,build_lanes=8" % (lanes, rng.randint(1, 4)))
    if kind == "water":
        return dict(kind=kind, size=int(round(_log(rng, 700, 60000))), coulomb="wolf", steps=steps, launch=launch)
    if kind == "water_rigid":
        return dict(kind=kind, size=int(round(_log(rng, 700, 60000))), coulomb=rng.choice(["pme", "pme", "wolf"]),
                    order=rng.choice([4, 4, 6]), steps=rng.randint(2, 4),
                    launch="lanes=%d,check_every=%d,build_lanes=8" % (lanes, rng.randint(1, 4)))
    return dict(kind="fm", size=2 * rng.randint(6, 8), frames=rng.randint(4, 64), launch="lanes=%d" % lanes)


# ------------------------------------------------------------------ inputs

def _jitter(s, rng, amp):
    """s with thermal displacements of amp A per axis (at most 2.5 amp)."""
    d = np.clip(rng.normal(0.0, amp, s.pos.shape), -2.5 * amp, 2.5 * amp)
    s.pos = S.wrap_centered(s.pos + d, s.box.astype(np.float64)).astype(np.float32)
    return s


def _systems(case, seed):
    """The replicas of an MD or single-point case, from the seed alone."""
    rng = np.random.default_rng([seed, 77])
    kind, n = case["kind"], case["size"]
    if kind in ("argon", "npt"):
        s = _jitter(S.argon(ncell=n, seed=seed), rng, 0.2)
        if kind == "npt":
            s = dataclasses.replace(s, integrator="leapfrog", thermostat="berendsen", tau=100.0, barostat="berendsen",
                                    P0=1.0, tau_p=200.0, compress=4.5e-4)
        return [s]
    if kind == "arxe":   # sizes, types and temperatures are the case's; positions and velocities the seed's
        batch = [_jitter(s, rng, 0.15) for s in S.arxe_replicas(nrep=n, nmax=case["nmax"])]
        return [dataclasses.replace(s, vel=S.maxwell_boltzmann(rng, s.mass, s.T0).astype(np.float32)) for s in batch]
    if kind in ("nacl", "forces"):
        ff = S.nacl_ff()
        if case["coulomb"] in ("rf", "damped"):   # reaction field at water's permittivity, as the parity tests
            ff = dataclasses.replace(ff, coulomb=COUL[case["coulomb"]], eps_rf=78.0, alpha=3.09 / ff.rc)
        s = _jitter(S.nacl(nsites=n, seed=seed, ff=ff), rng, 0.2)
    elif kind == "water":
        s = S.water(nmol=n, seed=seed)
    else:
        s = S.water(nmol=n, seed=seed, rigid=True)
    if case["coulomb"] == "pme":
        s = S.with_pme(s, spacing=1.0, order=case["order"])
    return [s]


def _fm_problem(case, seed):
    """Frames around the NaCl lattice, target forces of a perturbed model, trial parameters."""
    rng = np.random.default_rng([seed, 78])
    base = S.nacl(nsites=case["size"], seed=seed)
    box = base.box.astype(np.float64)
    d = rng.normal(0.0, 0.25, (case["frames"], base.n, 3))
    frames = S.wrap_centered(base.pos + np.clip(d, -0.6, 0.6), box).astype(np.float32)
    tgt_ff, tgt_q = S.perturb_nacl_ff(base.ff, seed=seed)
    targets = np.empty_like(frames)
    for k, x in enumerate(frames):
        s = dataclasses.replace(base, ff=tgt_ff, charge=base.charge * np.float32(tgt_q))
        targets[k] = _Forces([s], torch.as_tensor(x, dtype=torch.float64, device="cuda"))().cpu().numpy()
    eps, sig = S.eps_sig_from_lj(base.ff.lj1, base.ff.lj2)
    iu = np.triu_indices(base.ff.ntype)
    theta = np.concatenate([eps[iu], sig[iu], [1.0]])
    theta = theta * (1.0 + rng.uniform(-0.02, 0.02, theta.size))
    return base, frames, targets, theta


def prepare(case, seed):
    from md_gpu_amd import engine as E
    launch = dict((k, int(v)) for k, v in (kv.split("=") for kv in case["launch"].split(",") if kv))
    if case["kind"] == "fm":
        from md_gpu_amd.fit import ForceMatch
        base, frames, targets, theta = _fm_problem(case, seed)
        e = E.Engine.from_system(base)
        e.set_launch(**launch)
        return dict(case=case, e=e, fm=ForceMatch(e, base, frames, targets), theta=torch.as_tensor(theta))
    sys_ = _systems(case, seed)
    e = E.Engine.from_system(sys_)
    if launch:
        e.set_launch(**launch)
    return dict(case=case, e=e, pos=np.concatenate([s.pos for s in sys_]), vel=np.concatenate([s.vel for s in sys_]))


def run(state):
    case, e = state["case"], state["e"]
    if case["kind"] == "fm":
        from md_gpu_amd.fit import fm_loss
        theta = state["theta"].clone().requires_grad_()
        loss = fm_loss(theta, state["fm"])
        loss.backward()
        return {"loss": loss.detach(), "grad": theta.grad}
    if case["kind"] == "forces":
        e.upload(state["pos"], state["vel"])
        f, en, w = e.compute_forces()
        return {"force": f, "energy": en, "virial": w}
    e.run(case["steps"], stats=False)
    pos, vel, force = e.download()
    out = {"pos": pos, "vel": vel, "force": force}
    if case["kind"] == "npt":
        out["box"] = e.box()
    return out


def _pairs(n, box, rc):
    """Mean unordered pairs within rc at uniform density."""
    return 0.5 * n * (n / float(np.prod(box))) * 4.0 / 3.0 * math.pi * rc ** 3


def work(case):
    """Bytes: the state read once and what comes back written once.  Operations: the pair
    law of each unordered pair within the cutoff, per step (36 for Lennard-Jones, 45 with the
    reaction field, 60 and 65 with Wolf or damped Coulomb), and the transforms of PME."""
    kind, n = case["kind"], case["size"]
    per = {"argon": 36, "npt": 36, "arxe": 36, "water": 60, "water_rigid": 60}.get(kind, 65)
    if case.get("coulomb") == "rf":
        per = 45
    if kind == "fm":
        atoms = n ** 3
        p = _pairs(atoms, [2.82 * n] * 3, 12.0)
        return {"bytes": 28.0 * atoms * case["frames"], "flops": 110.0 * p * case["frames"]}
    if kind == "arxe":
        mean = (case["nmax"] - 256) / math.log(case["nmax"] / 256.0)
        atoms, pairs = n * mean, n * _pairs(mean, [(mean / 0.018) ** (1 / 3)] * 3, 2.5 * 4.10)
    elif kind in ("argon", "npt"):
        atoms = 4 * n ** 3
        pairs = _pairs(atoms, [n * 5.2486] * 3, 2.5 * 3.405)
    elif kind in ("nacl", "forces"):
        atoms = n ** 3
        pairs = _pairs(atoms, [2.82 * n] * 3, 12.0)
    else:
        atoms = 3 * n
        pairs = _pairs(atoms, [(n / 0.033428) ** (1 / 3)] * 3, 10.0)
    flops = per * pairs
    if case.get("coulomb") == "pme":
        edge = 2.82 * n if kind == "nacl" else (n / 0.033428) ** (1 / 3)
        k3 = edge ** 3
        flops += 2 * 2.5 * k3 * math.log2(k3) + atoms * case["order"] ** 3 * 9
    if kind == "forces":
        return {"bytes": (28.0 + 12.0) * atoms, "flops": flops}
    return {"bytes": (36.0 + 36.0) * atoms, "flops": flops * case["steps"]}


# ------------------------------------------------------------------ 64-bit restatement

def _near(x, box, rl):
    """(i, j) of all ordered pairs of one system within rl, sorted by i: by cells where the box
    holds at least three per edge, else all against all."""
    n, out = x.shape[0], []
    nc = torch.floor(box / rl).long()
    if n < 6000 or int(nc.min()) < 3:
        step = max(1, 40_000_000 // n)
        for a in range(0, n, step):
            d = x[a:a + step, None] - x[None]
            d -= box * torch.round(d / box)
            i, j = torch.nonzero((d * d).sum(-1) < rl * rl, as_tuple=True)
            out.append(torch.stack([i + a, j]))
        i, j = torch.cat(out, 1)
        return i[i != j], j[i != j]
    c = torch.floor((x / box + 0.5) * nc).long().clamp(min=0)
    c = torch.minimum(c, nc - 1)
    key = (c[:, 0] * nc[1] + c[:, 1]) * nc[2] + c[:, 2]
    ncell = int(nc.prod())
    order = torch.argsort(key)
    count = torch.bincount(key, minlength=ncell)
    first = torch.cumsum(count, 0) - count
    table = torch.full((ncell, int(count.max())), -1, dtype=torch.long, device=x.device)
    table[key[order], torch.arange(n, device=x.device) - first[key[order]]] = order
    cell = torch.arange(ncell, device=x.device)
    cc = torch.stack([cell // (nc[1] * nc[2]), cell // nc[2] % nc[1], cell % nc[2]], 1)
    off = torch.cartesian_prod(*[torch.arange(-1, 2, device=x.device)] * 3)
    nb = (cc[:, None] + off) % nc
    nb = (nb[..., 0] * nc[1] + nb[..., 1]) * nc[2] + nb[..., 2]
    m = table.shape[1]
    step = max(1, 60_000_000 // (27 * m * m))
    for a in range(0, ncell, step):
        own, cand = table[a:a + step], table[nb[a:a + step]].reshape(-1, 27 * m)
        ok = (own >= 0)[:, :, None] & (cand >= 0)[:, None]
        d = x[own][:, :, None] - x[cand][:, None]
        d -= box * torch.round(d / box)
        ok &= (d * d).sum(-1) < rl * rl
        b, p, q = torch.nonzero(ok, as_tuple=True)
        out.append(torch.stack([own[b, p], cand[b, q]]))
    i, j = torch.cat(out, 1)
    keep = i != j
    i, j = i[keep], j[keep]
    o = torch.argsort(i, stable=True)
    return i[o], j[o]


def _as_poly(t):
    return ((((1.061405429 * t - 1.453152027) * t + 1.421413741) * t - 0.284496736) * t + 0.254829592) * t


def _screen(r, alpha):
    """E(r) = erfc(alpha r) by Abramowitz and Stegun 7.1.26 and A(r) = E + 2 alpha r exp(-alpha^2 r^2) / sqrt(pi)."""
    if not torch.is_tensor(r):
        e, a = _screen(torch.tensor(float(r), dtype=torch.float64), alpha)
        return float(e), float(a)
    ex = torch.exp(-(alpha * r) ** 2)
    e = _as_poly(1.0 / (1.0 + 0.3275911 * alpha * r)) * ex
    return e, e + 2.0 * alpha / math.sqrt(math.pi) * r * ex


class _Forces:
    """Forces, energies and virial of replicas that share a force field, FP64, on the GPU."""

    def __init__(self, systems, x, pad=1.5):
        s0 = systems[0]
        dev = x.device
        f64 = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=dev)   # noqa: E731
        self.sys, self.ff, self.x, self.pad = systems, s0.ff, x, pad
        self.box = f64([s.box for s in systems])                      # (R, 3)
        self.rep = torch.repeat_interleave(torch.arange(len(systems), device=dev), torch.tensor([s.n for s in systems], device=dev))
        self.q = f64(np.concatenate([s.charge for s in systems]))
        self.type = torch.as_tensor(np.concatenate([s.type for s in systems]).astype(np.int64), device=dev)
        self.m = f64(np.concatenate([1e4 * s.mass for s in systems]))
        self.lj1, self.lj2 = f64(self.ff.lj1), f64(self.ff.lj2)
        self.rc = float(np.float32(self.ff.rc))
        self.coul = self.ff.coulomb if bool((self.q != 0).any()) else S.COUL_NONE
        self.excl = [f64(0)] * 0
        if len(s0.rigid) or len(s0.bonds):
            self.excl = torch.full((s0.n, 4), -1, dtype=torch.long, device=dev)
            pr = [s0.bonds[:, :2]] if len(s0.bonds) else [s0.rigid[:, [0, 1]], s0.rigid[:, [0, 2]], s0.rigid[:, [1, 2]]]
            pr = np.concatenate(pr).astype(np.int64)
            pr = np.concatenate([pr, pr[:, ::-1]])
            pr = pr[np.argsort(pr[:, 0], kind="stable")]
            slot = np.arange(len(pr)) - np.searchsorted(pr[:, 0], pr[:, 0])
            self.excl[torch.as_tensor(pr[:, 0], device=dev), torch.as_tensor(slot, device=dev)] = torch.as_tensor(pr[:, 1].copy(), device=dev)
        self.bonds = torch.as_tensor(s0.bonds.astype(np.int64), device=dev)
        self.angles = torch.as_tensor(s0.angles.astype(np.int64), device=dev)
        self.pme = s0.pme
        self.build()

    def build(self):
        self.x0, at, ii, jj = self.x.clone(), 0, [], []
        for r, s in enumerate(self.sys):
            i, j = _near(self.wrapped(self.x[at:at + s.n], self.box[r]), self.box[r], self.rc + self.pad)
            ii.append(i + at)
            jj.append(j + at)
            at += s.n
        i, j = torch.cat(ii), torch.cat(jj)
        count = torch.bincount(i, minlength=at)
        first = torch.cumsum(count, 0) - count
        self.nbr = torch.arange(at, device=i.device)[:, None].repeat(1, int(count.max()))   # itself: no neighbor
        self.nbr[i, torch.arange(i.numel(), device=i.device) - first[i]] = j
        if len(self.excl):
            bad = (self.nbr[:, :, None] == self.excl[:, None]).any(-1)
            self.nbr = torch.where(bad, torch.arange(at, device=i.device)[:, None], self.nbr)

    @staticmethod
    def wrapped(x, box):
        return x - box * torch.trunc(2.0 * x / box)

    def pairs(self, a, b, lj1=None, lj2=None, qs=1.0, energy=False):
        """Pair forces on atoms a..b (and their energies and virial, each pair half)."""
        x, nbr, rc = self.x, self.nbr[a:b], self.rc
        box = self.box[self.rep[a:b]][:, None]
        d = x[a:b, None] - x[nbr]
        d = d - box * torch.round(d / box)
        r2 = (d * d).sum(-1)
        on = (r2 <= float(np.float32(rc) * np.float32(rc))) & (nbr != torch.arange(a, b, device=x.device)[:, None])
        r2 = torch.where(on, r2, torch.ones_like(r2))
        lj1, lj2 = self.lj1 if lj1 is None else lj1, self.lj2 if lj2 is None else lj2
        ti, tj = self.type[a:b, None], self.type[nbr]
        i2 = 1.0 / r2
        i6 = i2 ** 3
        f = (lj1[ti, tj] * i6 - lj2[ti, tj]) * i6 * i2
        qq = 0.0
        if self.coul != S.COUL_NONE:
            qq = self.ff.qfac * (qs * qs) * self.q[a:b, None] * self.q[nbr]
            r = torch.sqrt(r2)
            if self.coul == S.COUL_RF:
                k = 2.0 * (self.ff.eps_rf - 1.0) / (2.0 * self.ff.eps_rf + 1.0) / rc ** 3
                f = f + qq * (1.0 / r - k * r2) * i2
                u = 1.0 / r + 0.5 * k * r2 - (1.0 / rc + 0.5 * k * rc * rc)
            else:
                e, big = _screen(r, self.ff.alpha)
                ec, ac = _screen(rc, self.ff.alpha) if self.coul == S.COUL_WOLF else (0.0, 0.0)
                f = f + qq * (big / r - ac / rc) * i2
                u = e / r - ec / rc + ac / rc * torch.log(r / rc) if energy else None
        f = torch.where(on, f, torch.zeros_like(f))
        F = (f[..., None] * d).sum(1)
        if not energy:
            return F
        c6 = rc ** -6
        ulj = (lj1[ti, tj] / 12.0 * i6 - lj2[ti, tj] / 6.0) * i6 - (lj1[ti, tj] / 12.0 * c6 - lj2[ti, tj] / 6.0) * c6
        uc = qq * u if self.coul != S.COUL_NONE else torch.zeros_like(ulj)
        half = [0.5 * torch.where(on, v, torch.zeros_like(v)).sum() for v in (ulj, uc, f * r2)]
        return F, half

    def __call__(self, energy=False):
        n = self.x.shape[0]
        if float((self.x - self.x0).norm(dim=1).max()) > 0.45 * self.pad:
            self.build()
        step = max(1, 24_000_000 // self.nbr.shape[1])
        F, tot = torch.empty_like(self.x), [0.0, 0.0, 0.0]
        for a in range(0, n, step):
            b = min(n, a + step)
            if energy:
                F[a:b], h = self.pairs(a, b, energy=True)
                tot = [t + v for t, v in zip(tot, h)]
            else:
                F[a:b] = self.pairs(a, b)
        if len(self.bonds) or len(self.angles):
            F += self.bonded()
        if self.pme:
            F += self.recip()
        return (F, tot) if energy else F

    def bonded(self):
        """-grad of the harmonic bond and angle energies k (x - x0)^2."""
        x = self.x.detach().requires_grad_()
        box = self.box[0]

        def vec(i, j):
            d = x[i] - x[j]
            return d - box * torch.round(d.detach() / box)
        u = 0.0
        if len(self.bonds):
            r = vec(self.bonds[:, 0], self.bonds[:, 1]).norm(dim=1)
            u = u + (self.ff.bond_k[0] * (r - self.ff.bond_r0[0]) ** 2).sum()
        if len(self.angles):
            p, o = vec(self.angles[:, 0], self.angles[:, 1]), vec(self.angles[:, 2], self.angles[:, 1])
            c = (p * o).sum(1) / (p.norm(dim=1) * o.norm(dim=1))
            u = u + (self.ff.angle_k[0] * (torch.acos(c) - self.ff.angle_t0[0]) ** 2).sum()
        return -torch.autograd.grad(u, x)[0]

    def splines(self, p, w):
        """M_p(w + j) and its derivative, j = 0..p-1."""
        a = [w, 1.0 - w]
        for k in range(2, p):
            z = torch.zeros_like(w)
            lo, hi = a + [z], [z] + a
            if k == p - 1:
                der = [u - v for u, v in zip(lo, hi)]
            a = [((w + j) * lo[j] + (k + 1 - w - j) * hi[j]) / k for j in range(k + 1)]
        return torch.stack(a, 1), torch.stack(der, 1)

    def recip(self):
        """The reciprocal part (smooth PME) and the correction of the excluded pairs."""
        K, p, beta, box, x, q = self.pme[:3], self.pme[3], self.ff.alpha, self.box[0], self.x, self.q
        dev, j = x.device, torch.arange(p, device=x.device)
        k, t, dt, b = [], [], [], []
        for a in range(3):
            u = (x[:, a] / box[a] + 0.5) * K[a]
            fl = torch.floor(u)
            k.append((fl.long()[:, None] - j) % K[a])
            th, dth = self.splines(p, u - fl)
            t.append(th)
            dt.append(dth)
            m4 = self.splines(p, torch.zeros(1, dtype=torch.float64, device=dev))[0][0]
            ph = 2.0 * math.pi / K[a] * torch.arange(K[a], device=dev, dtype=torch.float64)[:, None] * torch.arange(p - 1, device=dev)
            b.append(1.0 / (torch.cos(ph).matmul(m4[1:]) ** 2 + torch.sin(ph).matmul(m4[1:]) ** 2))
        at = ((k[0][:, :, None, None] * K[1] + k[1][:, None, :, None]) * K[2] + k[2][:, None, None, :])
        Q = torch.zeros(K[0] * K[1] * K[2], dtype=torch.float64, device=dev)
        wt = lambda u, v, w: u[:, :, None, None] * v[:, None, :, None] * w[:, None, None, :]   # noqa: E731
        Q.index_add_(0, at.reshape(-1), (q[:, None, None, None] * wt(*t)).reshape(-1))
        m = [torch.fft.fftfreq(K[a], 1.0 / K[a], device=dev, dtype=torch.float64) / box[a] for a in range(3)]
        m[2], b[2] = m[2][:K[2] // 2 + 1].abs(), b[2][:K[2] // 2 + 1]
        mm = m[0][:, None, None] ** 2 + m[1][:, None] ** 2 + m[2] ** 2
        mm[0, 0, 0] = 1.0
        C = self.ff.qfac * torch.exp(-(math.pi / beta) ** 2 * mm) / (math.pi * box.prod() * mm)
        C = C * b[0][:, None, None] * b[1][:, None] * b[2]
        C[0, 0, 0] = 0.0
        phi = torch.fft.irfftn(torch.fft.rfftn(Q.reshape(*K)) * C, s=K) * Q.numel()
        ph = phi.reshape(-1)[at]
        g = [(ph * wt(*[dt[c] if c == a else t[c] for c in range(3)])).sum((1, 2, 3)) * K[a] / box[a] for a in range(3)]
        F = -q[:, None] * torch.stack(g, 1)
        if len(self.excl):
            on = self.excl >= 0
            o = self.excl.clamp(min=0)
            d = x[:, None] - x[o]
            d = d - box * torch.round(d / box)
            r = torch.where(on, d.norm(dim=2), torch.ones_like(d[..., 0]))
            qq = torch.where(on, self.ff.qfac * q[:, None] * q[o], torch.zeros_like(r))
            fr = qq * (2.0 * beta / math.sqrt(math.pi) * torch.exp(-(beta * r) ** 2) / r - torch.erf(beta * r) / r ** 2) / r
            F += (fr[..., None] * d).sum(1)
        return F


def _shake(s, x0, x1, box):
    """x1 moved onto the rigid geometry of the molecules of s along the old bonds (to 1e-14)."""
    mol = torch.as_tensor(s.rigid.astype(np.int64), device=x0.device)
    im = torch.as_tensor(1.0 / s.mass[s.rigid[0]], device=x0.device)
    mi = lambda d: d - box * torch.round(d / box)   # noqa: E731
    old = [mi(x0[mol[:, a]] - x0[mol[:, 0]]) for a in range(3)]
    new = [mi(x1[mol[:, a]] - x1[mol[:, 0]]) for a in range(3)]
    ini = [v.clone() for v in new]
    for _ in range(200):
        worst = 0.0
        for a, b, d in ((0, 1, s.rigid_d[0]), (0, 2, s.rigid_d[0]), (1, 2, s.rigid_d[1])):
            v, r = new[a] - new[b], old[a] - old[b]
            diff = d * d - (v * v).sum(1)
            g = diff / (2.0 * (v * r).sum(1) * (im[a] + im[b]))
            new[a] = new[a] + (g * im[a])[:, None] * r
            new[b] = new[b] - (g * im[b])[:, None] * r
            worst = max(worst, float(diff.abs().max()) / (d * d))
        if worst < 1e-14:
            break
    x1 = x1.clone()
    for a in range(3):
        x1[mol[:, a]] += new[a] - ini[a]
    return x1


def _trajectory(systems, steps):
    """Positions (wrapped), velocities, forces and boxes after `steps` steps from the systems' states."""
    s0 = systems[0]
    cuda = lambda a: torch.as_tensor(np.concatenate(a).astype(np.float64), device="cuda")   # noqa: E731
    fo = _Forces(systems, cuda([s.pos for s in systems]), pad=2.0 if s0.name.startswith("water") else 1.0)
    v, m, R = cuda([s.vel for s in systems]), fo.m[:, None], len(systems)
    nf = torch.tensor([float(s.nf()) for s in systems], dtype=torch.float64, device="cuda")
    T0 = torch.tensor([s.T0 for s in systems], dtype=torch.float64, device="cuda")
    dt, tau, kb = s0.dt, s0.tau, S.KB_REF
    ke2 = lambda u: torch.zeros(R, dtype=torch.float64, device="cuda").index_add_(0, fo.rep, (m * u * u).sum(1))   # noqa: E731
    if s0.integrator == "vverlet":
        kT, xi, vxi = kb * T0, torch.zeros_like(T0), torch.zeros_like(T0)
        Q = nf * kT * tau * tau

        def half(K, xi, vxi):   # Nose-Hoover chain of one, half a step
            vxi = vxi + 0.25 * dt * (2.0 * K - nf * kT) / Q
            s = torch.exp(-0.5 * dt * vxi)
            K, xi = K * s * s, xi + 0.5 * dt * vxi
            return s, xi, vxi + 0.25 * dt * (2.0 * K - nf * kT) / Q
        nose = s0.thermostat == "nosehoover"
        F = fo()
        for _ in range(steps):
            if nose:
                sc, xi, vxi = half(0.5 * ke2(v), xi, vxi)
                v = v * sc[fo.rep][:, None]
            v = v + 0.5 * dt * F / m
            fo.x = fo.x + dt * v
            F = fo()
            v = v + 0.5 * dt * F / m
            if nose:
                sc, xi, vxi = half(0.5 * ke2(v), xi, vxi)
                v = v * sc[fo.rep][:, None]
    else:
        lam = torch.ones_like(T0)
        for _ in range(steps):
            F = fo(energy=s0.barostat != "none")
            F, tot = F if s0.barostat != "none" else (F, None)
            v = (v + dt * F / m) * lam[fo.rep][:, None]
            x = fo.x + dt * v
            if len(s0.rigid):
                x = _shake(s0, fo.x, x, fo.box[0])
                v = (x - fo.x) / dt
            k2 = ke2(v)
            if s0.thermostat == "berendsen":
                lam = torch.sqrt(1.0 + dt / tau * (T0 / (k2 / (nf * kb)) - 1.0))
            if tot is not None:
                P = (k2 + tot[2]) / (3.0 * fo.box.prod(1)) * 16605.390671738467
                mu = (1.0 - s0.compress * dt / s0.tau_p * (s0.P0 - P)) ** (1.0 / 3.0)
                x, fo.box = x * mu[fo.rep][:, None], fo.box * mu[:, None]
            fo.x = x
    return fo.wrapped(fo.x, fo.box[fo.rep]), v, F, fo.box


def exact(case, seed):
    if case["kind"] == "fm":
        base, frames, targets, theta = _fm_problem(case, seed)
        th = torch.tensor(theta, dtype=torch.float64, device="cuda", requires_grad=True)
        nt, M, loss = base.ff.ntype, 3.0 * frames.shape[0] * base.n, 0.0
        iu, k = np.triu_indices(nt), nt * (nt + 1) // 2
        where = np.zeros((nt, nt), np.int64)
        where[iu] = where[iu[::-1]] = np.arange(k)
        for x, t in zip(frames, targets):
            E, G = th[:k][where], th[k:2 * k][where]
            fo = _Forces([base], torch.as_tensor(x, dtype=torch.float64, device="cuda"), pad=0.01)
            F = fo.pairs(0, base.n, 48.0 * E * G ** 12, 24.0 * E * G ** 6, th[2 * k])
            part = ((F - torch.as_tensor(t, dtype=torch.float64, device="cuda")) ** 2).sum() / M
            part.backward()
            loss += float(part.detach())
        return {"loss": torch.tensor(loss, dtype=torch.float64), "grad": th.grad}
    sys_ = _systems(case, seed)
    if case["kind"] == "forces":
        F, tot = _Forces(sys_, torch.as_tensor(sys_[0].pos, dtype=torch.float64, device="cuda"))(energy=True)
        en = torch.zeros(1, 4, dtype=torch.float64)
        en[0, 0], en[0, 1] = float(tot[0]), float(tot[1])
        return {"force": F, "energy": en, "virial": torch.tensor([float(tot[2])], dtype=torch.float64)}
    x, v, F, box = _trajectory(sys_, case["steps"])
    out = {"pos": x, "vel": v, "force": F}
    if case["kind"] == "npt":
        out["box"] = box
    return out
