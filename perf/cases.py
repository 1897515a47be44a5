"""Measured cases: molecular-dynamics runs of bead-spring systems.

A case is a set of one or more systems that one call of ``Engine.step``
advances, after which the program reads them ("do"): a production run between
two outputs, the whole state of each ("state") or a trajectory frame of each
("frame": positions); or "forces", an evaluation of the current positions.  ``beads_lo`` / ``beads_hi`` and ``len_lo`` /
``len_hi`` bound the log-uniform bead counts and chain lengths of the systems
(equal bounds: one fixed size), ``ensemble`` is the integrator ("mixed":
Langevin, NVT and NPT in turn), ``steps`` the length of the run, ``thermo`` and
``stress`` the intervals of its records, and ``model`` the force field:

  kg     Kremer-Grest chains: LJ cut at 2.5, FENE + WCA bonds, harmonic angles
  blend  chains of two species with their own LJ parameters and masses
  table  chains of two species whose cross interaction is tabulated

The systems start from melts that plain torch operations relax here, from the
seed alone: random walks at the case's density, pushed apart by a soft
repulsion, then a short Brownian run with the bonds, angles and cores of the
force field, repeated periodically for the larger ones, with Maxwell
velocities.
"""
import math
import random

import numpy as np
import torch

DT, RC, SKIN = 0.001, 2.5, 0.3
FENE = (30.0, 1.5, 1.0, 1.0)          # k, R0, epsilon, sigma
ANGLE = (5.0, math.pi)                # k, theta0
MODELS = {  # LJ (epsilon, sigma) of each type pair, masses
    "kg": ([1.0, 1.0], [1.0]),
    "blend": ([1.0, 1.0, 0.75, 1.05, 0.75, 1.05, 0.5, 1.1], [1.0, 2.0]),
    "table": ([1.0, 1.0, 0.0, 0.0, 0.0, 0.0, 1.0, 1.0], [1.0, 1.0]),
}
ENSEMBLES = ("langevin", "nvt", "npt")
TABLE_POINTS, TABLE_LO = 2000, 0.5


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(name, systems, beads, length, ensemble="langevin", model="kg", rho=0.85, steps=40, thermo=0, stress=0,
          do="state"):
    lo, hi = (beads, beads) if isinstance(beads, int) else beads
    llo, lhi = (length, length) if isinstance(length, int) else length
    c = {"name": name} if name else {}
    c.update(do=do, systems=systems, beads_lo=lo, beads_hi=hi, len_lo=llo, len_hi=lhi, ensemble=ensemble,
             model=model, rho=rho, steps=steps, thermo=thermo, stress=stress)
    return c


def listed():
    return [
        # a small melt of a parameter scan, one system at a time
        _case("melt_2k", 1, 2000, 20),
        # stress autocorrelation (viscosity) of an odd-sized melt of long chains
        _case("stress_7k", 1, 7400, 185, ensemble="nvt", thermo=10, stress=1),
        # the bead-spring benchmark size, Langevin, at melt density
        _case("melt_30k", 1, 30000, 100),
        # the Nose-Hoover benchmark system: density 0.70
        _case("nvt_30k", 1, 30000, 100, ensemble="nvt", rho=0.7, thermo=20),
        _case("npt_30k", 1, 30000, 100, ensemble="npt", rho=0.7, thermo=20),
        # forces, energy and virial of a configuration (force dumps, analysis)
        _case("forces_30k", 1, 30000, 100, do="forces"),
        # two species with their own LJ parameters and masses; and tabulated
        _case("blend_12k", 1, 12000, 50, model="blend", thermo=20),
        _case("table_9k", 1, 9000, 60, model="table", thermo=20),
        # one system above 65,536 slots
        _case("npt_120k", 1, 120000, 75, ensemble="npt", thermo=20),
        # the large single melt: a run between two trajectory frames
        _case("melt_1m", 1, 1000000, 100, steps=100, do="frame"),
        # many small jobs of all ensembles in one batch
        _case("jobs_48", 48, (1000, 6000), (10, 100), ensemble="mixed", thermo=20),
        # the batched workload: uneven replicas at different points of their
        # runs, a frame of each
        _case("uneven_128", 128, (2000, 64000), (20, 200), steps=100, do="frame"),
    ]


def draw(rng):
    lu = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    kind = rng.random()
    model = rng.choice(("kg", "kg", "kg", "blend", "table"))
    ens = rng.choice(ENSEMBLES)
    rho = round(rng.uniform(0.65, 0.88), 3)
    thermo = rng.choice((0, 10, 20))
    if kind < 0.5:    # one system of the whole range
        length = lu(10, 200)
        n = max(1, lu(1000, 900000) // length) * length
        n = max(n, 1000 // length * length + length)
        big = n > 200000
        c = _case("", 1, n, length, ens, model, rho, 100 if big else rng.randint(20, 40), thermo,
                  rng.choice((0, 0, 2)), "frame" if big else "state")
    elif kind < 0.8:  # a batch
        hi = lu(4000, 64000)
        c = _case("", lu(4, 110), (max(1000, hi // rng.randint(2, 30)), hi), (lu(10, 30), lu(40, 200)),
                  rng.choice(("langevin", "mixed")), "kg", rho, rng.randint(40, 100), thermo, do="frame")
    else:
        length = lu(10, 200)
        n = max(1, lu(1000, 200000) // length) * length
        c = _case("", 1, max(n, 1000 // length * length + length), length, "langevin", model, rho, do="forces")
    return c


# ---------------------------------------------------------------------------
# starting configurations
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _specs(case, rng):
    """Chains, chain length, repeats per axis, temperature and ensemble of each
    system; the sizes follow from the case, temperatures and noise from `rng`."""
    sizes = random.Random("%s %s %s" % (case["systems"], case["beads_lo"], case["beads_hi"]))
    out = []
    for k in range(case["systems"]):
        u, w = sizes.random(), sizes.random()
        length = int(round(math.exp(math.log(case["len_lo"]) + u * math.log(case["len_hi"] / case["len_lo"]))))
        beads = math.exp(math.log(case["beads_lo"]) + w * math.log(case["beads_hi"] / case["beads_lo"]))
        # repeats of a relaxed block per axis: blocks of a few thousand beads
        # for the larger systems of a batch, of tens of thousands alone
        base = 2000.0 if case["systems"] > 1 else 30000.0
        m = max(1, int(round((beads / base) ** (1.0 / 3.0))))
        chains = max(1, int(round(beads / length)))
        while m > 1 and (chains % m ** 3 and case["systems"] == 1 or beads / m ** 3 < 900):
            m -= 1
        block = max(1, int(round(chains / m ** 3)))
        while block * length < 900:
            block += 1
        ens = ENSEMBLES[k % 3] if case["ensemble"] == "mixed" else case["ensemble"]
        T = 1.0 if case["systems"] == 1 else float(np.float32(rng.uniform(0.8, 1.2)))
        out.append({"block": block, "len": length, "m": m, "T": T, "ens": ens, "seed": 1000 + rng.randrange(1 << 30)})
    return out


def _wrap(d, L):
    return d - L * torch.round(d / L)


def _relax(specs, rho, gen, dev):
    """Unwrapped bead positions of every system's block, concatenated, and the offsets."""
    off, per = [0], []
    for s in specs:
        off.append(off[-1] + s["block"] * s["len"])
        per.append((s["block"] * s["len"] / rho) ** (1.0 / 3.0))
    n = off[-1]
    cnt = torch.tensor([b - a for a, b in zip(off, off[1:])], device=dev)
    sysid = torch.repeat_interleave(torch.arange(len(specs), device=dev), cnt)
    Lb = torch.tensor(per, device=dev, dtype=torch.float32)[sysid]
    length = torch.tensor([s["len"] for s in specs], device=dev)[sysid]
    first = torch.tensor(off[:-1], device=dev)[sysid]
    place = (torch.arange(n, device=dev) - first) % length  # place along the chain
    has = {k: (place >= -k) if k < 0 else (place < length - k) for k in (-2, -1, 1, 2)}
    # random walks of persistent bonds (about eight): exponential averages of
    # random vectors, scaled to the bond length and summed along each chain
    step = torch.randn(n, 3, device=dev, generator=gen)
    past = torch.cat([step[-63:], step]) if n > 63 else torch.cat([torch.randn(63, 3, device=dev, generator=gen), step])
    step = sum(math.exp(-k / 8.0) * past[63 - k:len(past) - k] for k in range(64))
    step = 0.97 * step / step.norm(dim=1, keepdim=True)
    step = torch.where((place == 0)[:, None], torch.rand(n, 3, device=dev, generator=gen) * Lb[:, None], step)
    run = torch.cumsum(step.double(), 0)
    start = torch.arange(n, device=dev) - place
    x = (run - (run - step.double())[start]).float()
    nc = torch.clamp((Lb / 1.4).long(), min=1)
    ncs = torch.tensor([max(1, int(float(np.float32(v)) / 1.4)) for v in per], device=dev) ** 3
    base = (torch.cumsum(ncs, 0) - ncs)[sysid]
    total, cap, rows = int(ncs.sum()), 12, 24
    shifts = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
    L1 = Lb[:, None]
    me = torch.arange(n, device=dev)

    def rowsof(x):
        """The nearest `rows` non-bonded beads of each bead (itself where there are fewer)."""
        w = x - L1 * torch.floor(x / L1)
        c = torch.minimum((w / L1 * nc[:, None]).long(), nc[:, None] - 1)
        key = base + (c[:, 0] * nc + c[:, 1]) * nc + c[:, 2]
        key, order = torch.sort(key, stable=True)
        begin = torch.searchsorted(key, torch.arange(total, device=dev))
        rank = me - begin[key]
        table = torch.full((total, cap), -1, device=dev, dtype=torch.long)
        keep = rank < cap
        table[key[keep], rank[keep]] = order[keep]
        got = []
        for part in torch.split(me, 200000):
            cc, k1 = c[part], nc[part]
            cand = torch.cat([table[base[part] + (((cc[:, 0] + a) % k1) * k1 + (cc[:, 1] + b) % k1) * k1 + (cc[:, 2] + d) % k1]
                              for a, b, d in shifts], 1)
            r2 = _wrap(w[part][:, None, :] - w[cand.clamp(min=0)], L1[part][:, None]).square().sum(-1)
            r2 = torch.where((cand < 0) | (cand == part[:, None]), torch.inf, r2)
            r2 = torch.where(((cand == part[:, None] + 1) & has[1][part][:, None]) | ((cand == part[:, None] - 1) & has[-1][part][:, None]),
                             torch.inf, r2)
            near, at = torch.topk(r2, rows, 1, largest=False)
            got.append(torch.where(near < 2.6, cand.gather(1, at), part[:, None]))
        return torch.cat(got)

    def along(x, k):
        return torch.where(has[k][:, None], torch.roll(x, -k, 0) - x, 0.0)

    def force(x, nb, soft):
        d = _wrap(x[:, None, :] - x[nb], L1[:, None])
        r2 = d.square().sum(-1)
        other = (nb != me[:, None]) & (r2 > 1e-8)
        if soft:
            r = torch.sqrt(r2.clamp(min=1e-6))
            f = torch.where(other & (r < 1.12), soft * (1.0 - r / 1.12) / r, 0.0)
        else:
            i6 = r2.clamp(min=0.3).reciprocal() ** 3
            f = torch.where(other & (r2 < 1.2599), 24.0 * i6 * (2.0 * i6 - 1.0) / r2.clamp(min=0.3), 0.0)
        F = (f[..., None] * d).sum(1)
        for k in (1, -1):  # bonds
            b = along(x, k)
            r2 = b.square().sum(1, keepdim=True).clamp(0.25, 2.1)
            i6 = r2.reciprocal() ** 3
            g = FENE[0] / (1.0 - r2 / FENE[1] ** 2) - torch.where(r2 < 1.2599, 24.0 * i6 * (2.0 * i6 - 1.0) / r2, 0.0)
            F = F + torch.where(has[k][:, None], g.clamp(-1000, 1000) * b, 0.0)
        # stiffness: a weak force that straightens consecutive bonds
        bend = torch.where((has[1] & has[-1])[:, None], along(x, 1) + along(x, -1), 0.0)
        return F + 4.0 * ANGLE[0] * (bend - 0.5 * torch.where(has[1][:, None], torch.roll(bend, -1, 0), 0.0)
                               - 0.5 * torch.where(has[-1][:, None], torch.roll(bend, 1, 0), 0.0))

    for it in range(240):
        if it % 8 == 0:
            nb = rowsof(x)
        F = 0.002 * force(x, nb, 25.0 + it)
        x = x + F * (0.06 / F.norm(dim=1, keepdim=True).clamp(min=0.06))
    for it in range(200):
        if it % 8 == 0:
            nb = rowsof(x)
        F = 2e-4 * force(x, nb, 0.0)
        F = F * (0.05 / F.norm(dim=1, keepdim=True).clamp(min=0.05))
        x = x + F + (0.02 if it < 185 else 0.008) * torch.randn(n, 3, device=dev, generator=gen)
    return x.double().cpu().numpy(), off, per


def _systems(case, seed):
    """Every system of the case as host arrays."""
    specs = _specs(case, random.Random(seed))
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    x, off, per = _relax(specs, case["rho"], gen, dev)
    lj, masses = MODELS[case["model"]]
    nr = np.random.default_rng(seed)
    out = []
    for k, s in enumerate(specs):
        b, m, length = x[off[k]:off[k + 1]], s["m"], s["len"]
        cells = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        full = (cells[:, None, :] * per[k] + b[None]).reshape(-1, 3)
        n = len(full)
        L = np.float32(m * per[k])
        image = np.floor(full / float(L))
        pos = (full - image * float(L)).astype(np.float32)
        over = pos >= L
        pos[over] = 0.0
        image = image.astype(np.int32) + over
        chain = np.arange(n) // length
        types = (chain % len(masses)).astype(np.int32)
        mass = np.asarray(masses, np.float32)[types]
        vel = nr.standard_normal((n, 3)) * np.sqrt(s["T"] / mass)[:, None]
        vel -= (vel * mass[:, None]).sum(0) / mass.sum()
        i = np.arange(n, dtype=np.int32)
        inner = i[i % length != length - 1]
        mid = i[i % length < length - 2]
        pos4 = np.concatenate([pos, types.view(np.float32)[:, None]], 1)
        out.append(dict(s, n=n, L=L, pos4=pos4, vel=vel.astype(np.float32), image=image.astype(np.int32), types=types,
                        mol=chain.astype(np.int32) + 1, bonds=np.stack([inner, inner + 1], 1),
                        angles=np.stack([mid, mid + 1, mid + 2, np.zeros_like(mid)], 1)))
        # where in its run the system is when the pass begins: replicas of a batch
        # were not all created at once
        out[-1]["before"] = k % 20 if case["systems"] > 1 and case["ensemble"] != "mixed" else 0
    return out


def _table():
    """A tabulated 9-6 pair: r, energy, force / r."""
    r = np.linspace(TABLE_LO, RC, TABLE_POINTS)
    s3 = (1.12 / r) ** 3
    return np.stack([r, s3 * s3 * (2.0 * s3 - 3.0), 18.0 * s3 * s3 * (s3 - 1.0) / r ** 2], 1).astype(np.float32)


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    import fastmd_amd as fmd
    systems = _systems(case, seed)
    lj, masses = MODELS[case["model"]]
    eng = fmd.Engine(0)
    sids, groups = [], {}
    for s in systems:
        d = fmd.Desc(s["pos4"], s["L"], lj, ntypes=len(masses), vel=s["vel"], image=s["image"], mol=s["mol"],
                     bonds=s["bonds"], bond_params=[FENE], angles=s["angles"], angle_params=[ANGLE], masses=masses,
                     rc=RC, skin=SKIN, dt=DT, ensemble=ENSEMBLES.index(s["ens"]), T=(s["T"], s["T"]),
                     Tdamp=1.0, P=(1.0, 1.0), Pdamp=1.0, chain=3, seed=s["seed"], nsteps=100000,
                     thermo_freq=case["thermo"], stress_freq=case["stress"],
                     tables=([-1, 0, 0, -1], [(TABLE_LO, RC, _table())]) if case["model"] == "table" else None)
        sids.append(eng.add(d))
        groups.setdefault(s["before"], []).append(sids[-1])
    for before, ids in groups.items():
        if before:
            eng.step(ids, before)
    return {"case": case, "engine": eng, "sids": sids, "n": [s["n"] for s in systems]}


def _thermo_row(t):
    return [t["ke"], t["pe"], t["temp"], *t["press"], t["L"]]


def run(state):
    case, eng, sids = state["case"], state["engine"], state["sids"]
    if case["do"] == "forces":
        f, vir, pe = eng.forces(sids[0])
        return {"force": f, "virial": vir.astype(np.float32), "pe": pe}
    eng.step(sids, case["steps"])
    total, frame = sum(state["n"]), case["do"] == "frame"
    x, v = torch.empty(total, 3), torch.empty(0 if frame else total, 3)
    rows, at = [], 0
    for sid, n in zip(sids, state["n"]):
        p, vel, image = eng.state(sid)
        # unwrapped positions, as mean square displacements need them
        torch.add(torch.from_numpy(p)[:, :3], torch.from_numpy(image), alpha=eng.state_box(sid), out=x[at:at + n])
        if not frame:
            v[at:at + n] = torch.from_numpy(vel)
        at += n
        if case["thermo"]:
            rows += [_thermo_row(t) for t in eng.drain_thermo(sid)[0]]
        rows.append(_thermo_row(eng.thermo(sid)))
    out = {"position": x, "thermo": np.array(rows, np.float32)}
    if not frame:
        out["velocity"] = v
    if case["stress"]:
        c, count = eng.corr(sids[0])
        out["corr"], out["count"] = c.astype(np.float32), count
    return out


def work(case):
    """Positions and velocities read and written each step, the pairs inside the
    cutoff once each (44 operations), bonds and angles."""
    lo, hi = case["beads_lo"], case["beads_hi"]
    n = case["systems"] * (lo if hi == lo else (hi - lo) / math.log(hi / lo))
    pairs = n * 0.5 * case["rho"] * 4.0 / 3.0 * math.pi * RC ** 3
    steps = 1 if case["do"] == "forces" else case["steps"]
    per_bead = 12 + 16 if case["do"] == "forces" else 48
    return {"bytes": steps * per_bead * n, "flops": steps * (44.0 * pairs + 150.0 * n)}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _half_list(x, L, reach):
    """Index pairs i < j within `reach` in a periodic box of side L (x wrapped)."""
    n, dev = len(x), x.device
    nc = int(L / reach)
    if nc < 3:
        i, j = torch.triu_indices(n, n, 1, device=dev)
        near = _wrap(x[i] - x[j], L).square().sum(1) < reach * reach
        return i[near], j[near]
    c = (x / L * nc).long().clamp(0, nc - 1)
    key = (c[:, 0] * nc + c[:, 1]) * nc + c[:, 2]
    key, order = torch.sort(key, stable=True)
    begin = torch.searchsorted(key, torch.arange(nc ** 3, device=dev))
    rank = torch.arange(n, device=dev) - begin[key]
    table = torch.full((nc ** 3, int(rank.max()) + 1), -1, device=dev, dtype=torch.long)
    table[key, rank] = order
    I, J = [], []
    for part in torch.split(torch.arange(n, device=dev), 40000):
        cc = c[part]
        for a in (-1, 0, 1):
            cand = torch.cat([table[(((cc[:, 0] + a) % nc) * nc + (cc[:, 1] + b) % nc) * nc + (cc[:, 2] + d) % nc]
                              for b in (-1, 0, 1) for d in (-1, 0, 1)], 1)
            r2 = _wrap(x[part][:, None] - x[cand.clamp(min=0)], L).square().sum(-1)
            k, q = torch.nonzero((cand > part[:, None]) & (r2 < reach * reach), as_tuple=True)
            I.append(part[k])
            J.append(cand[k, q])
    return torch.cat(I), torch.cat(J)


class _Exact:
    """The systems of one group, concatenated, in 64-bit floats."""

    def __init__(self, case, systems):
        self.case, self.dev = case, _device()
        t = lambda a, dt=torch.float64: torch.as_tensor(np.asarray(a), device=self.dev, dtype=dt)  # noqa: E731
        cat = lambda k: np.concatenate([s[k] for s in systems])  # noqa: E731
        self.n = [s["n"] for s in systems]
        off = np.concatenate([[0], np.cumsum(self.n)])
        shift = lambda k, w: np.concatenate([s[k][:, :w] + o for s, o in zip(systems, off)])  # noqa: E731
        self.sys = torch.repeat_interleave(torch.arange(len(systems), device=self.dev), t(self.n, torch.long))
        self.S, self.off = len(systems), off
        self.x, self.v = t(np.concatenate([s["pos4"][:, :3] for s in systems])), t(cat("vel"))
        self.image = t(cat("image"))
        self.types = t(cat("types"), torch.long)
        self.bonds, self.angles = t(shift("bonds", 2), torch.long), t(shift("angles", 3), torch.long)
        lj, masses = MODELS[case["model"]]
        self.nt = len(masses)
        self.lj = t(np.asarray(lj, np.float32)).reshape(-1, 2)
        self.m = t(np.asarray(masses, np.float32))[self.types][:, None]
        self.L = t([s["L"] for s in systems])
        self.gid = torch.arange(len(self.x), device=self.dev) - t(off[:-1], torch.long)[self.sys]
        self.seed = t([s["seed"] for s in systems], torch.long)[self.sys]
        self.T = t([s["T"] for s in systems])
        self.ens = systems[0]["ens"]
        self.dt = float(np.float32(DT))
        self.Nf = 3.0 * t(self.n)
        self.Q1, self.Qr = self.Nf * self.T, self.T.clone()  # Tdamp = 1
        self.W, self.V0 = (self.Nf + 3.0) * self.T, self.L ** 3  # Pdamp = 1
        self.eps, self.veps = torch.zeros_like(self.L), torch.zeros_like(self.L)
        self.xi = [torch.zeros_like(self.L) for _ in range(3)]
        self.table = t(_table())
        self.pending = torch.ones_like(self.L)
        self.age = 0
        self.forces()
        self.carry = self.kinetic()[1]

    def per_system(self, a):
        return torch.stack([a[p:q].sum(0) for p, q in zip(self.off, self.off[1:])])

    def forces(self):
        if self.age % 30 == 0:
            ij = [_half_list(self.x[a:b], float(L), RC + 0.45) for a, b, L in zip(self.off, self.off[1:], self.L)]
            i = torch.cat([p[0] + int(a) for p, a in zip(ij, self.off)])
            j = torch.cat([p[1] + int(a) for p, a in zip(ij, self.off)])
            key = lambda a, b: torch.minimum(a, b) * len(self.x) + torch.maximum(a, b)  # noqa: E731
            free = ~torch.isin(key(i, j), key(self.bonds[:, 0], self.bonds[:, 1]))  # bonded pairs have no LJ
            self.i, self.j = i[free], j[free]
        self.age += 1
        F, vir = torch.zeros_like(self.x), self.x.new_zeros(len(self.x), 6)
        energy = self.x.new_zeros(len(self.x))

        def tensor(f, d):
            return torch.stack([f[:, 0] * d[:, 0], f[:, 0] * d[:, 1], f[:, 0] * d[:, 2], f[:, 1] * d[:, 1],
                                f[:, 1] * d[:, 2], f[:, 2] * d[:, 2]], 1)

        def add(i, j, d, f, e):  # force f on i, -f on j, separation d
            F.index_add_(0, i, f)
            F.index_add_(0, j, -f)
            vir.index_add_(0, i, tensor(f, d))
            energy.index_add_(0, i, 0.5 * e)
            energy.index_add_(0, j, 0.5 * e)

        size = 20_000_000
        for a in range(0, len(self.i), size):
            i, j = self.i[a:a + size], self.j[a:a + size]
            d = _wrap(self.x[i] - self.x[j], self.L[self.sys[i]][:, None])
            r2 = d.square().sum(1)
            near = (r2 < RC * RC) & (r2 > 1e-10)
            i, j, d, r2 = i[near], j[near], d[near], r2[near]
            es = self.lj[self.types[i] * self.nt + self.types[j]]
            s6 = (es[:, 1] ** 2 / r2) ** 3
            f = (24.0 * es[:, 0] * s6 * (2.0 * s6 - 1.0) / r2).clamp(-1000.0, 1000.0)
            e = 4.0 * es[:, 0] * s6 * (s6 - 1.0)
            if self.case["model"] == "table":
                r = torch.sqrt(r2).clamp(TABLE_LO, RC)
                h = (RC - TABLE_LO) / (TABLE_POINTS - 1)
                k = ((r - TABLE_LO) / h).long().clamp(0, TABLE_POINTS - 2)
                w = ((r - TABLE_LO) / h - k)[:, None]
                row = self.table[k] * (1.0 - w) + self.table[k + 1] * w
                cross = self.types[i] != self.types[j]
                e, f = torch.where(cross, row[:, 1], e), torch.where(cross, row[:, 2], f)
            add(i, j, d, f[:, None] * d, e)
        i, j = self.bonds[:, 0], self.bonds[:, 1]
        d = _wrap(self.x[i] - self.x[j], self.L[self.sys[i]][:, None])
        k, R0, eps, sig = FENE
        r2 = d.square().sum(1).clamp(1e-6, R0 * R0 * 0.9999)
        s6 = torch.where(r2 < sig * sig * 2.0 ** (1.0 / 3.0), (sig * sig / r2) ** 3, 0.0)
        f = -k * R0 * R0 / (R0 * R0 - r2) + 24.0 * eps * s6 * (2.0 * s6 - 1.0) / r2
        e = -0.5 * k * R0 * R0 * torch.log(1.0 - r2 / (R0 * R0)) + torch.where(s6 > 0, 4.0 * eps * s6 * (s6 - 1.0) + eps, 0.0)
        add(i, j, d, f[:, None] * d, e)
        if len(self.angles):
            i, c, j = self.angles.unbind(1)
            L = self.L[self.sys[c]][:, None]
            a, b = _wrap(self.x[i] - self.x[c], L), _wrap(self.x[j] - self.x[c], L)
            la, lb = a.norm(dim=1, keepdim=True), b.norm(dim=1, keepdim=True)
            cr = torch.linalg.cross(a, b).norm(dim=1, keepdim=True)
            dot = (a * b).sum(1, keepdim=True)
            cos, dth = dot / (la * lb), torch.atan2(cr, dot) - float(np.float32(ANGLE[1]))
            g = 2.0 * ANGLE[0] * dth / (cr / (la * lb)).clamp(min=1e-6)
            fi, fj = g * (b / (la * lb) - cos * a / la ** 2), g * (a / (la * lb) - cos * b / lb ** 2)
            F.index_add_(0, i, fi)
            F.index_add_(0, j, fj)
            F.index_add_(0, c, -fi - fj)
            e = ANGLE[0] * dth[:, 0] ** 2
            for q in (i, c, j):
                energy.index_add_(0, q, e / 3.0)
            vir.index_add_(0, c, tensor(fi, a) + tensor(fj, b))
        self.F, self.pe, self.vir, self.energy = F, self.per_system(energy), self.per_system(vir), energy

    def kinetic(self):
        v = self.v * self.pending[self.sys][:, None]
        k = self.per_system(self.m * torch.stack([v[:, 0] ** 2, v[:, 0] * v[:, 1], v[:, 0] * v[:, 2], v[:, 1] ** 2,
                                                  v[:, 1] * v[:, 2], v[:, 2] ** 2], 1))
        return k, 0.5 * (k[:, 0] + k[:, 3] + k[:, 5])

    def noise(self, step):
        """Three normals of each bead from Philox4x32-10 keyed by (seed, bead, step)."""
        mask = 0xFFFFFFFF
        full = lambda c: torch.full_like(self.gid, c)  # noqa: E731
        c = [self.gid, full(step & mask), full(step >> 32), full(0x4C414E47)]
        k0, k1 = self.seed & mask, self.seed >> 32

        def product(m, b):  # high and low words of the 64-bit product of two 32-bit numbers
            lo, hi = (m & 0xFFFF) * b, (m >> 16) * b
            mid = hi + (lo >> 16)
            return (mid >> 16) & mask, ((mid & 0xFFFF) << 16) | (lo & 0xFFFF)

        for r in range(10):
            if r:
                k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
            h0, l0 = product(0xD2511F53, c[0])
            h1, l1 = product(0xCD9E8D57, c[2])
            c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        u = [((w >> 8).double() + 0.5) / 16777216.0 for w in c]
        a, b = torch.sqrt(-2.0 * torch.log(u[0])), torch.sqrt(-2.0 * torch.log(u[2]))
        return torch.stack([a * torch.cos(2 * math.pi * u[1]), a * torch.sin(2 * math.pi * u[1]),
                            b * torch.cos(2 * math.pi * u[3])], 1)

    def chain(self, KE):
        """One half-step of the Nose-Hoover chain: the velocity scale."""
        h, M, v = 0.5 * self.dt, 3, self.xi
        d2, d4, d8 = h, 0.5 * h, 0.25 * h
        G = [(2.0 * KE - self.Nf * self.T) / self.Q1, 0.0, 0.0]
        for k in (2, 1):
            e = torch.exp(-d8 * v[k + 1]) if k + 1 < M else 1.0
            v[k] = (v[k] * e + G[k] * d4) * e
        e0 = torch.exp(-d8 * v[1])
        v[0] = (v[0] * e0 + G[0] * d4) * e0
        s = torch.exp(-d2 * v[0])
        G[0] = (2.0 * KE * s * s - self.Nf * self.T) / self.Q1
        v[0] = (v[0] * e0 + G[0] * d4) * e0
        for k in (1, 2):
            e = torch.exp(-d8 * v[k + 1]) if k + 1 < M else 1.0
            G[k] = ((self.Q1 if k == 1 else self.Qr) * v[k - 1] ** 2 - self.T) / self.Qr
            v[k] = (v[k] * e + G[k] * d4) * e
        return s

    def step(self, number):
        h, dt = 0.5 * self.dt, self.dt
        by = lambda s: s[self.sys][:, None]  # noqa: E731
        if self.ens == "langevin":
            self.v = self.v + h / self.m * self.F
            self.x = self.x + h * self.v
            c1 = math.exp(-dt)
            self.v = c1 * self.v + torch.sqrt((1.0 - c1 * c1) * by(self.T) / self.m) * self.noise(number)
            self.x = self.x + h * self.v
        else:
            baro = 1.0
            if self.ens == "npt":
                vw = self.veps / self.W
                baro = torch.exp(-(1.0 + 3.0 / self.Nf) * vw * h)
                self.L = (self.V0 * torch.exp(3.0 * self.eps)) ** (1.0 / 3.0)
            scale = self.pending * self.chain(self.carry * baro ** 2) * baro
            self.v = self.v * by(scale) + h / self.m * self.F
            if self.ens == "npt":
                z = 0.5 * vw * dt
                sinh = torch.where(z.abs() < 1e-6, 1.0 + z * z / 6.0, torch.sinh(z) / z)
                self.x = self.x * by(torch.exp(vw * dt)) + self.v * by(dt * torch.exp(z) * sinh)
            else:
                self.x = self.x + dt * self.v
        k = torch.floor(self.x / by(self.L))
        self.x, self.image = self.x - k * by(self.L), self.image + k
        self.pending = torch.ones_like(self.L)
        self.placed = self.L
        self.forces()
        self.v = self.v + h / self.m * self.F
        if self.ens != "langevin":
            K, KE = self.kinetic()
            baro = 1.0
            if self.ens == "npt":
                V = self.V0 * torch.exp(3.0 * self.eps)
                P = (2.0 * KE + self.vir[:, 0] + self.vir[:, 3] + self.vir[:, 5]) / (3.0 * V)
                cb = 2.0 ** (1.0 / 3.0)
                for w in (1.0 / (2.0 - cb), -cb / (2.0 - cb), 1.0 / (2.0 - cb)):
                    half = self.veps + 1.5 * V * (P - 1.0) * w * dt
                    self.eps = self.eps + half * w * dt / self.W
                    self.veps = self.veps + 3.0 * self.V0 * torch.exp(3.0 * self.eps) * (P - 1.0) * w * dt
                baro = torch.exp(-(1.0 + 3.0 / self.Nf) * self.veps / self.W * h)
                self.L = (self.V0 * torch.exp(3.0 * self.eps)) ** (1.0 / 3.0)
            s = self.chain(KE * baro ** 2)
            self.pending = s * baro
            self.carry = KE * self.pending ** 2

    def row(self, s):
        K, KE = self.kinetic()
        n, V = self.n[s], float(self.L[s]) ** 3
        ke = float(KE[s]) / n
        return [ke, float(self.pe[s]) / n, 2.0 * ke / 3.0, *[float(p) / V for p in K[s] + self.vir[s]], float(self.L[s])]


def _correlate(samples):
    """Multiple-tau sums and counts of a list of six-component samples."""
    corr, count = np.zeros((16, 16, 6)), np.zeros((16, 16), np.int64)
    for level in range(16):
        for t, x in enumerate(samples):
            for lag in range(t % 16 + 1):
                corr[level, lag] += x * samples[t - lag]
                count[level, lag] += 1
        samples = [np.mean(samples[k:k + 16], 0) for k in range(0, len(samples) - 15, 16)]
    return corr, count


def exact(case, seed):
    if case["systems"] * case["beads_hi"] * case["steps"] > 200000000:
        return None  # minutes
    systems = _systems(case, seed)
    if case["do"] == "forces":
        g = _Exact(case, systems)
        return {"force": torch.cat([g.F, g.energy[:, None]], 1), "virial": g.vir[0], "pe": float(g.pe[0])}
    groups = {}
    for k, s in enumerate(systems):
        groups.setdefault((s["before"], s["ens"]), []).append(k)
    x, v, rows = [None] * len(systems), [None] * len(systems), [[] for _ in systems]
    corr = None
    for (before, ens), ids in groups.items():
        g, samples = _Exact(case, [systems[k] for k in ids]), []
        for number in range(1, before + case["steps"] + 1):
            g.step(number)
            if case["thermo"] and number % case["thermo"] == 0:
                for q, k in enumerate(ids):
                    rows[k].append(g.row(q))
            if case["stress"] and number % case["stress"] == 0:
                samples.append(np.array(g.row(0)[3:9]))
        for q, k in enumerate(ids):
            a, b = g.off[q], g.off[q + 1]
            x[k] = g.x[a:b] + g.image[a:b] * g.placed[q]
            v[k] = g.v[a:b] * g.pending[q]
            rows[k].append(g.row(q))
        if case["stress"]:
            corr = _correlate(samples)
    out = {"position": torch.cat(x), "thermo": np.array([r for s in rows for r in s])}
    if case["do"] == "state":
        out["velocity"] = torch.cat(v)
    if corr is not None:
        out["corr"], out["count"] = corr[0], corr[1]
    return out
