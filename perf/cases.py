"""Work that users of the library have it do, through its public entry points.

  fit    Fitness.compute: the fitness of a population over a training set, what
         every generation of a fitting job calls
  ga     Fitness.run_ga: whole generations with the population on the device,
         what a fitting job runs
  force  Fitness.find_force: per-atom force, virial and energy of one parameter
         set (labels, predictions)

over the potentials and set sizes of the benchmark (bench.py), of the served mix
(gpuga_amd/synth.py) and of the bundled reference jobs (tests/golden).  exact()
restates the formulas in 64 bits with torch.
"""
import math

import numpy as np
import torch

import gpuga_amd
from gpuga_amd import synth

# Minimal Tersoff bounds: one species, and two (tests/golden/si_type2's ranges).
ONE = (synth.TERSOFF_SI_MIN, synth.TERSOFF_SI_MAX)
TWO = (np.array([3.0, 1.3, 2.2, 1.8, 3.0, 1.3, 2.2, 1.8, 0.6, 0.2, -1.0, 2.7, 3.0], np.float32),
       np.array([3.2, 1.5, 2.3, 2.2, 3.2, 1.5, 2.3, 2.2, 0.9, 0.8, -0.5, 2.7, 3.0], np.float32))


def listed():
    return [
        # the smallest benchmark workload: a launch that cannot fill the GPU
        dict(name="fit_tersoff_small", kind="fit", pot="tersoff", P=50, Nc=60, rep=2, cutoff=3.0,
             force=0.2),
        # the benchmark's default: cells of 8 to 512 atoms, 20% with forces
        dict(name="fit_tersoff_mixed", kind="fit", pot="tersoff", P=200, Nc=1000, rep=0,
             cutoff=3.0, force=0.2),
        # a binary semiconductor (two species, 13 parameters), as tests/golden/gaas:
        # 217 cells, few of them with forces
        dict(name="fit_tersoff_binary", kind="fit", pot="tersoff2", P=200, Nc=217, rep=2,
             cutoff=3.2, force=0.02),
        # an outer radius past the second shell: up to 16 neighbours an atom
        dict(name="fit_tersoff_shells", kind="fit", pot="tersoff", P=100, Nc=100, rep=2,
             cutoff=4.0, force=0.2),
        # the rigid-ion benchmark: 96-atom oxide cells, about 95 neighbours
        dict(name="fit_ri", kind="fit", pot="ri", P=200, Nc=500, force=0.2),
        # an oxide job of the size of tests/golden/hfo2, a population of no round size
        dict(name="fit_ri_small", kind="fit", pot="ri", P=77, Nc=100, force=0.01),
        # the neural pair potential's benchmark
        dict(name="fit_nn2b", kind="fit", pot="nn2b", P=256, Nc=800, n=32, bf16=1, force=0.2),
        # a neural dimer curve, as tests/golden/nn2b: 402 cells of two atoms
        dict(name="fit_nn2b_dimers", kind="fit", pot="dimer", P=200, Nc=402, n=10, bf16=1,
             force=0.5),
        # the network with the species pair as an input, its layers in FP32
        dict(name="fit_nn2b_species", kind="fit", pot="species", P=100, Nc=150, n=20, bf16=0,
             force=0.2),
        # generations of a small job, back to back on the device
        dict(name="ga_tersoff", kind="ga", pot="tersoff", P=50, Nc=60, rep=2, cutoff=3.0,
             force=0.2, generations=10),
        # labels of the benchmark's default set
        dict(name="force_tersoff", kind="force", pot="tersoff", Nc=1000, rep=0, cutoff=3.0,
             force=0.2),
        # labels of a set of the neural pair potential
        dict(name="force_nn2b", kind="force", pot="nn2b", Nc=400, n=32, bf16=1, force=0.2),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["fit", "fit", "fit", "fit", "ga", "force"])
    pot = "tersoff" if kind == "ga" else rng.choice(
        ["tersoff", "tersoff", "tersoff2", "ri", "ri", "nn2b", "nn2b", "dimer", "species"])
    c = dict(kind=kind, pot=pot, force=rng.choice([0.01, 0.1, 0.2, 0.5]))
    if kind != "force":
        c["P"] = 2 * log(20, 60) if kind == "ga" else log(16, 250)
    if kind == "ga":
        c["generations"] = rng.randint(2, 10)
    if pot in ("tersoff", "tersoff2"):
        c["Nc"] = log(20, 60) if kind == "ga" else log(30, 400)
        c["rep"] = 2 if kind == "ga" else rng.choice([0, 2])
        c["cutoff"] = rng.choice([3.0, 3.2, 4.0]) if c["rep"] == 2 and c["Nc"] <= 100 else 3.1
    elif pot == "ri":
        c["Nc"] = log(20, 400)
    else:
        c["Nc"] = log(100, 500) if pot == "dimer" else log(30, 500)
        c["n"] = rng.choice([6, 10, 16, 20, 32])
        c["bf16"] = rng.randint(0, 1)
    return c


# ------------------------------------------------------------------ inputs

def _structures(c, seed):
    """The training set without labels, and a ground-truth parameter set."""
    pot, Nc = c["pot"], c["Nc"]
    if pot in ("tersoff", "tersoff2"):
        # the cells' sizes are the case's; strain and displacements are the seed's
        d = synth.tersoff_si(Nc=Nc, sizes="fixed" if c["rep"] else "loguniform",
                             reps=(c["rep"],) * 3, force_fraction=c["force"], strain=0.0,
                             disp=0.0, seed=2)
        rng = np.random.default_rng(seed)
        axis = 1 + rng.uniform(-0.03, 0.03, (Nc, 3))
        r = d["r"].reshape(3, -1) * np.repeat(axis, d["Na"], axis=0).T
        d["r"] = (r + rng.normal(0, 0.1, r.shape)).astype(np.float32).reshape(-1)
        d["box"] = (d["box"].reshape(Nc, 3, 3) * axis[:, :, None]).astype(np.float32).reshape(-1)
        lo, hi = (a.copy() for a in (ONE if pot == "tersoff" else TWO))
        truth = d["truth"].copy() if pot == "tersoff" else (0.5 * (lo + hi)).astype(np.float32)
        if c["cutoff"] > 3.5:  # the taper ends at the list's cut-off
            lo[-2], hi[-2] = c["cutoff"] - 1.0, c["cutoff"] - 0.6
            lo[-1] = hi[-1] = c["cutoff"]
            truth[-2:] = c["cutoff"] - 0.8, c["cutoff"]
        if pot == "tersoff2":  # zinc blende
            d["type"] = np.tile(np.repeat(np.arange(2, dtype=np.int32), 4), len(d["type"]) // 8)
            d["potential_type"] = 2
        d.update(cutoff=c["cutoff"], pmin=lo, pmax=hi, truth=truth)
    elif pot == "ri":
        d = synth.fluorite_ab2(Nc=Nc, force_fraction=c["force"], seed=seed)
    elif pot == "dimer":
        rng = np.random.default_rng(seed)
        n, ncf = c["n"], max(1, min(Nc - 1, round(Nc * c["force"])))
        r = np.zeros((3, 2 * Nc), np.float32)
        axis = rng.normal(size=(3, Nc))
        r[:, 1::2] = rng.uniform(1.2, 8.0, Nc) * axis / np.linalg.norm(axis, axis=0)
        d = dict(potential_type=3, num_neurons=n, cutoff=8.0, weights=(0.9, 0.1, 0.0),
                 Na=np.full(Nc, 2, np.int32), type=np.zeros(2 * Nc, np.int32), Nc_force=ncf,
                 box=np.tile(np.diag([30.0] * 3).reshape(-1), Nc).astype(np.float32),
                 r=r.reshape(-1), truth=synth.nn2b_truth(n))
    else:
        d = synth.wurtzite_ab(Nc=Nc, n=c["n"], force_fraction=c["force"], seed=seed,
                              species=pot == "species")
    if pot in ("dimer", "nn2b", "species"):
        V = len(d["truth"])
        d.update(pmin=np.full(V, -3, np.float32), pmax=np.full(V, 3, np.float32))
    return d


def _labelled(c, seed):
    """Labels of the ground truth, off by a few percent as a potential is from
    the calculations that it is fitted to."""
    d = _structures(c, seed)
    f, w, e = _Model(d).outputs(d["truth"])
    m = _Model.config_sums(d, w, e)
    rng = np.random.default_rng(seed + 1)

    def noisy(a):
        a = a.cpu().numpy()
        return (a + 0.03 * a.std() * rng.normal(size=a.shape)).astype(np.float32).reshape(-1)

    d["force_ref"], d["virial_ref"], d["pe_ref"] = noisy(f), noisy(m[1:]), noisy(m[0])
    return d


def _population(c, d, seed):
    """Every gene in [0, 1] as in the first generation for half of the individuals,
    the others near the ground truth as a fit that has converged."""
    rng = np.random.default_rng(seed + 2)
    g = rng.random((c["P"], len(d["pmin"])), dtype=np.float32)
    span = np.where(d["pmax"] > d["pmin"], d["pmax"] - d["pmin"], 1.0)
    best = np.clip((d["truth"] - d["pmin"]) / span, 0, 1)
    g[1::2] = np.clip(best + rng.normal(0, 0.05, g[1::2].shape), 0, 1)
    return g


def prepare(case, seed):
    """The resident training set, with its launch shape tuned for the population as
    a fitting job's first generation does, and the genes."""
    d = _labelled(case, seed) if case["kind"] != "force" else _structures(case, seed)
    fit = gpuga_amd.Fitness(arrays=d, nn2b_bf16=case.get("bf16", 1))
    s = dict(kind=case["kind"], fit=fit)
    if case["kind"] == "force":
        s["params"] = d["truth"]
        return s
    fit.autotune(case["P"])
    if case["kind"] == "fit":
        s["genes"] = _population(case, d, seed)
    else:
        s.update(P=case["P"], seed=seed, generations=case["generations"])
    return s


def run(state):
    fit = state["fit"]
    if state["kind"] == "fit":
        return fit.compute(state["genes"])
    if state["kind"] == "force":
        return fit.find_force(state["params"])
    P = state["P"]
    parents = P // 2 + P // 2 % 2  # children come in pairs
    ga = gpuga_amd.GA(P, parents, fit.V, maximum_generation=1000, mutation_rate=0.2,
                      seed=state["seed"])
    best, elite = fit.run_ga(ga, 0, state["generations"])
    return best, elite, ga.population


def _neighbours(c):
    if c["pot"] in ("tersoff", "tersoff2"):
        return 4 if c["cutoff"] < 3.5 else 14
    return {"ri": 95, "dimer": 0.9}.get(c["pot"], 42)


def work(case):
    """Positions, types, references and genes in, results out; arithmetic by the
    per-unit counts of bench.py."""
    c, m = case, _neighbours(case)
    N = c["Nc"] * (2 if c["pot"] == "dimer" else 96 if c["pot"] == "ri" else
                   (64 if c["rep"] else 120) if "tersoff" in c["pot"] else 72)
    n = c.get("n", 0)
    V = {"tersoff": 9, "tersoff2": 13, "ri": 15}.get(c["pot"], n * (n + 4) + 1)
    geometry = 16.0 * N + 64.0 * c["Nc"]
    if "tersoff" in c["pot"]:
        per = 106.0 * m + 57.0 * m * (m - 1)
    elif c["pot"] == "ri":
        per = m * (24.0 * c["force"] + 20.0 * (1 - c["force"]))
    else:
        per = m * (24.0 * c["force"] + 18.0 * (1 - c["force"]))
    if c["kind"] == "force":
        if n:  # the network once per unordered pair
            per = 0.5 * m * (4.0 * n * n + 20.0 * n)
        return dict(bytes=geometry + 40.0 * N + 4.0 * V, flops=per * N)
    G, P = c.get("generations", 1), c["P"]
    table = 1024 * (6.0 * n * n + 23.0 * n)
    return dict(bytes=G * (geometry + 12.0 * N * c["force"] + 28.0 * c["Nc"] + 4.0 * P * (V + 1)),
                flops=G * P * (per * N + table))


# ------------------------------------------------------------- 64-bit forms

class _Model:
    """The potentials over one training set in FP64 (the reference's
    src/minimal_tersoff.cu, src/ri.cu, src/nn2b.cu, by formula)."""

    def __init__(self, d):
        dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        f64 = dict(dtype=torch.float64, device=dev)
        self.type = d["potential_type"]
        self.n = d.get("num_neurons", 0)
        Na = np.asarray(d["Na"])
        self.N = int(Na.sum())
        first = np.concatenate([[0], np.cumsum(Na)])
        r = torch.tensor(np.asarray(d["r"], np.float32).reshape(3, -1).T.copy(), **f64)
        box = torch.tensor(np.asarray(d["box"], np.float32).reshape(-1, 3, 3), **f64)
        own, nbr, vec = [], [], []
        for na in np.unique(Na):
            group = np.flatnonzero(Na == na)
            for cs in np.array_split(group, max(1, len(group) * na * na // 4_000_000)):
                if not len(cs):
                    continue
                at = torch.tensor(first[cs][:, None] + np.arange(na), device=dev)
                x, b = r[at], box[torch.tensor(cs, device=dev)]
                s = (x[:, None] - x[:, :, None]).reshape(len(cs), -1, 3) @ torch.linalg.inv(b)
                v = ((s - s.round()) @ b).reshape(len(cs), na, na, 3)
                near = (v.square().sum(-1) < float(d["cutoff"]) ** 2) & ~torch.eye(
                    int(na), dtype=torch.bool, device=dev)
                q, i, j = near.nonzero(as_tuple=True)
                own.append(at[q, i])
                nbr.append(at[q, j])
                vec.append(v[q, i, j])
        own, nbr, vec = (torch.cat(a) for a in (own, nbr, vec))
        self.own, order = own.sort(stable=True)
        self.nbr, self.vec = nbr[order], vec[order]
        t = torch.tensor(np.asarray(d["type"]), device=dev)
        self.code = t[self.own] + t[self.nbr]
        if self.type in (1, 2):  # bonds padded to a rectangle of atoms x neighbours
            count = torch.bincount(self.own, minlength=self.N)
            self.slot = torch.arange(len(self.own), device=dev) - (count.cumsum(0) - count)[self.own]
            self.M = int(count.max())

    def _tersoff(self, p, vec):
        sets = [p[:4], p[:4] if self.type == 1 else p[4:8]]
        en, beta, h, r1, r2 = p[-5:]
        d = vec.norm(dim=1)
        fr = fa = 0.0
        for k, (D0, alpha, r0, S) in enumerate(sets):
            on = (self.code % 2 == k).to(d) if self.type == 2 else (1.0 if k == 0 else 0.0)
            fr = fr + on * D0 / (S - 1) * torch.exp(-math.sqrt(2 * S) * alpha * (d - r0))
            fa = fa + on * S * D0 / (S - 1) * torch.exp(-math.sqrt(2 / S) * alpha * (d - r0))
        taper = 0.5 + 0.5 * torch.cos(math.pi * (d.clamp(r1, r2) - r1) / (r2 - r1))
        fc = torch.where(d < r1, 1.0, torch.where(d < r2, taper, 0.0))

        def padded(x):
            return x.new_zeros((self.N, self.M) + x.shape[1:]).index_put((self.own, self.slot), x)

        u = padded(vec / d[:, None])
        g = beta * (u @ u.transpose(1, 2) - h) ** 2
        fcp = padded(fc)
        zeta = (g @ fcp[:, :, None])[..., 0] - g.diagonal(dim1=1, dim2=2) * fcp
        zeta = zeta[self.own, self.slot].clamp_min(1e-16)
        b = (1 + zeta ** en) ** (-0.5 / en)
        return 0.5 * fc * (fr - b * fa)

    def _ri(self, p, vec):
        d = vec.norm(dim=1)
        q2, kc, alpha, rc = p[0] ** 2, float(np.float32(14.399645)), 0.2, p[10]
        e = math.erfc(alpha * rc)
        v_rc = e / rc
        dv_rc = -e / rc ** 2 - 2 * alpha / math.sqrt(math.pi) * math.exp(-(alpha * rc) ** 2) / rc
        pick = [torch.tensor(x, dtype=d.dtype, device=d.device)[self.code.long()] for x in (
            p[1:10:3], p[2:10:3], p[3:10:3], [q2 * kc, -0.5 * q2 * kc, 0.25 * q2 * kc])]
        U = pick[0] * torch.exp(-d / pick[1]) - pick[2] * d ** -6
        U = U + pick[3] * (torch.erfc(alpha * d) / d - v_rc - dv_rc * (d - rc))
        D0, a, r0, S = p[11:15]
        morse = D0 / (S - 1) * (torch.exp(-math.sqrt(2 * S) * a * (d - r0))
                                - S * torch.exp(-math.sqrt(2 / S) * a * (d - r0)))
        return 0.5 * (U + torch.where(self.code == 1, morse, 0.0))

    def _nn2b(self, p):
        n, d = self.n, self.vec.norm(dim=1)
        p = torch.tensor(p, dtype=d.dtype, device=d.device)
        w0, b0, w1, b1, w2 = p[:n], p[n:2 * n], p[2 * n:n * (n + 2)], p[n * (n + 2):n * (n + 3)], \
            p[n * (n + 3):n * (n + 4)]
        x = d[:, None] * w0 - b0
        if self.type == 4:
            x = x + self.code[:, None] * p[n * (n + 4) + 1:]
        x = x.tanh()
        y = (1 - x * x) * w0
        w1 = w1.reshape(n, n).T
        x2 = (x @ w1 - b1).tanh()
        U = x2 @ w2 - p[n * (n + 4)]
        dU = ((1 - x2 * x2) * (y @ w1)) @ w2
        a = math.pi * (d.clamp(7.0, 8.0) - 7.0)  # the reference's fixed taper and its force
        fc = 0.5 + 0.5 * torch.cos(a)
        fcp = -0.5 * math.pi * torch.sin(a) * ((d >= 7.0) & (d < 8.0))
        U = U * fc
        return 0.5 * U, 0.5 * ((dU * fc + U * fcp) / d)[:, None] * self.vec

    def outputs(self, params):
        """Per-atom force [3][N], virial [6][N] and energy [N]."""
        p = [float(x) for x in np.asarray(params, np.float32)]
        if self.type >= 3:
            e, g = self._nn2b(p)
        else:
            vec = self.vec.clone().requires_grad_(True)
            e = self._ri(p, vec) if self.type == 0 else self._tersoff(p, vec)
            g, = torch.autograd.grad(e.sum(), vec)
            e = e.detach()
        zero = e.new_zeros(self.N)
        f = torch.stack([zero.index_add(0, self.own, g[:, k]).index_add(0, self.nbr, -g[:, k])
                         for k in range(3)])
        w = []
        for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (2, 0)):
            t = -0.5 * self.vec[:, a] * g[:, b]
            w.append(zero.index_add(0, self.own, t).index_add(0, self.nbr, t))
        return f, torch.stack(w), zero.index_add(0, self.own, e)

    @staticmethod
    def config_sums(d, w, e):
        c = torch.repeat_interleave(torch.tensor(np.asarray(d["Na"]), device=e.device))
        return e.new_zeros(7, len(d["Na"])).index_add(1, c, torch.cat([e[None], w]))


def _denormalised(d, genes):
    lo, hi = (np.asarray(d[k], np.float32) for k in ("pmin", "pmax"))
    return lo + ((hi - lo) * genes).astype(np.float32)


def exact(case, seed):
    if case["kind"] == "ga":  # a selection by rank has no 64-bit value to compare with
        return None
    if case["kind"] == "force":
        d = _structures(case, seed)
        return [a.reshape(-1) for a in _Model(d).outputs(d["truth"])]
    d = _labelled(case, seed)
    model, ncf = _Model(d), d["Nc_force"]
    dev = model.vec.device
    Nf = int(np.sum(d["Na"][:ncf]))
    ref = [torch.tensor(np.asarray(d[k]), dtype=torch.float64, device=dev)
           for k in ("force_ref", "virial_ref", "pe_ref")]
    fr, wr, er = ref[0].reshape(3, -1)[:, :Nf], ref[1].reshape(6, -1)[:, ncf:], ref[2][ncf:]
    wf, we, wv = (float(np.float32(x)) for x in d["weights"])
    scale_e = (er - er.min().clamp_max(0)).square().sum()
    fitness = []
    for p in _denormalised(d, _population(case, d, seed)):
        f, w, e = model.outputs(p)
        m = _Model.config_sums(d, w, e)[:, ncf:]
        fitness.append(we * ((m[0] - er).square().sum() / scale_e).sqrt()
                       + wv * ((m[1:] - wr).square().sum() / wr.square().sum()).sqrt()
                       + wf * ((f[:, :Nf] - fr).square().sum() / fr.square().sum()).sqrt())
    return torch.stack(fitness)
