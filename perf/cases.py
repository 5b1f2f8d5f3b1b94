"""The work a program built on remd_amd has it do, as measurable cases.

Five kinds of call, each through the package's public entry points:

interval  one REMD job: exchange intervals with the exchange on the device
          between them (execute_intervals), then the checkpoint that a run
          writes every few intervals
batch     several jobs of unequal size advanced together (Batch), with the
          host exchange and new conditions after every interval
serve     a short stream of jobs through the server: admission (creation,
          wall tables, first forces), batched intervals, exchange, retirement
forces    one force evaluation of a job (neighbour build, pair and wall
          forces, torques, energies) and the download of the states
wall      the nanotube wall table that every confined job starts from

Water models, cutoffs, wall parameters, densities, ladders and the sizes of
the named workloads are those of remd_amd.inputs.  Starting configurations
are molecules on a lattice inside the accessible region, relaxed by a short
rigid-body descent in plain torch, with thermal momenta per replica: a start
that a 2 fs step integrates, made from the seed alone.
"""
import math

import numpy as np
import torch

import remd_amd as ra
from remd_amd import inputs, serve

RC, RL, MARGIN = 9.0, 8.0, 0.5
MODELS = ("TIP3P", "TIP4P", "TIP5P")
PERIODIC = {0: (True, True, True), 1: (False, False, True), 2: (True, True, False)}
SGM_WALL, EPS_WALL, RHO_WALL, NFWALL = 3.277, 0.3886, 0.38016, 1000
# pressure ladder (Pa); the TIP5P of inputs.MOLTYPE binds weakly and boils
# under the barostat at ordinary pressures
PRESSURE = {"TIP3P": (0.1e6, 150e6), "TIP4P": (0.1e6, 150e6), "TIP5P": (400e6, 800e6)}
# FLOP of one ordered molecule pair inside the cutoff, FMA = 2 (one LJ site
# term 32, each Coulomb site term 27, 38 per pair)
PAIR_FLOPS = {"TIP3P": 313, "TIP4P": 313, "TIP5P": 502}
STATE_DOUBLES = 21  # r, v, f (3 each), q, p, n (4 each) per molecule


# ------------------------------------------------------------------- the list
def _job(confined, model, nmol, ntemp, npress, size=0.0, length=0.0, barostat=True):
    """One job's part of a case.  size: tube radius or slit width (A);
    length: tube length or lateral box (A), 0 = from the density."""
    return dict(confined=confined, model=model, nmol=nmol, ntemp=ntemp, npress=npress, size=size, length=length,
                barostat=barostat)


def listed():
    return [
        # the smallest call: forces of a two-replica job, where the launch,
        # the copies and the synchronisation are most of the time
        dict(name="forces-small-tube", kind="forces", precision=0, **_job(1, "TIP3P", 96, 2, 1, 7.0, 36.0)),
        # forces of a mid-size slit job in both directions of a restart or an
        # analysis run: neighbour build, forces, torques, energies, download
        dict(name="forces-slit", kind="forces", precision=0, **_job(2, "TIP4P", 797, 8, 1, 12.0)),
        # the flagship: 64 replicas of 144 TIP4P in a nanotube, 16 T x 4 P
        dict(name="tube144-tip4p-64rep", kind="interval", precision=0, intervals=4, steps=100,
             **_job(1, "TIP4P", 144, 16, 4, 7.0, 50.0)),
        # plain REMD of bulk water as a workstation user runs it: few
        # replicas, FP64 pair math, thermostat only
        dict(name="bulk256-tip4p-fp64", kind="interval", precision=1, intervals=2, steps=100,
             **_job(0, "TIP4P", 256, 4, 1, barostat=False)),
        # the nano-slit precision study's two runs: mixed and FP64 pair math
        dict(name="slit512-tip5p-128rep", kind="interval", precision=0, intervals=2, steps=100,
             **_job(2, "TIP5P", 512, 32, 4, 10.0, 40.0)),
        dict(name="slit512-tip5p-fp64", kind="interval", precision=1, intervals=1, steps=100,
             **_job(2, "TIP5P", 512, 32, 4, 10.0, 40.0)),
        # large replicas of the served stream: a bulk and a slit job whose
        # states exceed one workgroup's LDS, and a bulk job of its largest size
        dict(name="bulk1820-tip4p-16rep", kind="interval", precision=0, intervals=1, steps=100,
             **_job(0, "TIP4P", 1820, 16, 1)),
        dict(name="slit1374-tip5p-64rep", kind="interval", precision=0, intervals=1, steps=100,
             **_job(2, "TIP5P", 1374, 64, 1, 14.0)),
        dict(name="bulk2048-tip4p-8rep", kind="interval", precision=0, intervals=1, steps=100,
             **_job(0, "TIP4P", 2048, 8, 1)),
        # eight unequal tubes of two models, 32 replicas each, in one batch
        dict(name="uneven-tubes-256rep", kind="batch", precision=0, intervals=2, steps=100, first=5, jobs=8, ntemp=8,
             npress=4),
        # the served stream's life of a job, from admission to result, for
        # six jobs of all models and confinements
        dict(name="served-6jobs", kind="serve", precision=0, intervals=2, steps=100, jobs=6, lo=64, hi=640, reps=16),
        # the wall table of every new confined job
        dict(name="wall-tube-1000", kind="wall", nfwall=NFWALL, size=7.0),
    ]


def draw(rng):
    """One more case of the same kinds and ranges (nmol 64-2048, 2-128
    replicas, tubes of radius 5-15 A, slits 8-20 A wide)."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["interval", "interval", "interval", "forces", "batch", "serve", "wall"])
    if kind == "wall":
        return dict(kind=kind, nfwall=log_int(200, 4000), size=round(rng.uniform(5.0, 15.0), 3))
    if kind == "batch":
        return dict(kind=kind, precision=0, intervals=1, steps=100, first=rng.randint(5, 8), jobs=rng.randint(2, 5),
                    ntemp=rng.choice([3, 4, 8]), npress=rng.choice([1, 2, 4]))
    if kind == "serve":
        return dict(kind=kind, precision=0, intervals=rng.randint(1, 3), steps=100, jobs=rng.randint(2, 6), lo=64,
                    hi=log_int(200, 640), reps=rng.choice([8, 12, 16]))
    confined = rng.randrange(3)
    precision = rng.choice([0, 0, 0, 1])
    nmol = log_int(235 if confined == 0 else 64, 2048 if precision == 0 else 700)
    # the replicas that keep the pass below the largest listed one
    most = max(2, min(128, int(60000 / nmol)))
    size = {0: 0.0, 1: round(rng.uniform(5.0, 15.0), 2), 2: round(rng.uniform(8.0, 20.0), 2)}[confined]
    job = _job(confined, rng.choice(MODELS), nmol, log_int(2, most), 1, size)
    if kind == "forces":
        job["ntemp"] = min(16, job["ntemp"])
        return dict(kind=kind, precision=precision, **job)
    return dict(kind=kind, precision=precision, intervals=rng.randint(1, 2) if nmol < 700 else 1,
                steps=100 if nmol < 1000 else 50, **job)


# ------------------------------------------------------------- configurations
def _geometry(job):
    """(box, accessible height or radius) in A at 1 g/cm^3 of the accessible
    volume, boxes a little above the two cutoffs at least."""
    n, size, length = job["nmol"], job["size"], job["length"]
    if job["confined"] == 0:
        L = max((n * 29.9) ** (1.0 / 3.0), 2 * (RC + MARGIN) + 0.15)
        return (L, L, L), 0.0
    if job["confined"] == 1:
        Lz = length or max(n * 29.9 / (math.pi * (size - 1.7) ** 2), 2 * (RC + MARGIN) + 1.0)
        Lxy = 2.0 * (size + 9.0) + 4.0
        return (Lxy, Lxy, Lz), size - 2.8
    Lxy = length or max(math.sqrt(n * 29.9 / (size - 3.4)), 2 * (RC + MARGIN) + 1.0)
    return (Lxy, Lxy, size + 40.0), 0.5 * size - 2.6


def _lattice(job, rng):
    """nmol centred positions (A): the widest lattice that holds them, sites
    chosen at random."""
    box, acc = _geometry(job)
    n, conf = job["nmol"], job["confined"]

    def periodic(L, a):
        k = max(1, int(L / a))
        return (np.arange(k) + 0.5) * (L / k) - 0.5 * L

    def inside(h, a, even):
        k = int(2 * h / a) + 1
        if (k % 2 == 0) != even:
            k -= 1
        return (np.arange(k) - 0.5 * (k - 1)) * a if k > 0 else np.zeros(0)

    for a in np.arange(3.3, 1.9, -0.02):
        best = None
        for even in (False, True):
            if conf == 0:
                ax = [periodic(L, a) for L in box]
            elif conf == 1:
                ax = [inside(acc, a, even), inside(acc, a, even), periodic(box[2], a)]
            else:
                ax = [periodic(box[0], a), periodic(box[1], a), inside(acc, a, even)]
            x = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
            if conf == 1:
                x = x[x[:, 0] ** 2 + x[:, 1] ** 2 <= acc * acc + 1e-9]
            if best is None or len(x) > len(best):
                best = x
        if len(best) >= n:
            return best[np.sort(rng.permutation(len(best))[:n])], box, acc
    raise ValueError("no lattice holds %d molecules" % n)


def _rotate(q, b):
    """Space-frame vectors of body vectors b (S, 3) for quaternions q (N, 4)."""
    a0, a1, a2, a3 = q.unbind(-1)
    m = torch.stack([
        torch.stack([a0 * a0 + a1 * a1 - a2 * a2 - a3 * a3, 2 * (a1 * a2 - a0 * a3), 2 * (a1 * a3 + a0 * a2)], -1),
        torch.stack([2 * (a1 * a2 + a0 * a3), a0 * a0 - a1 * a1 + a2 * a2 - a3 * a3, 2 * (a2 * a3 - a0 * a1)], -1),
        torch.stack([2 * (a1 * a3 - a0 * a2), 2 * (a2 * a3 + a0 * a1), a0 * a0 - a1 * a1 - a2 * a2 + a3 * a3], -1),
    ], -2)
    return (m.unsqueeze(-3) * b.view(*([1] * (q.dim() - 1)), -1, 1, 3)).sum(-1), m


def _relaxed(job, rng, steps=200):
    """Rigid-body descent of one configuration: every molecule moves down the
    gradient of its energy with its 40 nearest neighbours held fixed."""
    x0, box, acc = _lattice(job, rng)
    mt = inputs.molecule(job["model"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f8 = dict(dtype=torch.float64, device=dev)
    x = torch.tensor(x0, **f8)
    q = torch.tensor(inputs.random_quaternions(rng, len(x0)), **f8)
    L = torch.tensor([b if p else 1e9 for b, p in zip(box, PERIODIC[job["confined"]])], **f8)
    body = torch.tensor(mt.r, **f8)
    qq = torch.tensor(np.outer(mt.q, mt.q), **f8)
    sig2, eps4 = float(mt.sigma[0]) ** 2, 4.0 * float(mt.eps[0])
    idx = None
    for it in range(steps):
        if it % 20 == 0:
            d = x[:, None] - x[None]
            d2 = (d - L * torch.round(d / L)).square().sum(-1)
            d2.fill_diagonal_(1e9)
            idx = d2.topk(min(40, len(x0) - 1), largest=False).indices
        sites = _rotate(q, body)[0]
        xi, qi = x.clone().requires_grad_(), q.clone().requires_grad_()
        si = _rotate(qi / qi.norm(dim=-1, keepdim=True), body)[0]
        g = xi[:, None] - x[idx]
        g = g - L * torch.round(g.detach() / L)
        d = g[:, :, None, None] + si[:, None, :, None] - sites[idx][:, :, None]
        r2 = d.square().sum(-1) + 0.1
        s6 = (sig2 / r2[:, :, 0, 0]) ** 3
        e = (eps4 * s6 * (s6 - 1)).sum() + (qq / r2.sqrt()).sum()
        if job["confined"] == 1:
            e = e + 50.0 * (xi[:, :2].norm(dim=-1) - acc).clamp_min(0).square().sum()
        elif job["confined"] == 2:
            e = e + 50.0 * (xi[:, 2].abs() - acc).clamp_min(0).square().sum()
        gx, gq = torch.autograd.grad(e, (xi, qi))
        fade = 1.0 - it / steps
        x = x - gx * (torch.clamp(0.08 * fade / gx.norm(dim=-1, keepdim=True).clamp_min(1e-9), max=0.001))
        q = q - gq * (torch.clamp(0.10 * fade / gq.norm(dim=-1, keepdim=True).clamp_min(1e-9), max=0.002))
        q = q / q.norm(dim=-1, keepdim=True)
    return x.cpu().numpy(), q.cpu().numpy(), box, mt


def _system(job, seed, steps=100):
    """The inputs.System of a job: one relaxed configuration, jittered and
    given thermal momenta at each replica's temperature."""
    rng = np.random.RandomState(seed % (1 << 31))
    x, q, box, mt = _relaxed(job, rng)
    T, P = inputs.make_ladder(job["ntemp"], job["npress"], inputs.geometric(240.0, 340.0, job["ntemp"]),
                              inputs.geometric(*PRESSURE[job["model"]], job["npress"]))
    conf = job["confined"]
    s = inputs.System(job["model"], job["nmol"], 1, (1, 2, 3)[conf] if job["barostat"] else 0, conf, 2.0, RC, RL, steps,
                      job["ntemp"], job["npress"], T, P)
    if conf:
        s.wall_length, s.nfwall = job["size"], NFWALL
        s.sgm_wall, s.eps_wall, s.rho_wall = SGM_WALL, EPS_WALL, RHO_WALL
    L = np.asarray(box)
    for t in T:
        r = np.mod((x + rng.normal(0.0, 0.02, x.shape)) / L + 0.5, 1.0)
        v, p = inputs.thermal_momenta(rng, mt, q, t, L)
        s.states.append(inputs.ReplicaState(r=r, v=v, q=q.copy(), p=p, L=tuple(L),
                                            ids=np.arange(job["nmol"], dtype=np.int32)))
    return s


def _batch_jobs(case):
    """The tubes of a batch: radii first, first + 1, ... A, 40 A long, TIP3P
    and TIP4P in turn."""
    out = []
    for k in range(case["jobs"]):
        R = float(case["first"] + k)
        nmol = int(round(math.pi * (R - 1.7) ** 2 * 40.0 / 29.9))
        out.append(_job(1, MODELS[k % 2], nmol, case["ntemp"], case["npress"], R, 40.0))
    return out


def _serve_jobs(case):
    """The jobs of a served stream: nmol over the logarithm of lo-hi, the
    confinements and the models in turn, replicas halved on larger jobs."""
    out = []
    for k in range(case["jobs"]):
        t = k / max(1, case["jobs"] - 1)
        nmol = int(round(case["lo"] * (case["hi"] / case["lo"]) ** t))
        conf = (1, 2, 0)[k % 3]
        nmol = max(nmol, 235) if conf == 0 else nmol
        out.append(_job(conf, MODELS[(k + k // 3) % 3], nmol, max(2, case["reps"] // (1 if nmol < 256 else 2)), 1,
                        (0.0, 6.0 + 0.9 * k, 9.0 + k)[conf]))
    return out


# ------------------------------------------------------------ prepare and run
class _Conditions:
    """What the exchange keeps for a job: the slot of each replica, its
    conditions and the rand() stream."""

    def __init__(self, system):
        self.T, self.P = system.T.copy(), system.P.copy()
        self.index = np.arange(system.nreplica, dtype=np.int32)
        self.rng = ra.GlibcRand(1)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "wall":
        R = case["size"] + 1e-3 * np.random.RandomState(seed % (1 << 31)).random_sample()
        return dict(case=case, R=R)
    if kind == "batch":
        systems = [_system(j, seed + 7919 * k, case["steps"]) for k, j in enumerate(_batch_jobs(case))]
        jobs = [ra.REMDGPU(s, precision=case["precision"]) for s in systems]
        batch = ra.Batch()
        for j in jobs:
            batch.add(j)
        return dict(case=case, systems=systems, jobs=jobs, batch=batch, cond=[_Conditions(s) for s in systems], step=0)
    if kind == "serve":
        systems = [_system(j, seed + 7919 * k, case["steps"]) for k, j in enumerate(_serve_jobs(case))]
        return dict(case=case, systems=systems)
    system = _system(case, seed, case.get("steps", 100))
    return dict(case=case, system=system, job=ra.REMDGPU(system, precision=case["precision"]),
                cond=_Conditions(system), step=0)


def _checkpoint(job):
    return np.frombuffer(job.checkpoint_save(), np.uint8)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "wall":
        return ra.wall_table(1, case["nfwall"], state["R"], SGM_WALL, EPS_WALL, RHO_WALL)
    if kind == "forces":
        job = state["job"]
        job.compute_forces(do_sort=True, margin=MARGIN)
        got = [job.state(k) for k in range(job.nrep)]
        return dict(f=np.stack([s["f"] for s in got]), n=np.stack([s["n"] for s in got]),
                    id=np.stack([s["id"] for s in got]), energy=job.all_averages()[:, :3])
    if kind == "interval":
        job, c, s = state["job"], state["cond"], state["system"]
        _, accepted, averages, _ = ra.execute_intervals(job, s.ntemp, s.npress, state["step"], case["intervals"], c.index,
                                                        c.T, c.P, c.rng)
        state["step"] += case["intervals"]
        return dict(averages=averages, accepted=accepted, index=c.index.copy(), T=c.T.copy(), P=c.P.copy(),
                    checkpoint=_checkpoint(job))
    if kind == "batch":
        averages = []
        for _ in range(case["intervals"]):
            for job, c in zip(state["jobs"], state["cond"]):
                job.set_conditions(c.T, c.P)
            state["batch"].execute()
            for job, c, s in zip(state["jobs"], state["cond"], state["systems"]):
                pot, vol = job.pot_vol()
                ra.exchange_host(s.ntemp, s.npress, state["step"], s.pconstant, pot, vol, c.index, c.T, c.P, c.rng)
            averages.append(np.concatenate([job.all_averages() for job in state["jobs"]]))
            state["step"] += 1
        return dict(averages=np.stack(averages), index=np.concatenate([c.index for c in state["cond"]]),
                    checkpoint=[_checkpoint(job) for job in state["jobs"]])
    requests = [serve.Request(k, 0.0, s, case["intervals"]) for k, s in enumerate(state["systems"])]
    backend = serve.GPUBackend(precision=case["precision"])
    results = serve.Server(backend).run(requests)
    backend.close()
    got = [results[k] for k in range(len(requests))]
    return dict(averages=[g.averages for g in got], index=[g.index for g in got],
                r=[g.state0["r"] for g in got], v=[g.state0["v"] for g in got], q=[g.state0["q"] for g in got],
                p=[g.state0["p"] for g in got])


# --------------------------------------------------------------- cost of a case
def _pairs(job):
    """Ordered molecule pairs inside the cutoff of one replica, counted on
    the lattice start."""
    x, box, _ = _lattice(job, np.random.RandomState(0))
    total = 0
    for a in range(0, len(x), 256):
        d = x[a:a + 256, None] - x[None]
        for k in range(3):
            if PERIODIC[job["confined"]][k]:
                d[..., k] -= box[k] * np.rint(d[..., k] / box[k])
        total += int((np.sum(d * d, -1) < RC * RC).sum())
    return total - len(x)


def _job_work(job, evaluations, integrate):
    nrep = job["ntemp"] * job["npress"]
    flops = evaluations * (_pairs(job) * PAIR_FLOPS[job["model"]] + job["nmol"] * (1000 if integrate else 100)) * nrep
    return 2 * nrep * job["nmol"] * STATE_DOUBLES * 8 + (16 * NFWALL if job["confined"] else 0), flops


def work(case):
    kind = case["kind"]
    if kind == "wall":
        # the angular sum: 10 000 terms of about 20 operations per node
        return dict(bytes=case["nfwall"] * 16, flops=case["nfwall"] * 10000 * 20)
    jobs = _batch_jobs(case) if kind == "batch" else _serve_jobs(case) if kind == "serve" else [case]
    evaluations = 1 if kind == "forces" else case["intervals"] * case["steps"] + (kind == "serve")
    got = [_job_work(j, evaluations, kind != "forces") for j in jobs]
    return dict(bytes=sum(g[0] for g in got), flops=sum(g[1] for g in got))


# ---------------------------------------------------------------- 64-bit values
def _wall_table(case_size, nfwall):
    """{f, e} of the tube wall at nfwall nodes: the angular integral over the
    cylinder, its derivative by central differences, per unit coordinate."""
    R = case_size
    dr = R / nfwall
    r = np.arange(nfwall) * dr
    phi = math.pi - np.arange(10000) * (math.pi / 10000)
    rho = np.sqrt(R * R + (r * r)[:, None] - 2.0 * R * r[:, None] * np.cos(phi)[None])
    s6 = SGM_WALL ** 6
    e = math.pi * RHO_WALL * EPS_WALL * s6 * R * (math.pi / 10000) * (63.0 / 32.0 * s6 * rho ** -11 - 3.0 * rho ** -5).sum(1)
    f = np.zeros(nfwall)
    f[1:-1] = -(e[2:] - e[:-2]) / (2.0 * dr * r[1:-1])
    f[0] = f[1]
    f[-1] = 2.0 * (f[-2] - f[-3]) + f[-3]
    return np.stack([f, e], 1)


def _slit_table(H, nfwall):
    """{f, e} of two 10-4 sheets at +-H/2, f per unit coordinate."""
    z = np.arange(nfwall) * (0.5 * H / nfwall)
    c = 2.0 * math.pi * RHO_WALL * EPS_WALL * SGM_WALL ** 2

    def e(h):
        return c * (0.4 * (SGM_WALL / h) ** 10 - (SGM_WALL / h) ** 4)

    def dedh(h):
        return c * (-4.0 * (SGM_WALL / h) ** 10 + 4.0 * (SGM_WALL / h) ** 4) / h

    f = np.zeros(nfwall)
    d = dedh(0.5 * H + z) - dedh(0.5 * H - z)
    f[1:] = -d[1:] / z[1:]
    f[0] = f[1]
    return np.stack([f, e(0.5 * H + z) + e(0.5 * H - z)], 1)


def _exact_forces(system, state, table):
    """COM forces, quaternion torques, order and the three energies of one
    replica from the definition, in 64 bits."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f8 = dict(dtype=torch.float64, device=dev)
    axis = 0 if system.confined == 2 else 2
    order = np.argsort(state.r[:, axis], kind="stable")
    L = torch.tensor(state.L, **f8)
    Lp = torch.tensor([b if p else 1e9 for b, p in zip(state.L, PERIODIC[system.confined])], **f8)
    x = (torch.tensor(state.r[order], **f8) - 0.5) * L
    q = torch.tensor(state.q[order], **f8)
    mt = inputs.molecule(system.model)
    body = torch.tensor(mt.r, **f8)
    off, m = _rotate(q, body)
    N, S = off.shape[:2]
    b = 0 if S == 3 else 1
    qq = torch.tensor(np.outer(mt.q, mt.q), **f8)[b:, b:]
    sig2, eps4 = float(mt.sigma[0]) ** 2, 4.0 * float(mt.eps[0])
    site = torch.zeros(N, S, 3, **f8)
    com = torch.zeros(N, 3, **f8)
    lj = cl = wall = 0.0
    k = 1.0 / (RL - RC) ** 5
    for a in range(0, N, 128):
        i = torch.arange(a, min(N, a + 128), device=dev)
        g = x[i][:, None] - x[None]
        g = g - Lp * torch.round(g / Lp)
        r = g.norm(dim=-1)
        ok = (r < RC) & (i[:, None] != torch.arange(N, device=dev)[None])
        r = torch.where(ok, r, torch.full_like(r, RL - 1.0))
        c_, l_ = r - RC, r - RL
        outer = ok & (r > RL)
        sw = torch.where(outer, k * c_ ** 3 * (10 * l_ * l_ - 5 * l_ * c_ + c_ * c_), ok.to(r.dtype))
        dsw = torch.where(outer, 30 * k * c_ * c_ * l_ * l_, torch.zeros_like(r))
        d = g[:, :, None, None] + off[i][:, None, :, None] - off[None, :, None]
        d2 = torch.where(ok[:, :, None, None], d.square().sum(-1), torch.ones_like(d[..., 0]))
        s6 = (sig2 / d2[:, :, 0, 0]) ** 3
        e_lj = eps4 * s6 * (s6 - 1)
        f = torch.zeros_like(d)
        f[:, :, 0, 0] = (12 * eps4 * s6 * (s6 - 0.5) / d2[:, :, 0, 0])[..., None] * d[:, :, 0, 0]
        ec = qq * d2[:, :, b:, b:].rsqrt()
        f[:, :, b:, b:] += (ec / d2[:, :, b:, b:])[..., None] * d[:, :, b:, b:]
        e_cl = ec.sum((-1, -2))
        site[i] = (sw[:, :, None, None] * f.sum(3)).sum(1)
        com[i] = (-(dsw * (e_lj + e_cl) / r)[..., None] * g).sum(1)
        lj += 0.5 * float((sw * e_lj).sum())
        cl += 0.5 * float((sw * e_cl).sum())
    if system.confined:
        tab = torch.tensor(table, **f8)
        p = x + off[:, 0]
        axes = [0, 1] if system.confined == 1 else [2]
        u = p[:, axes].norm(dim=-1)
        dr = (1.0 if system.confined == 1 else 0.5) * system.wall_length / system.nfwall
        j = (u / dr).long().clamp_max(system.nfwall - 2)
        w = (u / dr - j)[:, None]
        fe = tab[j] + (tab[j + 1] - tab[j]) * w
        site[:, 0, axes] += fe[:, :1] * p[:, axes]
        wall = float(fe[:, 1].sum())
    fb = (m.transpose(-1, -2).unsqueeze(1) * site.unsqueeze(-2)).sum(-1)
    n = torch.cat([(body * fb).sum((-1, -2))[:, None], torch.linalg.cross(body.expand_as(fb), fb).sum(1)], 1)
    return (com + site.sum(1)).cpu().numpy(), n.cpu().numpy(), order.astype(np.int32), (lj, cl, wall)


def exact(case, seed):
    kind = case["kind"]
    if kind == "wall":
        return _wall_table(prepare(case, seed)["R"], case["nfwall"])
    if kind == "forces":
        s = _system(case, seed)
        table = None if s.confined == 0 else _wall_table(s.wall_length, s.nfwall) if s.confined == 1 else _slit_table(
            s.wall_length, s.nfwall)
        got = [_exact_forces(s, st, table) for st in s.states]
        return dict(f=np.stack([g[0] for g in got]), n=np.stack([g[1] for g in got]), id=np.stack([g[2] for g in got]),
                    energy=np.array([g[3] for g in got]))
    # hundreds of steps of a chaotic system: no 64-bit trajectory stands for
    # the outputs of the others
    return None
