"""The work whose speed is followed: marches of FEL jobs on one GPU through the package's public
entry points, from a surrogate's data point (32 x 32 x 128 nodes) to the production run (256 x
256 x 2048 nodes, 16.8 million particles), a batched parameter scan, and the training and use of
the surrogate ensemble.

A march is what the drop-in host and the scan drivers do: a job set up through `mithra_amd.scan`,
a device domain, and a run of field steps with the radiation power sampled at every one.  It
returns the power rows and the state it leaves: every particle and the whole potentials and E/B of
a small mesh; of a large one, whose 25 GB a run keeps on the card, what such a job writes when its
diagnostics are due, E, B, A and phi over the mesh's mid-plane x = 0 and the bunch's charge-weighted
sums.  A bunch starts either at the job's own beginning, ahead of the undulator, or `inside`: as the
run finds it once all of it has entered, wiggling in the undulator's field and gathering E/B, where
a run spends most of its steps.

`exact` marches the same state in 64 bits with plain torch operations: NSFD update, TF/SF seed,
Mur boundaries, E/B, Boris push, zigzag deposition and the power's DFT, with E/B unrounded.
"""
import math
import tempfile

import numpy as np
import torch

from mithra_amd import abi, scan, surrogate

FP64, FP32 = abi.PRECISION_FP64, abi.PRECISION_FP32_BULK
WHOLE_NODES = 300_000        # meshes up to here return every potential and E/B
WHOLE_PARTICLES = 300_000    # bunches up to here return every particle


def march(name, n_perp, n_z, particles, steps, **more):
    case = dict(name=name, kind="march", n_perp=n_perp, n_z=n_z, particles=particles, steps=steps, gamma=800.0, K=1.2,
                lambda_u=2.0e4, spread=1e-3, current=1000.0, precision="fp64", step="plain", space_charge=False,
                seeded=False, inside=True, flattop=False, fixed_order=False)
    case.update(more)
    return case


INJECTOR = dict(gamma=59.7, K=0.8, lambda_u=2.0e4, spread=2e-3, current=500.0)   # 30 MeV, 500 A


def listed():
    return [
        # one point of the surrogate's generator: the smallest mesh, space charge and a seed, its
        # fields in FP32, step after step; the host is never far from the device here
        march("point", 32, 128, 16384, 64, precision="fp32", space_charge=True, seeded=True, inside=False, **INJECTOR),
        # a small odd-sized job marched as the drop-in host marches it, one call for each routine
        march("small-calls", 45, 203, 30012, 48, step="calls", space_charge=True, inside=False, **INJECTOR),
        # an ordinary scan point of odd sizes in FP32-bulk, and another in FP64 on the pipelined step
        march("scan-mid-fp32", 71, 397, 110000, 48, precision="fp32"),
        march("scan-mid-fp64", 90, 301, 200000, 48, step="pipelined", gamma=1200.0),
        # the largest scan point
        march("scan-large-fp32", 128, 1024, 1000000, 32, precision="fp32", gamma=1000.0),
        # FP64 runs that have to repeat bit for bit
        march("fixed-order", 64, 512, 300000, 24, fixed_order=True),
        # the space-charge, seeded workload
        march("space-charge", 128, 1024, 4194304, 16, step="pipelined", space_charge=True, seeded=True, **INJECTOR),
        # the production run, and one of half its mesh in FP32-bulk
        march("production", 256, 2048, 16777216, 16, step="pipelined", gamma=1957.9, K=1.4, lambda_u=1.8e4, spread=1e-4,
              current=3000.0, flattop=True),
        march("half-fp32", 211, 1531, 6000000, 16, precision="fp32", gamma=1957.9, K=1.4, lambda_u=1.8e4, spread=1e-4,
              current=3000.0, flattop=True),
        # a parameter scan marched as one batch of uneven instances
        dict(name="batch", kind="batch", instances=12, perp_lo=32, perp_hi=64, z_lo=128, z_hi=256, particles_lo=10000,
             particles_hi=100000, precision="fp32"),
        # the surrogate: epochs of training on the resident set, and the prediction of a large scan
        dict(name="train", kind="train", rows=1024, batch=256, epochs=8),
        dict(name="predict", kind="predict", rows=4096),
    ]


def draw(rng):
    def logu(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    what = rng.random()
    if what < 0.1:
        return dict(kind="train", rows=int(logu(300, 2048)), batch=rng.choice([64, 100, 128, 256]), epochs=rng.randint(1, 8))
    if what < 0.2:
        return dict(kind="predict", rows=int(logu(1, 8192)))
    if what < 0.3:
        lo, z = rng.randint(24, 40), rng.randint(100, 180)
        return dict(kind="batch", instances=rng.randint(3, 12), perp_lo=lo, perp_hi=lo + rng.randint(4, 24), z_lo=z,
                    z_hi=z + rng.randint(10, 80), particles_lo=10000, particles_hi=int(logu(20000, 100000)),
                    precision=rng.choice(["fp32", "fp64"]))
    nodes = logu(32 * 32 * 128, 200 * 200 * 1600)
    n_perp = min(240, max(28, int((nodes / 8.0) ** (1.0 / 3.0) * rng.uniform(0.75, 1.2))))
    n_z = min(2048, max(100, int(nodes / n_perp ** 2)))
    particles = int(logu(1e4, max(2e4, min(6e6, 0.2 * n_perp ** 2 * n_z)))) // 4 * 4
    steps = 48 if nodes < 4e6 else 16
    sc = rng.random() < 0.4
    case = march("", n_perp, n_z, particles, steps, precision=rng.choice(["fp64", "fp32"]),
                 step=rng.choice(["plain", "pipelined", "calls"]), space_charge=sc, seeded=sc and rng.random() < 0.6,
                 inside=rng.random() < 0.7, fixed_order=nodes < 4e6 and rng.random() < 0.1)
    if sc:
        case.update(INJECTOR)
    else:
        case.update(gamma=rng.uniform(100.0, 2000.0), K=rng.uniform(0.5, 2.0), lambda_u=rng.uniform(1e4, 3e4),
                    flattop=rng.random() < 0.3)
    del case["name"]
    return case


# ---------------------------------------------------------------- inputs

def instance(case, seed):
    """The scan instance of a march: the case's beam, a per cent or so away from it by the seed."""
    rng = np.random.default_rng(seed)
    u = lambda: 1.0 + 0.01 * rng.uniform(-1.0, 1.0)  # noqa: E731
    return scan.Instance(
        n_perp=case["n_perp"], n_z=case["n_z"], n_particles=4096 if case["inside"] else case["particles"],
        gamma=case["gamma"] * u(), K=case["K"] * u(), lambda_u=case["lambda_u"] * u(), spread=case["spread"] * u(),
        emittance=1.0 if case["space_charge"] else 0.0, current=case["current"] * u(), sr_frac=0.125,
        sz_frac=1.0 / 18.0 if case["space_charge"] and not case["inside"] else 0.125,
        space_charge=case["space_charge"], seed_power=1.0e6 if case["seeded"] else 0.0)


def inside_bunch(case, seed, inst, job):
    """(particles as n x 11 Charge records, bunch time) of a bunch all inside the undulator: a quiet
    start (four beamlets a quarter wavelength apart) in z, Gaussian or flat-top, Gaussian in x and
    y, each particle with the transverse momentum K cos(k_u z) its place in the undulator gives it;
    in the boosted frame."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    g, bp, und = job.grid(), job.bunch_params(), job.undulators()[0]
    n = case["particles"] // 4 * 4
    normal = lambda k: torch.randn(k, generator=gen, device="cuda", dtype=torch.float64)  # noqa: E731
    sr, _, sgb, electrons = scan.bunch_sizes(inst)
    base = torch.rand(n // 4, generator=gen, device="cuda", dtype=torch.float64)
    span = g.zmax - g.zmin
    z = (base - 0.5) * 0.66 * span if case["flattop"] else normal(n // 4).clamp(-3.0, 3.0) * 0.12 * span
    wave = inst.lambda_r * bp.gamma
    z = (z[:, None] + torch.arange(4, device="cuda", dtype=torch.float64) * (wave / 4.0)).reshape(-1)
    z = z + 0.5 * (g.zmin + g.zmax)
    wide = 0.4 * (g.xmax - g.xmin)
    x, y = (normal(n) * sr).clamp(-wide, wide), (normal(n) * sr).clamp(-wide, wide)
    tb = ((2.25 * und.lu + und.rb) / bp.gamma - float(z.min())) / (bp.beta * bp.c0) - bp.dt_shift
    lz = bp.gamma * (z + bp.beta * bp.c0 * (tb + bp.dt_shift)) - und.rb
    gam = inst.gamma * (1.0 + inst.spread * normal(n))
    gx = sgb * normal(n)
    gy = sgb * normal(n) + und.k * torch.cos(2.0 * math.pi / und.lu * lz)
    gz = bp.gamma * (torch.sqrt(gam * gam - 1.0 - gx * gx - gy * gy) - bp.beta * gam)
    rec = torch.empty((n, 11), device="cuda", dtype=torch.float64)
    rec[:, 0], rec[:, 10] = electrons / n, 1.0
    for c, v in enumerate((x, y, z, x, y, z, gx, gy, gz)):
        rec[:, 1 + c] = v
    return rec, tb


class March:
    """A domain with its job's constants and the accumulated times of its march."""

    def __init__(self, case, seed):
        self.case = case
        self.work = tempfile.TemporaryDirectory(prefix="mithra_perf_")
        inst = instance(case, seed)
        self.job = scan.set_up(inst, 0, self.work.name)
        self.t = self.job.times()
        self.seed, self.bp, self.und = self.job.seed(), self.job.bunch_params(), self.job.undulators()
        self.dom = scan.open_domain(self.job, FP64 if case["precision"] == "fp64" else FP32, case["steps"])
        self.grid = self.dom.grid
        self.time, self.tb, self.n = self.t["time"], self.t["time_bunch"], 0
        if case["inside"]:
            rec, self.tb = inside_bunch(case, seed, inst, self.job)
            self.dom.set_particles(rec.cpu().numpy())
        self.dom.set_lazy_fields(1)
        if case["fixed_order"]:
            self.dom.set_deterministic(True)
        if case["n_perp"] ** 2 * case["n_z"] > 30_000_000:   # runs of minutes tune their launches
            self.dom.autotune(reps=1)
            if case["step"] == "pipelined":
                self.dom.autotune_fused(reps=1)
        k, j = np.meshgrid(np.arange(self.grid.N2), np.arange(self.grid.N1), indexing="ij")
        self.plane = (k * self.grid.N1 * self.grid.N0 + self.grid.N0 // 2 * self.grid.N1 + j).reshape(-1)

    def run(self):
        case, dom, steps, t = self.case, self.dom, self.case["steps"], self.t
        dtb, n_sub = t["bunch_time_step"], t["n_sub"]
        for i in range(steps):
            if i == steps - 1:
                dom.set_lazy_fields(0)    # the diagnostics below read E/B everywhere
            if case["step"] == "calls":
                dom.field_update(self.time, self.seed)
                dom.bunch_advance(self.bp, self.und, self.tb, dtb, n_sub)
                dom.power_sample(self.n, i)
                dom.field_shift()
                dom.current_reset()
                dom.current_update()
            elif case["step"] == "pipelined":
                dom.step_pipelined(self.time, self.seed, self.bp, self.und, self.tb, dtb, n_sub, self.n, i,
                                   more=i < steps - 1)
            else:
                dom.step(self.time, self.seed, self.bp, self.und, self.tb, dtb, n_sub, self.n, i)
            for _ in range(n_sub):
                self.tb += dtb
            self.time += t["dt"]
            self.n += 1
        dom.set_lazy_fields(1)
        out = {"power": dom.power_fetch(0, steps, 1, 1)[:, 0, 0]}
        if self.grid.nodes <= WHOLE_NODES:
            out["e"], out["b"] = dom.get_fields()
            out["a"], phi = dom.get_potentials(0)
            out["a_before"], phi_before = dom.get_potentials(1)
            if phi is not None:
                out["phi"], out["phi_before"] = phi, phi_before
        else:
            out["e"], out["b"], out["a"], phi = dom.sample_nodes(self.plane)
            if self.grid.space_charge:
                out["phi"] = phi
        if case["particles"] <= WHOLE_PARTICLES:
            out["particles"] = dom.get_particles()
        else:
            out["bunch"] = dom.bunch_sums()
        return out

    def close(self):
        self.dom.close()
        self.job.close()
        self.work.cleanup()

    __del__ = close


class Scan:
    def __init__(self, case, seed):
        self.work = tempfile.TemporaryDirectory(prefix="mithra_perf_")
        insts = scan.generate(case["instances"], seed=int(seed), n_perp=(case["perp_lo"], case["perp_hi"]),
                              n_z=(case["z_lo"], case["z_hi"]), n_particles=(case["particles_lo"], case["particles_hi"]))
        # every seed's scan has the same sizes, so that one costs what another does
        like = scan.generate(case["instances"], seed=4, n_perp=(case["perp_lo"], case["perp_hi"]),
                             n_z=(case["z_lo"], case["z_hi"]), n_particles=(case["particles_lo"], case["particles_hi"]))
        for a, b in zip(insts, like):
            a.n_perp, a.n_z, a.n_particles = b.n_perp, b.n_z, b.n_particles
        self.prepared = scan.prepare(insts, self.work.name, FP64 if case["precision"] == "fp64" else FP32)

    def run(self):
        results, _, _ = scan.run_batch(self.prepared, autotune=False)
        return [{"power": P, "bunching": b} for P, b in results]

    def close(self):
        for p in self.prepared:
            p.dom.close()
            p.job.close()
        self.work.cleanup()

    __del__ = close


def network(case, seed):
    """(parameters per member, inputs, targets) of the surrogate's ensemble: He-normal weights and
    zero biases; standardised scalars and a bell-shaped current profile; smooth targets."""
    gen = torch.Generator().manual_seed(int(seed))
    params = []
    for _ in range(surrogate.MEMBERS):
        for di, do in zip(surrogate.DIMS[:-1], surrogate.DIMS[1:]):
            params += [torch.randn(di * do, generator=gen) * math.sqrt(2.0 / di), torch.zeros(do)]
    n, bins = case["rows"], surrogate.PROFILE_BINS
    s = torch.randn(n, 8, generator=gen)
    at = torch.linspace(-1.0, 1.0, bins)
    prof = torch.exp(-0.5 * (at / (0.12 * torch.exp(0.2 * s[:, 7:8]))) ** 2)
    x = torch.cat([s, prof], 1)
    mix = torch.randn(8, surrogate.DIMS[-1], generator=gen) / math.sqrt(8.0)
    t = torch.sin(s @ mix) + 0.1 * s[:, :1]
    return torch.cat(params).numpy(), x.numpy(), t.numpy()


class Network:
    LR, LR_MIN = 1e-3, 1e-6

    def __init__(self, case, seed):
        self.case = case
        params, self.x, t = network(case, seed)
        self.mlp = abi.MLP(surrogate.DIMS, members=surrogate.MEMBERS, seed=1)
        self.mlp.set_params(params)
        self.order = int(seed) % 1000
        if case["kind"] == "train":
            self.mlp.set_data(self.x, t)

    def run(self):
        if self.case["kind"] == "predict":
            return self.mlp.forward(self.x)
        loss = self.mlp.train_epochs(self.case["epochs"], min(self.case["batch"], self.case["rows"]), self.LR,
                                     self.LR_MIN, self.order)
        return {"loss": loss, "params": self.mlp.params()}

    def close(self):
        self.mlp.close()


def prepare(case, seed):
    kind = case["kind"]
    return March(case, seed) if kind == "march" else Scan(case, seed) if kind == "batch" else Network(case, seed)


def run(state):
    return state.run()


def work(case):
    """Bytes: of a march, each step, the two older levels of every potential read and the new one
    written, and a particle's position, momentum, charge and flag read and its position, momentum and
    flag written; of the networks, the parameters (and in training their two moments) once each way
    a step, the rows and the outputs.  Operations: 60 a node and component and 700 a particle and
    step; 2 a weight and row forward, 6 with the gradients."""
    if case["kind"] == "march":
        nodes, real = case["n_perp"] ** 2 * case["n_z"], 8 if case["precision"] == "fp64" else 4
        comps = 4 if case["space_charge"] else 3
        return {"bytes": case["steps"] * (nodes * comps * 3 * real + case["particles"] * 120),
                "flops": case["steps"] * (nodes * comps * 60 + case["particles"] * 700)}
    if case["kind"] == "batch":
        total = {"bytes": 0, "flops": 0}
        for i in scan.generate(case["instances"], seed=4, n_perp=(case["perp_lo"], case["perp_hi"]),
                               n_z=(case["z_lo"], case["z_hi"]), n_particles=(case["particles_lo"], case["particles_hi"])):
            nodes, real = i.n_perp ** 2 * i.n_z, 8 if case["precision"] == "fp64" else 4
            total["bytes"] += i.n_steps * (nodes * 9 * real + i.n_particles * 120)
            total["flops"] += i.n_steps * (nodes * 180 + i.n_particles * 700)
        return total
    dims = surrogate.DIMS
    weights = surrogate.MEMBERS * sum(a * b for a, b in zip(dims[:-1], dims[1:]))
    if case["kind"] == "predict":
        n = case["rows"]
        return {"bytes": 2 * weights + 4 * n * (dims[0] + surrogate.MEMBERS * dims[-1]), "flops": 2 * weights * n}
    batch = min(case["batch"], case["rows"])
    steps = case["epochs"] * (case["rows"] // batch)
    return {"bytes": steps * (24 * weights + batch * (2 * dims[0] + 4 * dims[-1])), "flops": 6 * steps * batch * weights}


# ---------------------------------------------------------------- the same in 64 bits

PI, EC, EM = 3.1415926535, 1.602e-19, 9.109e-31     # the constants the solver is defined with


def shifted(n, sz, sx, sy):
    """The interior's neighbours at offset (sz, sx, sy) of an array [z, x, y]."""
    cut = lambda s, size: slice(1 + s, size - 1 + s)  # noqa: E731
    return n[cut(sz, n.shape[0]), cut(sx, n.shape[1]), cut(sy, n.shape[2])]


def advance_interior(P, N, M, a, source, alpha, beta):
    """P, holding the source, becomes the new level at the interior nodes (NSFD)."""
    def pair(dx, dy):
        v = shifted(N, 0, dx, dy) + shifted(N, 0, -dx, -dy)
        return v + beta * (shifted(N, 1, dx, dy) + shifted(N, -1, dx, dy) + shifted(N, 1, -dx, -dy) +
                           shifted(N, -1, -dx, -dy))
    v = a[0] * shifted(N, 0, 0, 0) - shifted(M, 0, 0, 0)
    v += alpha * (a[1] * pair(1, 0) + a[2] * pair(0, 1))
    v += a[3] * (shifted(N, 1, 0, 0) + shifted(N, -1, 0, 0))
    inner = shifted(P, 0, 0, 0)
    inner.mul_(source).add_(v)


def boundaries(P, N, M, co):
    """Second-order Mur faces, edges and corners; axes z, x, y are 0, 1, 2."""
    c, ends = slice(1, -1), ((0, 1), (-1, -2))
    for B, axes in ((co.bB, (1, 2, 0)), (co.cB, (2, 1, 0)), (co.dB, (0, 1, 2))):   # normal, and two along the face
        p, n, m = (v.permute(axes) for v in (P, N, M))
        for i, o in ends:
            t = n[i, 2:, c] + n[i, :-2, c] + n[o, 2:, c] + n[o, :-2, c]
            u = n[i, c, 2:] + n[i, c, :-2] + n[o, c, 2:] + n[o, c, :-2]
            p[i, c, c] = (B[0] * (m[i, c, c] + p[o, c, c]) + B[1] * m[o, c, c] + B[2] * (n[i, c, c] + n[o, c, c]) +
                          B[3] * t + B[4] * u)
    for B, axes in ((co.eE, (1, 2, 0)), (co.fE, (2, 0, 1)), (co.gE, (0, 1, 2))):   # two across, and along the edge
        p, n, m = (v.permute(axes) for v in (P, N, M))
        for i, o in ends:
            for k, q in ends:
                four = n[i, k] + n[o, k] + n[i, q] + n[o, q]
                p[i, k, c] = (B[0] * (p[o, k, c] + m[i, q, c]) + B[1] * (m[o, k, c] + p[i, q, c]) +
                              B[2] * (m[i, k, c] + p[o, q, c]) + B[3] * four[c] + B[4] * (four[2:] + four[:-2]) -
                              m[o, q, c])
    h = co.hC
    for z, dz in ends:
        for x, dx in ends:
            for y, dy in ends:
                s = N[z, x, y] * h[16] + M[z, x, y] * h[8]
                for t, at in enumerate(((z, dx, y), (z, x, dy), (dz, x, y), (z, dx, dy), (dz, dx, y), (dz, x, dy),
                                        (dz, dx, dy))):
                    s = s + P[at] * h[1 + t] + N[at] * h[16] + M[at] * h[9 + t]
                P[z, x, y] = -s / h[0]


def seed_potential(s, x, y, z, time):
    """The Gaussian beam's boosted-frame vector potential (3 arrays) at points and a time."""
    def pulse(t, phase):
        w = torch.cos(2 * PI * s.f0 * (t - s.t0) + s.cep + phase) * torch.exp(-1.3863 * ((t - s.t0) / s.s) ** 2)
        return torch.where((t - s.t0).abs() > 10.0 * s.s, torch.zeros_like(w), w)
    r = (x - s.position[0], y - s.position[1],
         s.gamma * (z + s.beta * s.c0 * (time + s.dt_shift)) - s.position[2])
    d, p = s.direction, s.polarization
    q = (d[1] * p[2] - d[2] * p[1], d[2] * p[0] - d[0] * p[2], d[0] * p[1] - d[1] * p[0])
    dot = lambda v: r[0] * v[0] + r[1] * v[1] + r[2] * v[2]  # noqa: E731
    along, u, v = dot(d), dot(p), dot(q)
    tl = s.gamma * (time + s.dt_shift + s.beta / s.c0 * z) - along / s.c0
    lam = s.c0 / s.f0
    zp, zs = PI * s.radius[0] ** 2 / lam, PI * s.radius[1] ** 2 / lam
    wp, ws = torch.sqrt(1.0 + (along / zp) ** 2), torch.sqrt(1.0 + (along / zs) ** 2)
    phase = (0.5 * (torch.atan(along / zp) + torch.atan(along / zs) - PI) -
             PI * along / lam * ((u / (zp * wp)) ** 2 + (v / (zs * ws)) ** 2))
    size = torch.exp(-(u / (s.radius[0] * wp)) ** 2 - (v / (s.radius[1] * ws)) ** 2) / torch.sqrt(ws * wp) * s.amplitude
    f = torch.where(pulse(tl, torch.zeros_like(tl)).abs() < 1.0e-6, torch.zeros_like(tl), size * pulse(tl, phase))
    return f * p[0], f * p[1], f * p[2] * s.gamma


def inject(A, g, co, s, time):
    """The TF/SF planes: two node planes either side of each face, from their neighbours' seed."""
    axis = lambda lo, d, n: lo + d * torch.arange(n, device="cuda", dtype=torch.float64)  # noqa: E731
    at = (axis(g.zmin, g.dz, g.N2), axis(g.xmin, g.dx, g.N0), axis(g.ymin, g.dy, g.N1))
    size = (g.N2, g.N0, g.N1)
    for ax, coef in ((1, co.a[1]), (2, co.a[2]), (0, co.a[3])):
        n = size[ax]
        for to, frm, sign in ((1, 2, -1.0), (2, 1, 1.0), (n - 2, n - 3, -1.0), (n - 3, n - 2, 1.0)):
            z, x, y = torch.meshgrid(*[at[k][frm:frm + 1] if k == ax else at[k][2:-2] for k in range(3)], indexing="ij")
            where = tuple(slice(to, to + 1) if k == ax else slice(2, -2) for k in range(3))
            for c, f in enumerate(seed_potential(s, x, y, z, time)):
                A[c][where] += sign * coef * f


def evaluate(P, N, phi, g):
    """E and B (six arrays) from two levels, on the interior nodes; the end planes copy their neighbours."""
    out = [torch.zeros_like(N[0]) for _ in range(6)]
    def diff(f, ax, h):
        d = [0, 0, 0]
        d[ax] = 1
        return (shifted(f, *d) - shifted(f, *[-v for v in d])) / (2.0 * h)
    steps = ((0, g.dz), (1, g.dx), (2, g.dy))
    for c in range(3):
        e = (shifted(N[c], 0, 0, 0) - shifted(P[c], 0, 0, 0)) / g.dt
        if phi is not None:
            e -= diff(phi, *steps[(1, 2, 0)[c]])
        shifted(out[c], 0, 0, 0).copy_(e)
        # B = the curl of the mean of the two levels; components and axes x, y, z are axes 1, 2, 0
        p, q = (c + 1) % 3, (c + 2) % 3
        ap, aq = steps[(1, 2, 0)[p]], steps[(1, 2, 0)[q]]
        shifted(out[3 + c], 0, 0, 0).copy_(0.5 * (diff(N[q], *ap) + diff(P[q], *ap) - diff(N[p], *aq) - diff(P[p], *aq)))
    for f in out:
        f[0], f[-1] = f[1], f[-2]
    return out


def corners(g, frac):
    """The eight corners of a cell: (offset in nodes, weight's x, y and z factor) each."""
    lo, hi = [1.0 - f for f in frac], frac
    for k in (0, 1):
        for j in (0, 1):
            for i in (0, 1):
                yield k * g.N0 * g.N1 + i * g.N1 + j, (hi if i else lo)[0], (hi if j else lo)[1], (hi if k else lo)[2]


def inside(r, g):
    return ((r[0] < g.xmax - g.dx) & (r[0] > g.xmin + g.dx) & (r[1] < g.ymax - g.dy) & (r[1] > g.ymin + g.dy) &
            (r[2] < g.zp1) & (r[2] >= g.zp0))


def cell(r, g):
    u = [(r[c] - (g.xmin, g.ymin, g.zmin)[c]) / (g.dx, g.dy, g.dz)[c] for c in range(3)]
    i = [torch.floor(v) for v in u]
    return [v.long() for v in i], [v - w for v, w in zip(u, i)]


def push(r, gb, flag, eb, g, bp, und, tb):
    """One bunch sub-step; r, gb: lists of three arrays, replaced; flag updated in place."""
    zr = torch.remainder(r[2] - g.zmin, g.Lz) + g.zmin
    mine = (zr >= g.zp0) & (zr < g.zp1)
    B, E = [torch.zeros_like(r[0]) for _ in range(3)], [torch.zeros_like(r[0]) for _ in range(3)]
    for U in und[:1]:
        b0, ku = EM * bp.c0 * 2 * PI / U.lu * U.k / EC, 2 * PI / U.lu
        ct, st = math.cos(U.theta), math.sin(U.theta)
        lz = bp.gamma * (r[2] + bp.beta * bp.c0 * (tb + bp.dt_shift)) - U.rb
        ly = r[0] * ct + r[1] * st
        fringe = torch.exp(-(ku * lz) ** 2 / 2.0)
        before = lz < 0.0
        d = b0 * torch.cosh(ku * ly) * torch.where(before, fringe * ku * lz, torch.sin(ku * lz)) * bp.gamma
        B[0], B[1] = d * ct, d * st
        B[2] = b0 * torch.sinh(ku * ly) * torch.where(before, fringe, torch.cos(ku * lz))
        E[0], E[1] = -d * bp.c0 * bp.beta * st, d * bp.c0 * bp.beta * ct
    use = (flag == 1.0) & inside(r, g)
    (i, j, k), frac = cell(r, g)
    m = torch.where(use, (k * g.N0 + i) * g.N1 + j, torch.zeros_like(k))
    for off, wx, wy, wz in corners(g, frac):
        w = torch.where(use, wx * wy * wz, torch.zeros_like(wx))
        for c in range(3):
            E[c] += w * eb[c].view(-1)[m + off]
            B[c] += w * eb[3 + c].view(-1)[m + off]
    reached = bp.gamma * (r[2] + bp.beta * bp.c0 * (tb + bp.dt_shift)) > -und[0].dist
    flag.copy_(torch.where(mine & (flag != 1.0), reached.double(), flag))
    cross = lambda a, b: [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]  # noqa: E731
    norm = lambda v: torch.sqrt(1.0 + v[0] * v[0] + v[1] * v[1] + v[2] * v[2])  # noqa: E731
    um = [gb[c] + bp.r1 * E[c] for c in range(3)]
    d = norm(um)
    up = [bp.r2 / d * v + um[c] for c, v in enumerate(cross(um, B))]
    f = 2.0 / (d / bp.r2 + bp.r2 / d * (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]))
    new = [f * v + um[c] + bp.r1 * E[c] for c, v in enumerate(cross(up, B))]
    s = bp.dtb / norm(new)
    for c in range(3):
        gb[c] = torch.where(mine, new[c], gb[c])
        r[c] = torch.where(mine, r[c] + s * new[c], r[c])


def deposit(J, rho, q, rp, rm, g):
    """The zigzag current of rm -> rp, and the charge at rp, added to J (three arrays) and rho."""
    (ip, _), (im, _) = cell(rp, g), cell(rm, g)
    lo, d = (g.xmin, g.ymin, g.zmin), (g.dx, g.dy, g.dz)
    relay = []
    for c in range(3):
        a, b = torch.minimum(ip[c], im[c]).double(), torch.maximum(ip[c], im[c]).double()
        relay.append(torch.minimum(a * d[c] + d[c] + lo[c], torch.maximum(b * d[c] + lo[c], 0.5 * (rm[c] + rp[c]))))
    bp, bm = inside(rp, g), inside(rm, g)

    def half(ok, i, r, way):
        m = torch.where(ok, (i[2] * g.N0 + i[0]) * g.N1 + i[1], torch.zeros_like(i[0]))
        _, f = cell([0.5 * (r[c] + relay[c]) for c in range(3)], g)
        w0 = torch.where(ok, 0.5 * q, torch.zeros_like(q))
        for off, wx, wy, wz in corners(g, f):
            for c, w in enumerate((wy * wz, wx * wz, wx * wy)):
                J[c].view(-1).index_add_(0, m + off, w0 * w * way[c])
        return m

    m = half(bp, ip, rp, [rp[c] - relay[c] for c in range(3)])
    if rho is not None:
        w0 = torch.where(bp, q, torch.zeros_like(q))
        for off, wx, wy, wz in corners(g, cell(rp, g)[1]):
            rho.view(-1).index_add_(0, m + off, w0 * wx * wy * wz)
    half(bm, im, rm, [relay[c] - rm[c] for c in range(3)])


class Exact:
    """The march of one domain in 64 bits."""

    def __init__(self, job, rec, tb, t, dom):
        self.g, self.co, self.bp, self.und, self.seed = job.grid(), job.coeffs(), job.bunch_params(), job.undulators(), job.seed()
        g = self.g
        self.t, self.time, self.tb, self.n = t, t["time"], tb, 0
        comps = 4 if g.space_charge else 3
        self.level = [[torch.zeros(g.N2, g.N0, g.N1, device="cuda", dtype=torch.float64) for _ in range(comps)] for _ in range(3)]
        for at, level in ((1, 0), (2, 1)):            # new, now, before
            if abs(self.seed.amplitude) > 1.0e-50:
                a, phi = dom.get_potentials(level)
                a = torch.from_numpy(a).cuda().view(g.N2, g.N0, g.N1, 3)
                for c in range(3):
                    self.level[at][c].copy_(a[..., c])
        rec = rec.cuda()
        self.q, self.flag = rec[:, 0].contiguous(), rec[:, 10].contiguous()
        self.r = [rec[:, 1 + c].contiguous() for c in range(3)]
        self.gb = [rec[:, 7 + c].contiguous() for c in range(3)]
        _, _, self.Nf, self.pc, z, w = job.power()
        # the DFT's phases, and the plane's cell
        ang = torch.arange(self.Nf, device="cuda", dtype=torch.float64) * (float(w[0]) * g.dt)
        self.cos, self.sin = torch.cos(ang), torch.sin(ang)
        self.z = float(z[0])
        self.ring = torch.zeros(self.Nf, 4, g.N0 - 4, g.N1 - 4, device="cuda", dtype=torch.float64)
        self.power = []

    def sample(self, eb):
        g, bp = self.g, self.bp
        if not g.zp0 <= self.z < g.zp1:
            return self.power.append(0.0)
        u = (self.z - g.zmin) / g.dz
        k, f = int(u), u - int(u)
        ex, ey, _, bx, by, _ = [((1.0 - f) * v[k] + f * v[k + 1])[2:-2, 2:-2] for v in eb]
        self.ring[self.n % self.Nf] = bp.gamma * torch.stack([ex + bp.c0 * bp.beta * by, ey - bp.c0 * bp.beta * bx,
                                                              bx - bp.beta / bp.c0 * ey, by + bp.beta / bp.c0 * ex])
        re, im = torch.tensordot(self.cos, self.ring, 1), torch.tensordot(self.sin, self.ring, 1)
        self.power.append(self.pc * float((re[0] * re[3] + im[0] * im[3] - re[1] * re[2] - im[1] * im[2]).sum()))

    def step(self):
        P, N, M = self.level
        g, co = self.g, self.co
        for c in range(len(P)):
            advance_interior(P[c], N[c], M[c], co.a, co.a[5] if c == 3 else co.a[4], co.alpha, co.beta)
        if abs(self.seed.amplitude) > 1.0e-50:
            inject(P, g, co, self.seed, self.time)
        for p, n, m in zip(P, N, M):
            boundaries(p, n, m, co)
        eb = evaluate(P, N, N[3] if len(P) == 4 else None, g)
        before = list(self.r)
        for _ in range(self.t["n_sub"]):
            push(self.r, self.gb, self.flag, eb, g, self.bp, self.und, self.tb)
            self.tb += self.t["bunch_time_step"]
        self.sample(eb)
        self.level = [M, P, N]
        for v in M:
            v.zero_()
        deposit(M, M[3] if len(P) == 4 else None, self.q, self.r, before, g)
        self.time += self.t["dt"]
        self.n += 1
        self.eb, self.before = eb, before


def exact_march(case, seed):
    s = March({**case, "fixed_order": False}, seed)
    e = Exact(s.job, torch.from_numpy(s.dom.get_particles()), s.tb, s.t, s.dom)
    for _ in range(case["steps"]):
        e.step()
    flat = lambda v: torch.stack(list(v), -1).reshape(-1)  # noqa: E731
    out = {"power": np.array(e.power)}
    _, now, old = e.level
    if e.g.nodes <= WHOLE_NODES:
        out.update(e=flat(e.eb[:3]), b=flat(e.eb[3:]), a=flat(now[:3]), a_before=flat(old[:3]))
        if e.g.space_charge:
            out.update(phi=now[3].reshape(-1), phi_before=old[3].reshape(-1))
    else:
        mid = lambda v: torch.stack([f[:, e.g.N0 // 2].reshape(-1) for f in v], -1)  # noqa: E731
        out.update(e=mid(e.eb[:3]), b=mid(e.eb[3:]), a=mid(now[:3]))
        if e.g.space_charge:
            out["phi"] = mid(now[3:])[:, 0]
    if case["particles"] <= WHOLE_PARTICLES:
        out["particles"] = torch.stack([e.q, *e.r, *e.before, *e.gb, e.flag], 1)
    else:
        q = e.q
        out["bunch"] = torch.stack([q.sum()] + [(q * v ** k).sum() for vs in (e.r, e.gb) for k in (1, 2) for v in vs])
    s.close()
    return out


def exact_batch(case, seed):
    s = Scan(case, seed)
    if sum(p.inst.n_steps for p in s.prepared) > 4000:
        s.close()
        return None
    out = []
    for p in s.prepared:
        e = Exact(p.job, torch.from_numpy(p.dom.get_particles()), p.t["time_bunch"], p.t, p.dom)
        b = []
        for i in range(p.inst.n_steps):
            e.step()
            if i % p.inst.every == 0:
                b.append(float(torch.hypot((e.q * torch.cos(p.k * e.r[2])).sum(), (e.q * torch.sin(p.k * e.r[2])).sum()) / e.q.sum()))
        at = [i * p.inst.every for i in range(scan.SAMPLES) if i * p.inst.every < p.inst.n_steps]
        out.append({"power": np.array(e.power)[at], "bunching": np.array(b[:len(at)])})
    s.close()
    return out


def permutations(seed, n, epochs):
    """Fisher-Yates permutations on a 64-bit Mersenne twister (Matsumoto and Nishimura's mt19937-64),
    a number below a bound taken by multiplication and rejection (Lemire's method)."""
    top, low, full = 0xFFFFFFFF80000000, 0x7FFFFFFF, (1 << 64) - 1
    mt = [seed & full]
    for i in range(1, 312):
        mt.append((6364136223846793005 * (mt[-1] ^ (mt[-1] >> 62)) + i) & full)

    def numbers():
        while True:
            for i in range(312):
                x = (mt[i] & top) | (mt[(i + 1) % 312] & low)
                mt[i] = mt[(i + 156) % 312] ^ (x >> 1) ^ (0xB5026F5AA96619E9 if x & 1 else 0)
            for x in list(mt):
                x ^= (x >> 29) & 0x5555555555555555
                x ^= (x << 17) & 0x71D67FFFEDA60000
                x ^= (x << 37) & 0xFFF7EEE000000000
                yield (x ^ (x >> 43)) & full

    gen = numbers()
    for _ in range(epochs):
        q = list(range(n))
        for i in range(n - 1, 0, -1):
            v = next(gen) * (i + 1)
            if v & full < i + 1:
                while v & full < (-(i + 1) & full) % (i + 1):
                    v = next(gen) * (i + 1)
            j = v >> 64
            q[i], q[j] = q[j], q[i]
        yield q


def exact_network(case, seed):
    params, x, t = (torch.from_numpy(v).cuda().double() for v in network(case, seed))
    dims, members = surrogate.DIMS, surrogate.MEMBERS
    w = params.view(members, -1).clone().requires_grad_(True)

    def predict(rows):
        h, at = rows.expand(members, *rows.shape), 0
        for l, (di, do) in enumerate(zip(dims[:-1], dims[1:])):
            h = torch.stack([h[e] @ w[e, at:at + di * do].view(di, do) + w[e, at + di * do:at + (di + 1) * do]
                             for e in range(members)])
            at += (di + 1) * do
            h = torch.nn.functional.silu(h) if l + 2 < len(dims) else h
        return h

    if case["kind"] == "predict":
        with torch.no_grad():
            return predict(x)
    batch = min(case["batch"], case["rows"])
    steps = case["rows"] // batch
    m, v, count, losses = torch.zeros_like(w), torch.zeros_like(w), 0, []
    for ep, order in enumerate(permutations(int(seed) % 1000, case["rows"], case["epochs"])):
        lr = max(Network.LR * 0.5 * (1.0 + math.cos(math.pi * ep / case["epochs"])), Network.LR_MIN)
        total = 0.0
        for b in range(steps):
            at = torch.tensor(order[b * batch:(b + 1) * batch], device="cuda")
            loss = ((predict(x[at]) - t[at]) ** 2).mean((1, 2))
            grad, = torch.autograd.grad(loss.sum(), w)
            total += float(loss.sum()) / (steps * members)
            count += 1
            with torch.no_grad():
                m = 0.9 * m + 0.1 * grad
                v = 0.999 * v + 0.001 * grad * grad
                w -= lr * (m / (1.0 - 0.9 ** count)) / (torch.sqrt(v / (1.0 - 0.999 ** count)) + 1e-8)
        losses.append(total)
    return {"loss": np.array(losses), "params": w.detach().reshape(-1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "march":
        # seconds on the card, by nodes and particles
        return exact_march(case, seed)
    return exact_batch(case, seed) if kind == "batch" else exact_network(case, seed)
