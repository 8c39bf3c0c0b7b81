"""Performance cases of the particle-field path, through its public entry points.

Each case is one call pattern of a user's program: a splitting with its
particles and fields on the GPU advanced by some steps and read back, the
reverse mode with its gradients, an ensemble, and the device-resident 2D
deposit and evaluation. Initial states are the benchmark workloads' (1D2V
Weibel, 1D1V and 2D3V Landau damping), drawn on the GPU from a seed.

`exact` restates each path operator by operator in plain torch, in float64.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gempic.jl_amd"))

import gempic_amd as G  # noqa: E402
import gempic_amd.device  # noqa: E402

DT = 0.05
SIGMA1 = 0.02 / math.sqrt(2.0)
SIGMA2 = math.sqrt(12.0) * SIGMA1


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # a first look at a set-up, and what the smoke run does: the step is
        # all launches and latency
        dict(name="weibel_16k", kind="strang", n=16384, nx=32, degree=3, k=1.25, steps=200,
             arithmetic="fused", sort=20),
        # strong Landau damping with the electrostatic splitting, a size that
        # a laptop user of the method runs
        dict(name="landau_1d1v_100k", kind="landau1", n=100000, nx=32, degree=3, k=0.5, steps=500,
             sort=20),
        # a medium run with the library's defaults (the reference's rounding),
        # a particle count and a grid that nothing is tuned for
        dict(name="weibel_300k_reference", kind="strang", n=300001, nx=50, degree=3, k=1.25,
             steps=200, arithmetic="reference", sort=20),
        # the benchmark's Weibel run
        dict(name="weibel_4m", kind="strang", n=4194304, nx=32, degree=3, k=1.25, steps=400,
             arithmetic="fused", sort=40),
        # a state larger than the caches, finer grid
        dict(name="weibel_12m", kind="strang", n=12582912, nx=64, degree=3, k=1.25, steps=200,
             arithmetic="fused", sort=40),
        # the Boris splitting
        dict(name="boris_1m", kind="boris", n=1048576, nx=32, degree=3, k=1.25, steps=300,
             sort=20),
        # gradients of a small problem, every state kept (an optimiser's inner loop)
        dict(name="adjoint_60k", kind="adjoint", n=60000, nx=32, degree=3, k=1.25, steps=100,
             every=1, arithmetic="fused", sort=20),
        # gradients of a production-sized problem with checkpoints
        dict(name="adjoint_1m", kind="adjoint", n=1048576, nx=32, degree=3, k=1.25, steps=200,
             every=50, arithmetic="reference", sort=20),
        # a parameter scan: independent instances of uneven sizes and grids
        dict(name="ensemble_24", kind="ensemble", instances=24, n_min=65536, n_max=524288,
             steps=200, arithmetic="fused", sort=20),
        # 2D3V Landau damping: a coarse run on an uneven grid
        dict(name="landau_2d3v_150k", kind="split2d", n=150000, nx=48, ny=36, degree=3, k=0.5,
             steps=50),
        # 2D3V Landau damping at the production size
        dict(name="landau_2d3v_16m", kind="split2d", n=16777216, nx=64, ny=64, degree=3, k=0.5,
             steps=40),
        # the 2D particle-mesh coupling on particles the program keeps on the
        # GPU: charge deposit and the two field components at the particles
        dict(name="coupling_2d_16m", kind="coupling2d", n=16777216, nx=64, ny=64, degree=3, k=0.5,
             deterministic=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["strang", "strang", "strang", "landau1", "boris", "adjoint", "ensemble",
                       "split2d", "split2d", "coupling2d"])
    if kind == "strang":
        return dict(kind=kind, n=_log(rng, 10000, 8000000), nx=2 * rng.randint(8, 40),
                    degree=rng.choice([2, 3, 3]), k=round(rng.uniform(1.0, 1.5), 3),
                    steps=rng.randint(50, 200), arithmetic=rng.choice(["fused", "reference"]),
                    sort=rng.choice([20, 20, 40]))
    if kind == "landau1":
        return dict(kind=kind, n=_log(rng, 20000, 2000000), nx=2 * rng.randint(8, 32), degree=3,
                    k=0.5, steps=rng.randint(100, 400), sort=20)
    if kind == "boris":
        return dict(kind=kind, n=_log(rng, 50000, 6000000), nx=2 * rng.randint(8, 32), degree=3,
                    k=round(rng.uniform(1.0, 1.5), 3), steps=rng.randint(50, 200), sort=20)
    if kind == "adjoint":
        return dict(kind=kind, n=_log(rng, 30000, 2000000), nx=2 * rng.randint(8, 32), degree=3,
                    k=round(rng.uniform(1.0, 1.5), 3), steps=rng.randint(40, 160),
                    every=rng.choice([1, 10, 25, 50]), arithmetic=rng.choice(["fused", "reference"]),
                    sort=20)
    if kind == "ensemble":
        return dict(kind=kind, instances=rng.randint(4, 32), n_min=16384,
                    n_max=_log(rng, 65536, 500000), steps=rng.randint(50, 150),
                    arithmetic=rng.choice(["fused", "reference"]), sort=20)
    if kind == "split2d":
        # a coarse run or a production one
        n = _log(rng, 50000, 190000) if rng.random() < 0.4 else _log(rng, 1600000, 8000000)
        return dict(kind=kind, n=n, nx=rng.randint(16, 64),
                    ny=rng.randint(16, 64), degree=rng.choice([2, 3, 3]), k=0.5,
                    steps=rng.randint(20, 50))
    return dict(kind=kind, n=_log(rng, 100000, 20000000), nx=rng.randint(16, 64),
                ny=rng.randint(16, 64), degree=rng.choice([1, 2, 3, 3]), k=0.5,
                deterministic=rng.random() < 0.4)


# ---------------------------------------------------------------------------
# initial states (on the GPU, from the seed alone)

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _cos_density(g, n, k, alpha):
    """n points of the density 1 + alpha cos(k x) on [0, 2 pi / k): newton on the cdf."""
    L = 2.0 * math.pi / k
    u = L * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    x = u.clone()
    for _ in range(30):
        x = x - (x + alpha / k * torch.sin(k * x) - u) / (1.0 + alpha * torch.cos(k * x))
    return x.clamp_(0.0, math.nextafter(L, 0.0))


def _normal(g, n):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float64)


def _weibel(n, nx, degree, k, seed, alpha=1e-4, beta=1e-4):
    """Rows x, v1, v2, w, and B0."""
    g = _gen(seed)
    L = 2.0 * math.pi / k
    rows = [_cos_density(g, n, k, alpha), SIGMA1 * _normal(g, n), SIGMA2 * _normal(g, n),
            torch.full((n,), L, device="cuda", dtype=torch.float64)]
    phase = 2.0 * math.pi * float(torch.rand(1, generator=g, device="cuda"))
    b0 = beta * np.cos(k * (L / nx) * (np.arange(nx) + 0.5) + phase)
    return rows, b0, L


def _landau1(n, k, seed):
    g = _gen(seed)
    L = 2.0 * math.pi / k
    return [_cos_density(g, n, k, 0.5), _normal(g, n),
            torch.full((n,), L, device="cuda", dtype=torch.float64)], L


def _landau2(n, k, seed):
    """Rows x1, x2, v1, v2, v3, w of 1 + 0.01 cos(k x1) cos(k x2), v ~ N(0, I)."""
    g = _gen(seed)
    L = 2.0 * math.pi / k
    x2 = L * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    u = L * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    a = 0.01 * torch.cos(k * x2)            # given x2, x1 has the density 1 + a cos(k x1)
    x1 = u.clone()
    for _ in range(12):
        x1 = x1 - (x1 + a / k * torch.sin(k * x1) - u) / (1.0 + a * torch.cos(k * x1))
    x1 = x1.clamp_(0.0, math.nextafter(L, 0.0))
    return [x1, x2, _normal(g, n), _normal(g, n), _normal(g, n),
            torch.full((n,), L * L, device="cuda", dtype=torch.float64)], L


def _fill(pg, rows):
    """The reference's (D + V + n_weights) x N column-major particle matrix."""
    pg.array[:] = torch.stack(rows, dim=1).cpu().numpy().T


# ---------------------------------------------------------------------------
# what a user's program holds before the call

def _splitting(rows, nx, L, degree, cls, V, b0, arithmetic=None, sort=20):
    n = rows[0].numel()
    mesh = G.OneDGrid(0.0, L, nx)
    pg = G.ParticleGroup(1, V, n, common_weight=1.0 / n)
    _fill(pg, rows)
    ks0 = G.ParticleMeshCoupling1D(mesh, n, degree, "galerkin")
    ks1 = G.ParticleMeshCoupling1D(mesh, n, degree - 1, "galerkin")
    mx = G.Maxwell1DFEM(mesh, degree)
    e = [np.zeros(nx), np.zeros(nx)]
    b = b0.copy()
    if cls is G.HamiltonianSplittingBoris:
        h = cls(mx, ks0, ks1, pg, e, b, sync=False)
    else:
        h = cls(1, V, mx, ks0, ks1, pg, e, b, sync=False)
    if arithmetic is not None:
        h.set_arithmetic(arithmetic)
    h.set_sort_interval(sort)
    G.solve_poisson_(e[0], h, np.zeros(nx))      # E1 from the particles' charge
    h.to_device(particles=False)
    return h


def _instances(case, seed):
    """Parameters of the ensemble's instances: (n, nx, k, alpha, beta, dt)."""
    r = np.random.default_rng(int(seed))
    sizes = np.random.default_rng(case["instances"] * 1000003 + case["n_max"])
    out = []
    for _ in range(case["instances"]):
        n = int(sizes.integers(case["n_min"], case["n_max"] + 1))
        nx = int(sizes.choice([16, 32, 64]))
        k = float(r.uniform(1.0, 1.5))
        alpha, beta = np.exp(r.uniform(math.log(1e-5), math.log(1e-3), 2))
        # the field solver is stable for dt < 0.64 dx
        out.append((n, nx, k, float(alpha), float(beta), min(DT, 0.5 * 2.0 * math.pi / k / nx)))
    return out


def _dt(case):
    return min(DT, 0.5 * 2.0 * math.pi / case["k"] / case["nx"])


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("strang", "boris", "adjoint"):
        rows, b0, L = _weibel(case["n"], case["nx"], case["degree"], case["k"], seed)
        cls = G.HamiltonianSplittingBoris if kind == "boris" else G.HamiltonianSplitting
        s["h"] = _splitting(rows, case["nx"], L, case["degree"], cls, 2, b0,
                            case.get("arithmetic"), case["sort"])
        s["dt"] = _dt(case)
        if kind == "boris":
            G.staggering_(s["h"], s["dt"])
    elif kind == "landau1":
        rows, L = _landau1(case["n"], case["k"], seed)
        s["h"] = _splitting(rows, case["nx"], L, case["degree"], G.HamiltonianSplitting, 1,
                            np.zeros(case["nx"]), None, case["sort"])
        s["dt"] = DT
    elif kind == "ensemble":
        hs, dts = [], []
        for i, (n, nx, k, alpha, beta, dt) in enumerate(_instances(case, seed)):
            rows, b0, L = _weibel(n, nx, 3, k, seed * 1000 + i, alpha, beta)
            hs.append(_splitting(rows, nx, L, 3, G.HamiltonianSplitting, 2, b0,
                                 case["arithmetic"], case["sort"]))
            dts.append(dt)
        s["hs"], s["dt"], s["ens"] = hs, dts, G.Ensemble(hs)
    elif kind == "split2d":
        n, nx, ny, p = case["n"], case["nx"], case["ny"], case["degree"]
        rows, L = _landau2(n, case["k"], seed)
        mesh = G.TwoDGrid(0.0, L, nx, 0.0, L, ny)
        pg = G.ParticleGroup(2, 3, n, common_weight=1.0 / n)
        _fill(pg, rows)
        mx = G.TwoDMaxwell(mesh, p)
        ks = [G.ParticleMeshCoupling2D(pg, mesh, p, "galerkin"),
              G.ParticleMeshCoupling2D(pg, mesh, p - 1, "galerkin")]
        e = [np.zeros(nx * ny) for _ in range(3)]
        b = _b0_2d(nx, ny, seed)
        h = G.HamiltonianSplitting2D3V(mx, ks[0], ks[1], pg, e, b, sync=False)
        G.compute_e_from_rho_(e, mx, h.rho())
        h.to_device(particles=False)
        s["h"], s["dt"] = h, DT
    else:
        n, nx, ny = case["n"], case["nx"], case["ny"]
        x, y, w, f1, f2 = _coupling_inputs(case, seed)
        L = 2.0 * math.pi / case["k"]
        D = G.device.DeviceArray.from_numpy
        s["pm"] = G.ParticleMeshCoupling2D(G.ParticleGroup(2, 2, n),
                                           G.TwoDGrid(0.0, L, nx, 0.0, L, ny), case["degree"],
                                           "galerkin")
        s["x"], s["y"], s["w"] = D(x.cpu().numpy()), D(y.cpu().numpy()), D(w.cpu().numpy())
        s["f"] = (D(f1.cpu().numpy()), D(f2.cpu().numpy()))
        # the outputs, in memory of the program's own
        s["rho"], s["out"] = G.device.DeviceArray(nx * ny), (G.device.DeviceArray(n),
                                                             G.device.DeviceArray(n))
        s["views"] = [_as_tensor(a) for a in (s["rho"],) + s["out"]]
    return s


class _Array:
    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=(a.size,), typestr="<f8", version=2,
                                             strides=None, data=(a.ptr.value, False))


def _as_tensor(a):
    return torch.as_tensor(_Array(a), device="cuda")


def _b0_2d(nx, ny, seed):
    """A small smooth magnetic field (the three components' degrees of freedom)."""
    r = np.random.default_rng(int(seed))
    i, j = np.meshgrid(np.arange(nx), np.arange(ny), indexing="xy")
    out = []
    for _ in range(3):
        a, b = 2.0 * math.pi * r.random(2)
        out.append(0.05 * (np.cos(2 * math.pi * i / nx + a) * np.cos(2 * math.pi * j / ny + b)).ravel())
    return out


def _coupling_inputs(case, seed):
    g = _gen(seed)
    rows, _ = _landau2(case["n"], case["k"], seed)
    nn = case["nx"] * case["ny"]
    return rows[0], rows[1], torch.full_like(rows[0], 1.0 / case["n"]), _normal(g, nn), _normal(g, nn)


# ---------------------------------------------------------------------------
# one pass

def _state_1d(h):
    h.to_host()
    a = h.particle_group.array
    out = dict(x=a[0], v1=a[1], e1=h.e_dofs[0])
    if h.dims[1] == 2:
        out.update(v2=a[2], e2=h.e_dofs[1], b=h.b_dofs, j2=h.j_dofs[1])
    else:
        out.update(j1=h.j_dofs[0])
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("strang", "landau1", "boris"):
        G.strang_splitting_(state["h"], state["dt"], case["steps"])
        return _state_1d(state["h"])
    if kind == "adjoint":
        h = state["h"]
        h.to_device()
        r = G.strang_splitting_adjoint_(h, state["dt"], case["steps"],
                                        checkpoint_every=case["every"])
        gp = r.g_particles
        return dict(loss=np.float64(r.loss), g_x=gp[0], g_v1=gp[1], g_v2=gp[2], g_e1=r.g_e1, g_e2=r.g_e2,
                    g_b=r.g_b, g_length=np.float64(r.g_length), g_weight_sum=np.float64(r.g_weight_sum))
    if kind == "ensemble":
        G.ensemble_strang_splitting_(state["ens"], state["dt"], case["steps"])
        parts = [_state_1d(h) for h in state["hs"]]
        out = {key: np.concatenate([p[key] for p in parts]) for key in ("e1", "e2", "b", "j2")}
        out["particles"] = [h.particle_group.array[:3] for h in state["hs"]]
        return out
    if kind == "split2d":
        h = state["h"]
        h.strang_splitting(state["dt"], case["steps"])
        h.to_host()
        a = h.particle_group.array
        return dict(x1=a[0], x2=a[1], v1=a[2], v2=a[3], v3=a[4], e=list(h.e_dofs),
                    b=list(h.b_dofs), j=list(h.j_dofs))
    state["views"][0].zero_()                    # add_charge! adds
    G.add_charge_device_(state["rho"], state["pm"], state["x"], state["y"], state["w"],
                         deterministic=case["deterministic"], async_=True)
    G.evaluate_multiple_device(state["pm"], (state["x"], state["y"]), state["f"], state["out"],
                               async_=True)
    return state["views"]


# ---------------------------------------------------------------------------
# what a pass cannot do without: the state read and written once a step (8
# bytes a value), and the splines' and pushes' operations

def work(case):
    kind = case["kind"]
    if kind in ("strang", "boris"):
        # x, v1, v2, w in; x, v1, v2 out
        return dict(bytes=56.0 * case["n"] * case["steps"], flops=200.0 * case["n"] * case["steps"])
    if kind == "landau1":
        return dict(bytes=40.0 * case["n"] * case["steps"], flops=80.0 * case["n"] * case["steps"])
    if kind == "adjoint":
        # the recorded forward step, the re-run of each interval, and the reverse
        # pass (the state and the cotangents in, the cotangents out)
        again = 56.0 if case["every"] > 1 else 24.0
        return dict(bytes=(56.0 + again + 80.0) * case["n"] * case["steps"],
                    flops=800.0 * case["n"] * case["steps"])
    if kind == "ensemble":
        n = sum(i[0] for i in _instances(case, 0))
        return dict(bytes=56.0 * n * case["steps"], flops=200.0 * n * case["steps"])
    if kind == "split2d":
        # five state components and the weight in, five out
        return dict(bytes=88.0 * case["n"] * case["steps"], flops=900.0 * case["n"] * case["steps"])
    # x, y, w in; x, y in, two values out
    return dict(bytes=56.0 * case["n"], flops=(3 * 2 * (case["degree"] + 1) ** 2 + 50.0) * case["n"])


def tolerance(case):
    # sums of 64-bit values in another order: 4e-15 seen in the single calls,
    # and up to 3e-13 where rounding travels through a run's steps (particles
    # stored in another order, or the other arithmetic)
    if case["kind"] == "coupling2d":
        return {"rel": 2e-14, "max": 1e-12}
    return {"rel": 2e-12, "max": 2e-11}


# ---------------------------------------------------------------------------
# the same in plain torch

def _basis(p, t):
    """Values at offset t of the uniform B-splines of degree p, first node first."""
    if p == 0:
        return [torch.ones_like(t)]
    if p == 1:
        return [1.0 - t, t]
    s = 1.0 - t
    if p == 2:
        return [0.5 * s * s, 0.5 + t * s, 0.5 * t * t]
    return [s * s * s / 6.0, 2.0 / 3.0 + t * t * (0.5 * t - 1.0),
            2.0 / 3.0 + s * s * (0.5 * s - 1.0), t * t * t / 6.0]


def _primitive(p, t):
    """Integrals of _basis(p, .) from 0 to t."""
    if p == 0:
        return [t]
    if p == 1:
        return [t - 0.5 * t * t, 0.5 * t * t]
    t2, t3 = t * t, t * t * t
    if p == 2:
        return [0.5 * t - 0.5 * t2 + t3 / 6.0, 0.5 * t + 0.5 * t2 - t3 / 3.0, t3 / 6.0]
    t4 = t2 * t2
    return [(t - 1.5 * t2 + t3 - 0.25 * t4) / 6.0, (4.0 * t - 2.0 * t3 + 0.75 * t4) / 6.0,
            (t + 1.5 * t2 + t3 - 0.75 * t4) / 6.0, 0.25 * t4 / 6.0]


def _scatter(idx, val, size):
    """sum of val at idx, over private copies of the (small) grid."""
    copies = max(1, min(4096, (1 << 22) // size))
    lane = torch.arange(idx.numel(), device="cuda") % copies
    return torch.zeros(copies * size, device="cuda", dtype=torch.float64).scatter_add(
        0, lane * size + idx, val).view(copies, size).sum(0)


def _mass_line(p, n):
    line = {0: [1.0], 1: [4 / 6, 1 / 6], 2: [66 / 120, 26 / 120, 1 / 120],
            3: [2416 / 5040, 1191 / 5040, 120 / 5040, 1 / 5040]}[p]
    c = torch.zeros(n, device="cuda", dtype=torch.float64)
    for j, v in enumerate(line):
        c[j % n] = c[j % n] + v
        if j:
            c[-j % n] = c[-j % n] + v
    return c


class _Run1D:
    """The 1D splittings, operator by operator."""

    def __init__(self, n_total, nx, L, p, v1_only=False):
        self.nx, self.L, self.dx, self.p, self.n = nx, L, L / nx, p, n_total
        self.m0, self.m1 = torch.fft.fft(_mass_line(p, nx)), torch.fft.fft(_mass_line(p - 1, nx))
        th = 2.0 * math.pi * torch.arange(nx, device="cuda", dtype=torch.float64) / nx
        self.d = 1.0 - torch.exp(1j * th)          # u[i] - u[i + 1]
        self.v1_only = v1_only

    def _mul(self, a, f):
        return torch.fft.ifft(a * torch.fft.fft(f)).real

    def weak_curl(self, b):
        return self._mul(self.m1 / self.m0 * self.d, b)

    def curl(self, e):
        return torch.roll(e, 1) - e

    def poisson(self, rho):
        a = torch.zeros_like(self.m1)
        a[1:] = 1.0 / (self.m1[1:] * (self.d[1:].abs() ** 2))
        phi = self._mul(a, rho)
        return torch.roll(phi, 1) - phi

    def cell(self, x):
        xi = x / self.dx
        c = torch.trunc(xi.detach())
        return xi - c, c.long()

    def at(self, p, x, f):
        t, c = self.cell(x)
        return sum(f[(c - p + i) % self.nx] * b for i, b in enumerate(_basis(p, t)))

    def deposit(self, p, x, q):
        t, c = self.cell(x)
        return sum(_scatter((c - p + i) % self.nx, q * b, self.nx) for i, b in enumerate(_basis(p, t)))

    def path(self, x, xn, q, v2, b):
        """j1 of the move x -> xn, and v2 after it (the cells by truncation)."""
        p, nx = self.p - 1, self.nx
        t, c = self.cell(x)
        if self.v1_only:
            xi = xn / self.dx
            cn = torch.floor(xi.detach())
            tn, cn = xi - cn, cn.long()
        else:
            tn, cn = self.cell(xn)
        d = cn - c
        j = torch.zeros(nx, device="cuda", dtype=torch.float64)
        far = int(d.abs().max())
        for s in range(far + 1):
            right = d >= 0
            cs = torch.where(right, c + s, c - s)
            live = s <= d.abs()
            lo = t if s == 0 else torch.where(right, torch.zeros_like(t), torch.ones_like(t))
            up = torch.where(d.abs() == s, tn, torch.where(right, torch.ones_like(t), torch.zeros_like(t)))
            if not bool(live.any()):
                break
            a, e = _primitive(p, lo), _primitive(p, up)
            for i in range(p + 1):
                w = torch.where(live, (e[i] - a[i]) * self.dx, torch.zeros_like(t))
                k = (cs - p + i) % nx
                j = j + _scatter(k, q * w, nx)
                if v2 is not None:
                    v2 = v2 - b[k] * w
        return j, v2

    def strang(self, s, dt):
        x, v1, v2, q, e1, e2, b = s
        p, h = self.p, 0.5 * dt

        def hb(e2, b):
            return e2 + h / self.dx * self.weak_curl(b)

        def he(v1, v2, b):
            return (v1 + h * self.at(p - 1, x, e1), v2 + h * self.at(p, x, e2),
                    b + h / self.dx * self.curl(e2))

        def hp2(v1, e2):
            v1 = v1 + h * v2 * self.at(p - 1, x, b)
            j = h * self.deposit(p, x, q * v2)
            return v1, e2 - self._mul(1.0 / self.m0, j) / self.dx, j

        e2 = hb(e2, b)
        v1, v2, b = he(v1, v2, b)
        v1, e2, j2 = hp2(v1, e2)
        xn = x + dt * v1
        j1, v2 = self.path(x, xn, q, v2, b)
        e1 = e1 - self._mul(1.0 / self.m1, j1) / self.dx
        x = xn - self.L * torch.floor(xn.detach() / self.L)
        v1, e2, j2 = hp2(v1, e2)
        v1, v2, b = he(v1, v2, b)
        e2 = hb(e2, b)
        return [x, v1, v2, q, e1, e2, b], j2

    def strang1(self, s, dt):
        """1D1V: HB Hp1 HB."""
        x, v, q, e = s
        v = v + 0.5 * dt * self.at(self.p - 1, x, e)
        xn = x + dt * v
        j, _ = self.path(x, xn, q, None, None)
        e = e - self._mul(1.0 / self.m1, j) / self.dx
        x = xn - self.L * torch.floor(xn / self.L)
        return [x, v + 0.5 * dt * self.at(self.p - 1, x, e), q, e], j

    def push_j(self, x, v1, v2, q, dt):
        xn = x + dt * v1
        xm = 0.5 * (x + xn)
        j1, j2 = self.deposit(self.p - 1, xm, q * v1), self.deposit(self.p, xm, q * v2)
        return xn - self.L * torch.floor(xn / self.L), j1, j2

    def mid_update(self, e1m, e2m, b, j1, j2, dt):
        return (e1m - self._mul(1.0 / self.m1, j1) / self.dx,
                e2m + dt / self.dx * self.weak_curl(b) - self._mul(1.0 / self.m0, j2) / self.dx)

    def boris(self, rows, e1, b, dt, steps):
        x, v1, v2, q = rows
        p = self.p
        e2 = torch.zeros_like(e1)
        x, j1, j2 = self.push_j(x, v1, v2, q, 0.5 * dt)
        e1m, e2m = self.mid_update(e1, e2, b, 0.5 * dt * j1, 0.5 * dt * j2, 0.5 * dt)
        for _ in range(steps):
            bn = b + dt / self.dx * self.curl(e2m)
            bm, b = 0.5 * (b + bn), bn
            f1, f2, fb = self.at(p - 1, x, e1m), self.at(p, x, e2m), self.at(p - 1, x, bm)
            v1, v2 = v1 + 0.5 * dt * f1, v2 + 0.5 * dt * f2
            r = 0.5 * dt * fb
            c, sn = (1.0 - r * r) / (1.0 + r * r), 2.0 * r / (1.0 + r * r)
            v1, v2 = c * v1 + sn * v2, c * v2 - sn * v1
            v1, v2 = v1 + 0.5 * dt * f1, v2 + 0.5 * dt * f2
            x, j1, j2 = self.push_j(x, v1, v2, q, dt)
            e1, e2, j2 = e1m, e2m, dt * j2
            e1m, e2m = self.mid_update(e1m, e2m, b, dt * j1, j2, dt)
        return dict(x=x, v1=v1, v2=v2, e1=e1, e2=e2, b=b, j2=j2)


def _start_1d(case, seed, alpha=1e-4, beta=1e-4):
    rows, b0, L = _weibel(case["n"], case["nx"], case["degree"], case["k"], seed, alpha, beta)
    n = case["n"]
    r = _Run1D(n, case["nx"], L, case["degree"])
    q = rows[3] / n
    e1 = r.poisson(r.deposit(r.p, rows[0], q))
    return r, [rows[0], rows[1], rows[2], q], e1, torch.as_tensor(b0, device="cuda")


def _numpy(d):
    return {k: None if v is None else v.detach().cpu().numpy() for k, v in d.items()}


def _exact_strang(case, seed, dt, alpha=1e-4, beta=1e-4):
    r, rows, e1, b = _start_1d(case, seed, alpha, beta)
    s = rows + [e1, torch.zeros_like(e1), b]
    for _ in range(case["steps"]):
        s, j2 = r.strang(s, dt)
    return dict(x=s[0], v1=s[1], v2=s[2], e1=s[4], e2=s[5], b=s[6], j2=j2)


def _exact_adjoint(case, seed):
    from torch.utils.checkpoint import checkpoint
    dt = _dt(case)
    r, rows, e1, b = _start_1d(case, seed)
    leaf = [rows[0], rows[1], rows[2], e1, torch.zeros_like(e1), b]
    for v in leaf:
        v.requires_grad_(True)
    s = leaf[:3] + [rows[3]] + leaf[3:]

    def step(*a):
        out, _ = r.strang(list(a), dt)
        return tuple(out)

    loss = 0.0
    for _ in range(case["steps"]):
        s = checkpoint(step, *s, use_reentrant=False)
        loss = loss + dt * 0.5 * r.dx * (s[6] * r._mul(r.m1, s[6])).sum()
    g = torch.autograd.grad(loss, leaf)
    return dict(loss=loss, g_x=g[0], g_v1=g[1], g_v2=g[2], g_e1=g[3], g_e2=g[4], g_b=g[5],
                g_length=None, g_weight_sum=None)


class _Run2D:
    """The 2D3V splitting, operator by operator; grids as [ny, nx]."""

    def __init__(self, nx, ny, L, p):
        self.nx, self.ny, self.L, self.p = nx, ny, L, p
        self.dx, self.dy = L / nx, L / ny
        self.mx = [torch.fft.fft(_mass_line(d, nx)) * self.dx for d in (p, p - 1)]
        self.my = [torch.fft.fft(_mass_line(d, ny)) * self.dy for d in (p, p - 1)]

    def mass(self, f, a, c, inverse=False):
        """The tensor mass matrix of degrees p - a along x, p - c along y."""
        m = self.my[c][:, None] * self.mx[a][None, :]
        g = torch.fft.fft2(f)
        return torch.fft.ifft2(g / m if inverse else g * m).real

    def line(self, x, d):
        xi = x / d
        c = torch.ceil(xi) - 1.0
        return xi - c, c.long()

    def weights(self, x, d, p):
        t, c = self.line(x, d)
        return [(c - p + i, b) for i, b in enumerate(_basis(p, t))]

    def path(self, a, e, d):
        """Nodes and integrals along [a, e] of the splines of degree p - 1."""
        p = self.p
        xa, xe = a / d, e / d
        ca, ce = torch.floor(xa).long(), torch.floor(xe).long()
        first = torch.minimum(ca, ce) - p + 1
        count = int((ca - ce).abs().max()) + p

        def big(u):          # integral of the spline that starts at 0, up to u
            u = u.clamp(0.0, float(p))
            s, sign = 0.0, 1.0
            for j in range(p + 1):
                s = s + sign * math.comb(p, j) * (u - j).clamp(min=0.0) ** p
                sign = -sign
            return s / math.factorial(p)

        return [(first + i, d * (big(xe - (first + i)) - big(xa - (first + i)))) for i in range(count)]

    def gather(self, f, wx, wy):
        f = f.reshape(-1)
        v = 0.0
        for iy, by in wy:
            row = (iy % self.ny) * self.nx
            r = 0.0
            for ix, bx in wx:
                r = r + f[row + ix % self.nx] * bx
            v = v + r * by
        return v

    def deposit(self, q, wx, wy):
        size = self.nx * self.ny
        out = torch.zeros(size, device="cuda", dtype=torch.float64)
        for iy, by in wy:
            row = (iy % self.ny) * self.nx
            for ix, bx in wx:
                out = out + _scatter(row + ix % self.nx, q * bx * by, size)
        return out.view(self.ny, self.nx)

    def hb(self, e, b, dt):
        w = [self.mass(b[0], 0, 1), self.mass(b[1], 1, 0), self.mass(b[2], 1, 1)]

        def nxt(f, ax):
            return torch.roll(f, -1, ax)

        c = [-(w[2] - nxt(w[2], 0)) / self.dy, (w[2] - nxt(w[2], 1)) / self.dx,
             (w[0] - nxt(w[0], 0)) / self.dy - (w[1] - nxt(w[1], 1)) / self.dx]
        deg = [(1, 0), (0, 1), (0, 0)]
        return [e[k] + dt * self.mass(c[k], *deg[k], inverse=True) for k in range(3)]

    def b_update(self, e, b, dt):
        def prv(f, ax):
            return torch.roll(f, 1, ax)
        return [b[0] - dt * (e[2] - prv(e[2], 0)) / self.dy,
                b[1] + dt * (e[2] - prv(e[2], 1)) / self.dx,
                b[2] - dt * ((e[1] - prv(e[1], 1)) / self.dx - (e[0] - prv(e[0], 0)) / self.dy)]

    def he(self, s, dt):
        x, y, v1, v2, v3, q, e, b = s
        p = self.p
        wx, wy = [self.weights(x, self.dx, p - a) for a in (0, 1)], [self.weights(y, self.dy, p - a) for a in (0, 1)]
        return [x, y, v1 + dt * self.gather(e[0], wx[1], wy[0]), v2 + dt * self.gather(e[1], wx[0], wy[1]),
                v3 + dt * self.gather(e[2], wx[0], wy[0]), q, e, self.b_update(e, b, dt)]

    def hp3(self, s, dt):
        x, y, v1, v2, v3, q, e, b = s
        p = self.p
        wx, wy = [self.weights(x, self.dx, p - a) for a in (0, 1)], [self.weights(y, self.dy, p - a) for a in (0, 1)]
        v1 = v1 - dt * v3 * self.gather(b[1], wx[1], wy[0])
        v2 = v2 + dt * v3 * self.gather(b[0], wx[0], wy[1])
        j = dt * self.deposit(q * v3, wx[0], wy[0])
        return [x, y, v1, v2, v3, q, [e[0], e[1], e[2] - self.mass(j, 0, 0, True)], b], j

    def hp1(self, s, dt):
        x, y, v1, v2, v3, q, e, b = s
        p = self.p
        xn = x + dt * v1
        wx, wy = self.path(x, xn, self.dx), [self.weights(y, self.dy, p - a) for a in (0, 1)]
        v2, v3 = v2 - self.gather(b[2], wx, wy[1]), v3 + self.gather(b[1], wx, wy[0])
        j = self.deposit(q, wx, wy[0])
        x = xn - self.L * torch.floor(xn / self.L)
        return [x, y, v1, v2, v3, q, [e[0] - self.mass(j, 1, 0, True), e[1], e[2]], b], j

    def hp2(self, s, dt):
        x, y, v1, v2, v3, q, e, b = s
        p = self.p
        yn = y + dt * v2
        wx, wy = [self.weights(x, self.dx, p - a) for a in (0, 1)], self.path(y, yn, self.dy)
        v1, v3 = v1 + self.gather(b[2], wx[1], wy), v3 - self.gather(b[0], wx[0], wy)
        j = self.deposit(q, wx[0], wy)
        y = yn - self.L * torch.floor(yn / self.L)
        return [x, y, v1, v2, v3, q, [e[0], e[1] - self.mass(j, 0, 1, True), e[2]], b], j

    def poisson(self, rho):
        """E of the potential with (grad, M1 grad) phi = rho."""
        kx = 2.0 * math.pi * torch.arange(self.nx, device="cuda", dtype=torch.float64) / self.nx
        ky = 2.0 * math.pi * torch.arange(self.ny, device="cuda", dtype=torch.float64) / self.ny
        gx = ((2.0 - 2.0 * torch.cos(kx)) / self.dx ** 2)[None, :] * self.my[0][:, None] * self.mx[1][None, :]
        gy = ((2.0 - 2.0 * torch.cos(ky)) / self.dy ** 2)[:, None] * self.my[1][:, None] * self.mx[0][None, :]
        op = gx + gy
        op[0, 0] = 1.0
        f = torch.fft.fft2(rho) / op
        f[0, 0] = 0.0
        phi = torch.fft.ifft2(f).real
        return [(torch.roll(phi, 1, 1) - phi) / self.dx, (torch.roll(phi, 1, 0) - phi) / self.dy]


def _exact_split2d(case, seed):
    n, nx, ny = case["n"], case["nx"], case["ny"]
    rows, L = _landau2(n, case["k"], seed)
    r = _Run2D(nx, ny, L, case["degree"])
    q = rows[5] / n
    wx, wy = r.weights(rows[0], r.dx, r.p), r.weights(rows[1], r.dy, r.p)
    e = r.poisson(r.deposit(q, wx, wy)) + [torch.zeros(ny, nx, device="cuda", dtype=torch.float64)]
    b = [torch.as_tensor(f, device="cuda").view(ny, nx) for f in _b0_2d(nx, ny, seed)]
    s, h = rows[:5] + [q, e, b], 0.5 * DT
    for _ in range(case["steps"]):
        s[6] = r.hb(s[6], s[7], h)
        s = r.he(s, h)
        s, _ = r.hp3(s, h)
        s, _ = r.hp2(s, h)
        s, j1 = r.hp1(s, DT)
        s, j2 = r.hp2(s, h)
        s, j3 = r.hp3(s, h)
        s = r.he(s, h)
        s[6] = r.hb(s[6], s[7], h)
    out = _numpy(dict(x1=s[0], x2=s[1], v1=s[2], v2=s[3], v3=s[4]))
    out.update(e=[f.reshape(-1).cpu().numpy() for f in s[6]], b=[f.reshape(-1).cpu().numpy() for f in s[7]],
               j=[f.reshape(-1).cpu().numpy() for f in (j1, j2, j3)])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "coupling2d":
        x, y, w, f1, f2 = _coupling_inputs(case, seed)
        nx, ny = case["nx"], case["ny"]
        r = _Run2D(nx, ny, 2.0 * math.pi / case["k"], max(1, case["degree"]))
        wx, wy = r.weights(x, r.dx, case["degree"]), r.weights(y, r.dy, case["degree"])
        return [r.deposit(w, wx, wy).reshape(-1), r.gather(f1, wx, wy), r.gather(f2, wx, wy)]
    if kind == "ensemble":
        parts = []
        if sum(i[0] for i in _instances(case, seed)) * case["steps"] > 2e9:
            return None
        for i, (n, nx, k, alpha, beta, dt) in enumerate(_instances(case, seed)):
            c = dict(n=n, nx=nx, degree=3, k=k, steps=case["steps"])
            parts.append(_numpy(_exact_strang(c, seed * 1000 + i, dt, alpha, beta)))
        out = {key: np.concatenate([p[key] for p in parts]) for key in ("e1", "e2", "b", "j2")}
        out["particles"] = [np.stack([p["x"], p["v1"], p["v2"]]) for p in parts]
        return out
    size = case["n"] * case["steps"]
    if size > (5e8 if kind == "split2d" else 4e8 if kind == "adjoint" else 3e9):
        return None
    if kind == "strang":
        return _numpy(_exact_strang(case, seed, _dt(case)))
    if kind == "adjoint":
        return _numpy(_exact_adjoint(case, seed))
    if kind == "split2d":
        return _exact_split2d(case, seed)
    if kind == "boris":
        r, rows, e1, b = _start_1d(case, seed)
        return _numpy(r.boris(rows, e1, b, _dt(case), case["steps"]))
    rows, L = _landau1(case["n"], case["k"], seed)
    r = _Run1D(case["n"], case["nx"], L, case["degree"], v1_only=True)
    q = rows[2] / case["n"]
    s = [rows[0], rows[1], q, r.poisson(r.deposit(r.p, rows[0], q))]
    for _ in range(case["steps"]):
        s, j = r.strang1(s, DT)
    return _numpy(dict(x=s[0], v1=s[1], e1=s[3], j1=j))
