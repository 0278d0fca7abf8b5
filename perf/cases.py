"""The work a user of this framework has it do, as timed cases.

Twelve listed cases cover the configurations the benchmark and the tests run: the barotropic
vorticity (BVE) step and its FMM velocity from 6 x 28^2 to 6 x 512^2 particles, the Poisson solve,
the pair sums of a shallow-water stage, an ensemble, a 4D-Var gradient, the lat-lon tree and the
direct sums.  ``draw`` gives further cases of the same ranges.

Particles sit on the cubed sphere in 6 * 4^(levels-1) leaves of m x m Chebyshev nodes; the FMM
proxies have degree d.  ``exact`` restates each path as an O(N^2) sum in plain FP64 torch, so its
distance to an FMM result is the FMM's truncation error plus the rounding of the precision.
"""
import importlib
import math

import numpy as np
import torch
import torch.utils.checkpoint

sb = importlib.import_module("spectral-bslpm_amd")
autograd = importlib.import_module("spectral-bslpm_amd.autograd")

EPS = 1e-4          # kernel regularisation of the vortex and shallow-water kernels
OMEGA = 7.292e-5    # rotation rate, 1/s
LAP_EPS = 0.1       # width of the regularised-Laplacian kernel
FLOP = {"vortex": 27, "log": 13, "swe": 40, "lap": 30}  # per pair; division, root, log count one


def listed():
    return [
        # the smallest velocity evaluation of the tests' sizes, in the layout with particles = proxies
        # (even degree 6): launches and latency
        dict(name="velocity_28", kind="velocity", levels=3, d=6, m=7, theta=0.7, precision="fp64"),
        # one BVE step at 6 x 64^2, the small configuration (equal-area weights), FP64
        dict(name="step_64", kind="step", levels=4, d=8, m=8, theta=0.7, precision="fp64", members=1, dt=3600.0,
             weights="equal_area"),
        # one FP64 velocity evaluation at 6 x 224^2: odd sizes, 49 points per leaf and per panel
        dict(name="velocity_224", kind="velocity", levels=6, d=6, m=7, theta=0.7, precision="fp64"),
        # the headline BVE step at 6 x 512^2, mixed precision
        dict(name="step_512_mixed", kind="step", levels=7, d=8, m=8, theta=0.7, precision="mixed", members=1,
             dt=3600.0),
        # the sphere Poisson solve at 6 x 256^2, FP64
        dict(name="poisson_256", kind="poisson", levels=6, d=10, m=8, theta=0.6, precision="fp64", targets=0),
        # the same solve evaluated at 4,096 points off the grid, FP64
        dict(name="poisson_256_targets", kind="poisson", levels=6, d=10, m=8, theta=0.6, precision="fp64",
             targets=4096),
        # the two FMM evaluations of a shallow-water stage at 6 x 192^2, mixed precision
        dict(name="swe_192_mixed", kind="swe", levels=6, d=5, m=6, theta=0.7, precision="mixed"),
        # one step of a 16-member BVE ensemble at 6 x 96^2, mixed precision
        dict(name="ensemble_96", kind="step", levels=5, d=8, m=6, theta=0.7, precision="mixed", members=16, dt=3600.0),
        # loss and gradient of a 4-step vorticity 4D-Var at 6 x 96^2 (forward and backward), mixed precision
        dict(name="gradient_96", kind="gradient", levels=5, d=8, m=6, theta=0.7, precision="mixed", steps=4, every=2,
             dt=900.0),
        # the shallow-water velocity on the 1 degree lat-lon grid's particle tree, FP64
        dict(name="latlon_1deg", kind="latlon", rows=180, d=10, theta=0.5),
        # the all-pairs log sum over 6 x 64^2 points, FP64
        dict(name="direct_log_64", kind="direct_log", sources=24576),
        # the velocity at 4,096 points from 6 x 256^2 sources (the check of an FMM evaluation), FP64
        dict(name="direct_velocity_256", kind="direct_velocity", targets=4096, sources=393216),
    ]


def draw(rng):
    kind = rng.choice(["velocity", "step", "poisson", "swe", "gradient", "latlon", "direct_log", "direct_velocity"])
    precision = rng.choice(["fp64", "mixed"])

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def grid(lmin, lmax):
        d, m = rng.choice([(8, 8), (8, 6), (8, 9), (6, 7), (6, 8), (10, 8), (10, 11), (5, 6), (4, 5), (9, 7)])
        return dict(levels=rng.randint(lmin, lmax), d=d, m=m, theta=rng.choice([0.5, 0.6, 0.7]), precision=precision)

    if kind == "velocity":
        return dict(kind=kind, **grid(3, 6))
    if kind == "step":
        members = rng.choice([1, 1, 3, 8, 16])
        return dict(kind=kind, **grid(3, 6 if members == 1 else 4), members=members,
                    dt=float(rng.choice([900, 1800, 3600])))
    if kind == "poisson":
        return dict(kind=kind, **grid(3, 6), targets=rng.choice([0, log_int(100, 20000)]))
    if kind == "swe":
        return dict(kind=kind, **grid(3, 6))
    if kind == "gradient":
        return dict(kind=kind, **grid(3, 5), steps=rng.randint(2, 4), every=rng.choice([1, 2, 4]), dt=900.0)
    if kind == "latlon":
        return dict(kind=kind, rows=log_int(40, 180), d=rng.choice([6, 8, 10]), theta=rng.choice([0.5, 0.7]))
    if kind == "direct_log":
        return dict(kind=kind, sources=log_int(1000, 60000))
    return dict(kind=kind, targets=log_int(100, 20000), sources=log_int(1000, 400000))


# ---------------------------------------------------------------- inputs


def _gpu(v):
    return torch.from_numpy(np.ascontiguousarray(v)).cuda()


def _config(case):
    k = dict(levels=case["levels"], interp_degree=case["d"], leaf_degree=case["m"] - 1, fmm_theta=case["theta"],
             weights=case.get("weights", "clenshaw_curtis"), kernel_eps=EPS, omega=OMEGA, precision=case["precision"],
             delta_t=case.get("dt", 3600.0))
    if case["kind"] == "step":
        k.update(use_graph=True, multi_rhs=case["members"] > 1 and case["precision"] == "mixed")
    return sb.RunConfig(**k)


def _vortices(p, area, seed, count=12):
    """Gaussian vortices of either sign (amplitudes 1e-5 to 3e-5 1/s, widths 0.05 to 0.2 rad), mean removed."""
    rng = np.random.default_rng(seed)
    c = rng.normal(size=(count, 3))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    amp = rng.uniform(1e-5, 3e-5, count) * rng.choice([-1.0, 1.0], count)
    width = rng.uniform(0.05, 0.2, count)
    w = torch.zeros_like(p[0])
    for k in range(count):
        r = torch.acos((p[0] * c[k, 0] + p[1] * c[k, 1] + p[2] * c[k, 2]).clamp(-1.0, 1.0))
        w += amp[k] * torch.exp(-(r / width[k]) ** 2)
    return w - (w * area).sum() / (4 * math.pi)


def _forcing(p, seed):
    """A zero-mean sum of spherical harmonics of degree 1 to 8 with amplitudes N(0, (1+l)^-2)."""
    return _gpu(sb.workloads.random_sh_forcing(*[v.cpu().numpy() for v in p], lmax=8, seed=seed)[0])


def _points(n, seed):
    return [_gpu(v) for v in sb.workloads.random_unit_vectors(n, seed)]


def _fields(case, seed, p, area):
    """The state of a case on the cubed-sphere particles: what its path starts from."""
    kind = case["kind"]
    if kind == "poisson":
        return dict(f=_forcing(p, seed))
    if kind == "swe":
        return dict(vor=_vortices(p, area, seed), div=0.1 * _vortices(p, area, seed + 1),
                    height=5960.0 + 1e7 * _vortices(p, area, seed + 2))
    vor = _vortices(p, area, seed)
    if kind == "step" and case["members"] > 1:
        vor = torch.stack([vor + 0.1 * _vortices(p, area, 1000 * (j + 1) + seed) for j in range(case["members"])])
    return dict(vor=vor)


def _direct_inputs(case, seed):
    n = case["sources"]
    src = _points(n, seed)
    area = torch.full((n,), 4 * math.pi / n, dtype=torch.float64, device="cuda")
    tgt = _points(case["targets"], seed + 1) if "targets" in case else None
    return src, area, _vortices(src, area, seed + 2), tgt


def _latlon_inputs(case, seed):
    lats, lons, x, y, z, area = sb.latlon.cell_grid(180.0 / case["rows"])
    vor, div, _ = sb.latlon.initial_state("tc5", lats, lons)
    p, a = [_gpu(v.ravel()) for v in (x, y, z)], _gpu(area.ravel())
    return (p, a, _gpu(vor.ravel()) + 0.2 * _vortices(p, a, seed), _gpu(div.ravel()) + 0.1 * _vortices(p, a, seed + 1),
            (x, y, z))


def _observations(seed, vor):
    """2,048 points and the values seen there: the field's scale, with noise."""
    values = np.random.default_rng(seed).normal(size=2048)
    return _points(2048, seed + 1), _gpu(values) * vor.square().mean().sqrt()


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("direct_log", "direct_velocity"):
        s["ctx"] = sb.Context(sb.RunConfig(levels=2, interp_degree=4, kernel_eps=EPS))
        s["src"], s["area"], s["vor"], s["tgt"] = _direct_inputs(case, seed)
        return s
    if kind == "latlon":
        ctx = sb.Context(sb.RunConfig(levels=2, interp_degree=case["d"], kernel_eps=EPS, fmm_theta=case["theta"]))
        _, s["area"], s["vor"], s["div"], host = _latlon_inputs(case, seed)
        s["tree"] = ctx.irregular(*host, 4 * (case["d"] + 1) ** 2)
        return s
    s["stream"] = torch.cuda.Stream() if kind == "step" else torch.cuda.current_stream()
    with torch.cuda.stream(s["stream"]):
        ctx = s["ctx"] = sb.Context(_config(case))
    x, y, z, area = [_gpu(v) for v in ctx.spec_points()]
    s["p"], s["area"] = (x, y, z), area
    s.update(_fields(case, seed, s["p"], area))
    torch.cuda.synchronize()
    if kind == "step":
        s["start"] = s["vor"].clone()
        s["vel"] = [torch.zeros_like(s["vor"]) for _ in range(3)]
        if ctx.sizes.N >= 1 << 20:  # a long run of a large field picks its launch shape first
            with torch.cuda.stream(s["stream"]):
                ctx.autotune(area, s["vor"])
    if kind == "poisson" and case["targets"]:
        s["tgt"] = _points(case["targets"], seed + 5)
    if kind == "gradient":
        s["obs"], s["values"] = _observations(seed + 7, s["vor"])
    return s


# ---------------------------------------------------------------- one pass


def run(s):
    case = s["case"]
    kind, ctx = case["kind"], s.get("ctx")
    if kind == "velocity":
        return ctx.bve_velocity(s["area"], s["vor"])
    if kind == "step":
        # every pass steps the same initial state (a device copy first, as the benchmark's repeated steps)
        with torch.cuda.stream(s["stream"]):
            s["vor"].copy_(s["start"])
            if case["members"] > 1:
                ctx.bve_back_rk4_step_ensemble(*s["p"], s["area"], s["vor"], s["vel"])
            else:
                ctx.bve_back_rk4_step(*s["p"], s["area"], s["vor"], s["vel"])
        return [s["vor"]] + s["vel"]
    if kind == "poisson":
        if case["targets"]:
            return ctx.poisson_solve_targets(s["area"], s["f"], *s["tgt"])
        return ctx.poisson_solve(s["area"], s["f"])
    if kind == "swe":
        vel = ctx.swe_velocity(s["area"], s["vor"], s["div"])
        q_part, q_proxy = ctx.upward_pass(s["area"], s["height"])
        phi_part, phi_proxy = ctx.laplacian_interactions(q_part, q_proxy)
        return vel + [ctx.downward_pass(phi_proxy, phi_part)]
    if kind == "gradient":
        return autograd.bve_4dvar(ctx, *s["p"], s["area"], s["vor"], case["steps"], case["every"], s["obs"],
                                  s["values"])
    if kind == "latlon":
        return s["tree"].swe_velocity(s["area"], s["vor"], s["div"])
    if kind == "direct_log":
        return ctx.direct_sum_inv_lap(*s["src"], s["area"], s["vor"])
    return ctx.direct_sum_bve_vel_targets(*s["tgt"], *s["src"], s["area"], s["vor"])


# ---------------------------------------------------------------- what a pass cannot do without


def _tree_pairs(case):
    """Point pairs of one FMM evaluation: sums over the interaction list, leaves hold m^2 points, proxies (d+1)^2."""
    t = sb.HostTree(_config(case))
    kinds = t.interaction_list()[:, 2]
    m2, n = t.sizes.m2, t.sizes.n
    nt = np.where(kinds <= 1, m2, n).astype(np.int64)
    ns = np.where((kinds == 0) | (kinds == 2), m2, n).astype(np.int64)
    return int((nt * ns).sum()), t.sizes.N


def work(case):
    kind = case["kind"]
    if kind == "direct_log":
        n = case["sources"]
        return dict(bytes=8 * 6 * n, flops=FLOP["log"] * n * n)
    if kind == "direct_velocity":
        t, n = case["targets"], case["sources"]
        return dict(bytes=8 * (6 * t + 5 * n), flops=FLOP["vortex"] * t * n)
    if kind == "latlon":
        lats, lons, x, y, z, _ = sb.latlon.cell_grid(180.0 / case["rows"])
        t = sb.HostIrregTree(x, y, z, 4 * (case["d"] + 1) ** 2, case["d"], case["theta"])
        kinds = t.interaction_list()
        held = t.panels()[0][:, 8].astype(np.int64)  # points per panel
        n = t.n
        nt = np.where(kinds[:, 2] <= 1, held[kinds[:, 0]], n)
        ns = np.where((kinds[:, 2] == 0) | (kinds[:, 2] == 2), held[kinds[:, 1]], n)
        return dict(bytes=8 * 9 * t.N, flops=FLOP["swe"] * int((nt * ns).sum()))
    pairs, n = _tree_pairs(case)
    if kind == "velocity":
        return dict(bytes=8 * 5 * n, flops=FLOP["vortex"] * pairs)
    if kind == "step":  # four velocity evaluations; geometry in, state in and out, velocity out
        return dict(bytes=8 * n * (4 + 5 * case["members"]), flops=4 * FLOP["vortex"] * pairs * case["members"])
    if kind == "poisson":
        return dict(bytes=8 * (3 * n + 4 * case["targets"]), flops=FLOP["log"] * pairs)
    if kind == "swe":
        return dict(bytes=8 * 8 * n, flops=(FLOP["swe"] + FLOP["lap"]) * pairs)
    # each step's four evaluations forward, and twice their work in reverse
    return dict(bytes=8 * 6 * n, flops=case["steps"] * 4 * 3 * FLOP["vortex"] * pairs)


def tolerance(case):
    """About four times what a second implementation of the same sums shows.  FP64: an FMM run in
    sequential order differs by up to 2.4e-14 (velocities), the direct velocity by 1.2e-13 (its near
    pairs amplify the rounding of x.y).  Mixed: the vector-unit and matrix-core kernels differ from
    each other and from FP64 by up to 4.5e-7 (6 x 28^2; 5e-8 to 2e-7 at the larger sizes)."""
    if case.get("precision") == "mixed":
        return {"rel": 2e-6}
    return {"rel": {"direct_velocity": 5e-13, "gradient": 1e-12}.get(case["kind"], 1e-13)}


# ---------------------------------------------------------------- the same in plain FP64 torch


class _Sphere:
    """O(N^2) sums over particles X [N][3] and the interpolation on their leaves (node a*m + c, a along xi)."""

    def __init__(self, p, area, levels=0, m=0):
        self.X = torch.stack([v.reshape(-1) for v in p], 1)
        self.area = area.reshape(-1)
        self.n1, self.m = 1 << max(levels - 1, 0), m
        if levels:
            self.cheb = torch.tensor([math.cos(math.pi * i / (m - 1)) for i in range(m)], dtype=torch.float64).cuda()
            self.bw = torch.tensor([(0.5 if i in (0, m - 1) else 1.0) * (-1) ** i for i in range(m)],
                                   dtype=torch.float64).cuda()
            face, i, j = self._cell(self.X.view(-1, m * m, 3).mean(1))[:3]
            self.leaf = torch.empty((6, self.n1, self.n1), dtype=torch.int64, device="cuda")
            self.leaf[face, i, j] = torch.arange(face.numel(), device="cuda")

    @staticmethod
    def _project(p):
        return p / p.norm(dim=-1, keepdim=True)

    @staticmethod
    def rows(targets, fn, n):
        """fn over blocks of target rows whose n-column matrices stay below 1 GiB."""
        step = max(1, (1 << 27) // n)
        return torch.cat([fn(targets[i:i + step]) for i in range(0, targets.shape[0], step)])

    def velocity(self, vor, disp=None, targets=None, differentiable=False):
        y = self.X if disp is None else self._project(self.X + disp)
        src = (-(self.area * vor) / (4 * math.pi)).unsqueeze(1) * y

        def block(t, y, src):
            return torch.linalg.cross(t, (1.0 / ((1.0 - t @ y.T) + EPS)) @ src)

        def one(t):
            if differentiable:
                return torch.utils.checkpoint.checkpoint(block, t, y, src, use_reentrant=False)
            return block(t, y, src)

        return self.rows(self.X if targets is None else targets, one, y.shape[0])

    def psi(self, f, targets=None):
        q = -(self.area * f) / (4 * math.pi)

        def one(t):
            dot = t @ self.X.T
            return torch.where(dot < 1.0 - 1e-15, torch.log1p(-dot.clamp(max=1.0 - 1e-15)), 0.0) @ q

        return self.rows(self.X if targets is None else targets, one, q.numel())

    def swe(self, vor, div, sign):
        qz, qd = [-(self.area * v) / (4 * math.pi) for v in (vor, sign * div)]
        X = self.X

        def one(t):
            dot = t @ X.T
            r = 1.0 / ((1.0 - dot) + EPS)
            rot = torch.linalg.cross(t, r @ (qz.unsqueeze(1) * X))
            return rot + r @ (qd.unsqueeze(1) * X) - t * ((r * dot) @ qd).unsqueeze(1)

        return self.rows(X, one, X.shape[0])

    def laplacian(self, f):
        q, e = self.area * f, LAP_EPS

        def one(x):
            t = x @ self.X.T
            t2 = t * t
            a = math.exp(-1.0 / e) * math.pi ** -1.5 * (2.0 * t * (-1.0 + 3.0 * e + t2))
            b = 2.0 * e * e + 2.0 * t2 * (t2 - 1.0) + e * (7.0 * t2 - 1.0)
            return ((a + (1.0 + torch.erf(t / e)) * torch.exp((t2 - 1.0) / e) / (math.sqrt(e) * math.pi) * b)
                    @ q) / e ** 2.5

        return self.rows(self.X, one, q.numel())

    def _cell(self, p):
        """Face, leaf column and row, and the label coordinates of points [k][3]."""
        x, y, z = p.unbind(-1)
        ax, ay, az = x.abs(), y.abs(), z.abs()
        on_x = (ax >= ay) & (ax >= az)
        on_y = ~on_x & (ay >= ax) & (ay >= az)
        face = torch.where(on_x, torch.where(x >= 0, 0, 2),
                           torch.where(on_y, torch.where(y >= 0, 1, 3), torch.where(z >= 0, 4, 5)))
        at = face.unsqueeze(-1)
        den = torch.stack([x, y, x, y, z, z], -1).gather(-1, at).squeeze(-1)
        xi = torch.atan(torch.stack([y, -x, y, -x, y, -y], -1).gather(-1, at).squeeze(-1) / den)
        eta = torch.atan(torch.stack([z, z, -z, -z, -x, -x], -1).gather(-1, at).squeeze(-1) / den)
        h = (math.pi / 2) / self.n1
        i, j = [((v.detach() + math.pi / 4) / h).floor().long().clamp(0, self.n1 - 1) for v in (xi, eta)]
        return face, i, j, xi, eta

    def interp(self, fields, p):
        """Barycentric interpolation of leaf fields [N] (a list) at points p -> [len(p)][k]."""
        face, i, j, xi, eta = self._cell(p)
        leaf, h = self.leaf[face, i, j], (math.pi / 2) / self.n1

        def weights(t, k):
            node = (0.5 * h) * self.cheb.unsqueeze(0) + (-math.pi / 4 + (k.double() + 0.5) * h).unsqueeze(1)
            gap = t.unsqueeze(1) - node
            r = self.bw.unsqueeze(0) / torch.where(gap.abs() < 1e-15, torch.full_like(gap, 1e-15), gap)
            return r / r.sum(1, keepdim=True)

        wx, we = weights(xi, i), weights(eta, j)
        got = [((f.view(-1, self.m, self.m)[leaf] * we.unsqueeze(1)).sum(2) * wx).sum(1) for f in fields]
        return torch.stack(got, 1)

    def step(self, vor, dt, differentiable=False):
        """One backward Runge-Kutta step: (vorticity after it, velocity before it)."""
        X = self.X
        v = [self.velocity(vor, differentiable=differentiable)]
        for tau in (0.5 * dt, 0.5 * dt, dt):
            p = self._project(X + tau * v[-1])
            v.append(self.velocity(vor + 2 * OMEGA * (X[:, 2] - p[:, 2]), tau * v[-1],
                                   differentiable=differentiable))
        k1 = v[3]
        k2 = self.interp(v[2].unbind(1), self._project(X - 0.5 * dt * k1))
        k3 = self.interp(v[1].unbind(1), self._project(X - 0.5 * dt * k2))
        k4 = self.interp(v[0].unbind(1), self._project(X - dt * k3))
        a = self._project(X - dt / 6.0 * k1)
        a = self._project(a + dt / 3.0 * k2)
        a = self._project(a + dt / 3.0 * k3)
        dep = self._project(a + dt / 6.0 * k4)
        return self.interp([vor], dep)[:, 0] + 2 * OMEGA * (dep[:, 2] - X[:, 2]), v[0]


def _seconds(n, evaluations, targets=None):
    """About what the plain sums take: some 80 bytes of traffic per pair at 3 TB/s."""
    return evaluations * (targets or n) * n * 80 / 3e12


def exact(case, seed):
    kind = case["kind"]
    if kind == "direct_log":
        (x, y, z), area, vor, _ = _direct_inputs(case, seed)
        n, q = case["sources"], area * vor

        def one(i):  # the dot product rounded term by term, the point itself left out
            dot = x[i, None] * x + y[i, None] * y + z[i, None] * z
            term = torch.log((1.0 - dot).clamp(min=1e-300))
            term[torch.arange(i.numel(), device="cuda"), i] = 0.0
            return term @ q

        return _Sphere.rows(torch.arange(n, device="cuda"), one, n) * (-1.0 / (4 * math.pi))
    if kind == "direct_velocity":
        src, area, vor, tgt = _direct_inputs(case, seed)
        return list(_Sphere(src, area).velocity(vor, targets=torch.stack(tgt, 1)).unbind(1))
    if kind == "latlon":
        p, area, vor, div, _ = _latlon_inputs(case, seed)
        return list(_Sphere(p, area).swe(vor, div, -1.0).unbind(1))

    x, y, z, area = [_gpu(v) for v in sb.HostTree(_config(case)).spec_points()]
    n, targets = x.numel(), case.get("targets", 0)
    evaluations = {"velocity": 1, "poisson": 1, "swe": 3, "step": 4 * case.get("members", 1),
                   "gradient": 16 * case.get("steps", 1)}[kind]
    if _seconds(n, evaluations, targets) > 15:
        return None
    given = _fields(case, seed, (x, y, z), area)
    S = _Sphere((x, y, z), area, case["levels"], case["m"])
    shape = x.shape
    if kind == "velocity":
        return [v.reshape(shape) for v in S.velocity(given["vor"].reshape(-1)).unbind(1)]
    if kind == "poisson":
        at = torch.stack(_points(targets, seed + 5), 1) if targets else None
        psi = S.psi(given["f"].reshape(-1), at)
        return psi if targets else psi.reshape(shape)
    if kind == "swe":
        vor, div, height = [given[k].reshape(-1) for k in ("vor", "div", "height")]
        return [v.reshape(shape) for v in S.swe(vor, div, 1.0).unbind(1)] + [S.laplacian(height).reshape(shape)]
    if kind == "step":
        vors = given["vor"].reshape(case["members"], -1)
        got = [S.step(v, case["dt"]) for v in vors]
        out = [torch.stack([g[0] for g in got])] + [torch.stack([g[1][:, c] for g in got]) for c in range(3)]
        return [v.reshape(given["vor"].shape) for v in out]
    obs, values = _observations(seed + 7, given["vor"])
    w = given["vor"].reshape(-1).clone().requires_grad_(True)
    v = w
    for _ in range(case["steps"]):
        v = S.step(v, case["dt"], differentiable=True)[0]
    loss = 0.5 * ((S.interp([v], torch.stack(obs, 1))[:, 0] - values) ** 2).sum()
    loss.backward()
    return [loss.detach(), w.grad.reshape(shape)]
