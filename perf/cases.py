"""The work that programs have naga_amd do, as measurable cases.

A case is a dict of plain values.  ``listed()`` names the standing ones,
``draw(rng)`` makes further ones of the same ranges, ``prepare(case, seed)``
builds what a program holds before the call (nodes, engines with their set-up
done, device arrays), ``run(state)`` is one pass through the public entry
points, ``work(case)`` the bytes and operations a pass cannot do without, and
``exact(case, seed)`` the pass's results in 64 bits, computed with plain torch.

Kinds of cases:

* ``step``     an engine with its domain advanced by some steps, then read;
* ``batch``    many D2Q9 scenes advanced together, then read;
* ``solve``    a whole solve of a node cloud: set-up, pulse, steps, result;
* ``knn``      exact nearest neighbours on device arrays;
* ``weights``  the divergence operator's stencils and weights for a cloud.
"""
from __future__ import annotations

import itertools
import math

import numpy as np
import torch

import naga_amd
from naga_amd import workloads

TAU = 0.6


# ------------------------------------------------------------------- cases
def listed() -> list:
    step = dict(kind="step", shape="box", rbf=1, k_min=0)
    return [
        # the headline scene: the unit cube at h = 0.01, one frame of 50 steps
        dict(step, name="cube_1m", lattice=27, h=0.01, k=32, steps=50),
        # the same scene at twice the spacing: a mid-size interactive run
        dict(step, name="cube_133k", lattice=27, h=0.02, k=32, steps=100),
        # a small cube, where a step is short kernels one after another
        dict(step, name="cube_9k", lattice=27, h=0.05, k=32, steps=200),
        # a narrower stencil than the default one
        dict(step, name="cube_133k_k24", lattice=27, h=0.02, k=24, steps=50),
        # the irregular domain: cube minus a refined sphere, widths 24-48
        dict(step, name="shell_2m", lattice=27, shape="sphere", h=0.008, k=48, k_min=24, steps=20),
        # the plain 2D scene of 10,201 nodes
        dict(step, name="square_10k", lattice=9, h=0.01, k=16, steps=250),
        # a fine 2D scene of a million nodes
        dict(step, name="square_1m", lattice=9, h=0.001, k=16, steps=100),
        # 256 small 2D scenes with obstacles stepped together
        dict(kind="batch", name="batch_256", scenes=256, n_lo=2000, n_hi=50000, steps=100),
        # whole solves of a node cloud, as a serving loop or a sweep runs them:
        # 3D with the reference's multiquadric stencils, 2D with obstacles
        dict(kind="solve", name="solve_cube", lattice=27, shape="box", h=0.02, k=32, k_min=0,
             rbf=0, steps=20),
        dict(kind="solve", name="solve_square", lattice=9, shape="circles", h=0.005, k=16,
             k_min=0, rbf=1, steps=50),
        # neighbour search over a million nodes, without allocation
        dict(kind="knn", name="knn_1m", cloud="nodes", dims=3, n=1030301, queries=1030301, k=32),
        # the divergence operator of a 3D cloud, returned to the host
        dict(kind="weights", name="weights_64k", cloud="nodes", dims=3, n=64000, k=32, rbf=1),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["step", "step", "step", "solve", "batch", "knn", "weights"])
    if kind == "batch":
        lo = int(_log_uniform(rng, 2e3, 1e4))
        return dict(kind="batch", scenes=rng.randint(3, 96), n_lo=lo, n_hi=int(lo * rng.uniform(1.5, 5)),
                    steps=rng.randint(20, 100))
    if kind in ("knn", "weights"):
        D, k = rng.choice([2, 3]), rng.randint(8, 48)
        cloud = rng.choice(["nodes", "random"])
        if kind == "knn":
            n = int(_log_uniform(rng, 5e3, 1e6))
            return dict(kind=kind, cloud=cloud, dims=D, n=n, queries=int(_log_uniform(rng, 1e3, n)),
                        k=k)
        return dict(kind=kind, cloud="nodes", dims=D, n=int(_log_uniform(rng, 2e3, 6.4e4)),
                    k=max(k, 12), rbf=rng.choice([0, 1]))
    lattice = rng.choice([9, 27])
    D = 2 if lattice == 9 else 3
    n = _log_uniform(rng, 2e3 if D == 2 else 5e3, 1e6 if kind == "step" else 1.5e5)
    case = dict(kind=kind, lattice=lattice, shape="box", h=1.0 / (n ** (1.0 / D) - 1.0),
                k=rng.randint(12, 24) if D == 2 else rng.choice([16, 20, 24, 32, 32, 48]), k_min=0,
                rbf=1, steps=max(10, min(200, int(2e7 / n))) if kind == "step" else rng.randint(5, 50))
    if D == 2 and rng.random() < 0.4:
        case["shape"] = "circles"
    elif D == 3 and case["h"] <= 0.05 and rng.random() < 0.3:
        case.update(shape="sphere", k=48, k_min=24)
    elif rng.random() < 0.3:
        case.update(k=32, rbf=0)  # the reference's stencils: k = 32, multiquadric
    return case


# ----------------------------------------------------------------- inputs
def _nodes(case, seed):
    """The scene's nodes in the provider's order, their places from the seed.
    The obstacles belong to the case, and with them the number of nodes: the
    seed then moves the bulk nodes by up to 0.05 of the finest spacing."""
    D, h = (2 if case["lattice"] == 9 else 3), case["h"]
    layer = min(8 * h, 0.1)
    if case["shape"] == "box":
        return naga_amd.UniformGridProvider([0] * D, [1] * D, h, layer, 0.5, jitter=0.25,
                                            seed=seed).get()
    if case["shape"] == "sphere":  # refined twice within 0.05 of its surface
        nodes = naga_amd.ObstacleGridProvider([0] * 3, [1] * 3, h, [([0.5] * 3, 0.15)], layer, 0.5,
                                              jitter=0.1, refine_width=0.05).get()
    else:
        rng = np.random.default_rng(7)
        circles = [(rng.uniform(0.15, 0.85, 2).tolist(), float(rng.uniform(0.03, 0.1)))
                   for _ in range(3)]
        nodes = naga_amd.ObstacleGridProvider([0] * 2, [1] * 2, h, circles, layer, 0.5,
                                              jitter=0.2, immersed_layer_thickness=3 * h,
                                              immersed_absorption_rate=0.5).get()
    n, fine = nodes.num_bulk_points, h * (0.5 if case["shape"] == "sphere" else 1.0)
    nodes.points[:n] += 0.05 * fine * np.random.default_rng(seed).uniform(-1, 1, (n, D)).astype(
        np.float32)
    return nodes


def _pulse(case, seed):
    """Centre, amplitude and width of the initial pulse."""
    D = 2 if case["lattice"] == 9 else 3
    rng = np.random.default_rng([seed, 1])
    return [float(rng.uniform(0.2, 0.3))] + rng.uniform(0.35, 0.65, D - 1).tolist(), 1e-3, 0.05


def _time_step(case):
    return 0.4 * case["h"] * (0.5 if case["shape"] == "sphere" else 1.0)


def _engine(case):
    eng = naga_amd.SimulationEngine(lattice=case["lattice"], k=case["k"], rbf=case["rbf"],
                                    k_min=case["k_min"])
    p = naga_amd.problem_parameters(case["lattice"], TAU, _time_step(case))
    eng.set_problem_parameters(p["nu"], 1.0, p["dt"], p["c"])
    return eng


def _cloud(case, n, seed):
    """n points: scene nodes in the provider's order, or uniform random ones."""
    D = case["dims"]
    if case["cloud"] == "random":
        return np.random.default_rng(seed).random((n, D), dtype=np.float32)
    side = round(n ** (1.0 / D))
    while (side ** D) < n:
        side += 1
    h = 1.0 / (side - 1)
    pts = naga_amd.UniformGridProvider([0] * D, [1] * D, h, 0.1, 0.5, jitter=0.25,
                                       seed=seed).get().points
    return np.ascontiguousarray(pts[:n])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "solve"):
        nodes, pulse = _nodes(case, seed), _pulse(case, seed)
        eng = _engine(case)
        if kind == "step":
            eng.init_domain(nodes)
            eng.set_initial_pulse(*pulse)
        return dict(case=case, engine=eng, nodes=nodes, pulse=pulse)
    if kind == "batch":
        scenes = workloads.batched_scenes(case["scenes"], case["n_lo"], case["n_hi"])
        rng = np.random.default_rng(seed)
        engines = []
        for scene in scenes:  # the scenes belong to the case, their pulses to the seed
            scene.pulse = rng.uniform(0.2, 0.8, 2).tolist()
            engines.append(workloads.batched_engine(scene)[0])
        return dict(case=case, engines=engines, batch=naga_amd.SceneBatch(engines))
    if kind == "weights":
        return dict(case=case, points=_cloud(case, case["n"], seed))
    ref = _cloud(case, case["n"], seed)
    query = ref if case["queries"] == case["n"] else _cloud(case, case["queries"], seed + 1)
    dev = torch.device("cuda")
    ref_d = torch.from_numpy(ref).to(dev)
    return dict(case=case, ref=ref_d,
                query=ref_d if query is ref else torch.from_numpy(query).to(dev),
                d2=torch.empty(case["queries"], case["k"], dtype=torch.float32, device=dev),
                idx=torch.empty(case["queries"], case["k"], dtype=torch.int32, device=dev))


# -------------------------------------------------------------------- pass
def _fields(eng):
    """Density, its perturbation (in the state's precision) and velocity."""
    m = eng.macroscopic(fresh=True)
    return dict(rho=m["rho"], drho=m["drho"].astype(np.float32), u=m["u"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        state["engine"].step_forward(case["steps"])
        return _fields(state["engine"])
    if kind == "solve":
        eng = state["engine"]
        eng.init_domain(state["nodes"])
        eng.set_initial_pulse(*state["pulse"])
        eng.step_forward(case["steps"])
        return _fields(eng)
    if kind == "batch":
        state["batch"].step_forward(case["steps"])
        each = [_fields(e) for e in state["engines"]]
        return {f: np.concatenate([m[f] for m in each], axis=-1) for f in ("rho", "drho", "u")}
    if kind == "weights":
        op = naga_amd.DivergenceOperator.create(state["points"], k=case["k"], rbf=case["rbf"])
        return dict(weights=op.weights(), indices=op.support_indices().view(np.int32))
    ref, query, d2, idx = (state[v] for v in ("ref", "query", "d2", "idx"))
    status = naga_amd.load().naga_knn_noalloc(
        ref.data_ptr(), ref.shape[0], query.data_ptr(), query.shape[0], case["dims"], case["k"],
        d2.data_ptr(), idx.data_ptr(), torch.cuda.current_stream().cuda_stream)
    if status:
        raise RuntimeError(naga_amd.load().naga_last_error().decode())
    return dict(d2=d2, idx=idx)


# -------------------------------------------------------------------- work
def _node_count(case):
    if case["kind"] == "batch":  # mean of the log-uniform sizes
        lo, hi = case["n_lo"], case["n_hi"]
        return case["scenes"] * (hi - lo) / math.log(hi / lo)
    n = (1.0 / case["h"] + 1.0) ** (2 if case["lattice"] == 9 else 3)
    if case["shape"] == "sphere":  # the shell holds eight times as many
        n += 7 * 4 * math.pi / 3 * (0.2 ** 3 - 0.15 ** 3) / case["h"] ** 3
    return n


def _step_work(Q, D, k):
    """FP32 state and records, 32-bit indices: the collision, filter and
    boundary passes and four RK4 stages of one node."""
    return (76 * Q + 8 * k + 16 * k * (1 + D),
            4 * k * (2 * Q + Q * (2 * D - 1)) + 3 * k * Q + 60 * Q)


def _solve_flops(k, D):
    """One node's RBF system: its entries, D quadrature right-hand sides over
    4^D points, the factorisation and the solves."""
    n = k + D + 1
    return 8 * k * k + 4 ** D * k * (10 + 2 * D) + 2 * n ** 3 / 3 + 2 * D * n * n


def work(case):
    kind = case["kind"]
    if kind == "knn":
        n, q, D, k = case["n"], case["queries"], case["dims"], case["k"]
        return dict(bytes=4 * D * (n + (q if q != n else 0)) + 8 * q * k, flops=3 * D * q * k)
    if kind == "weights":
        n, D, k = case["n"], case["dims"], case["k"]
        return dict(bytes=4 * D * n + n * k * (4 + 8 * D), flops=n * _solve_flops(k, D))
    Q = 9 if kind == "batch" else case["lattice"]
    D = 2 if Q == 9 else 3
    k = 18 if kind == "batch" else 1.2 * case["k_min"] if case["k_min"] else case["k"]
    n = _node_count(case)
    b, f = _step_work(Q, D, k)
    read = n * (8 + 4 * D)  # the fields read at the end
    bytes_, flops = n * case["steps"] * b + read, n * case["steps"] * f
    if kind == "solve":
        bytes_ += n * (4 * D + k * (4 + 4 * (1 + D) + 8) + 4 * Q)
        flops += n * _solve_flops(k, D)
    return dict(bytes=bytes_, flops=flops)


# ------------------------------------------------------------------- exact
# The method in 64 bits with plain torch: stencils by comparing every pair,
# weights by dense solves, and a step written over whole arrays.
_VEL = {
    9: [(0, 0), (-1, 1), (-1, 0), (-1, -1), (0, -1), (1, -1), (1, 0), (1, 1), (0, 1)],
    27: [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1),
         (1, 1, 0), (-1, 1, 0), (1, -1, 0), (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1),
         (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1), (0, -1, -1), (1, 1, 1), (-1, 1, 1),
         (1, -1, 1), (-1, -1, 1), (1, 1, -1), (-1, 1, -1), (1, -1, -1), (-1, -1, -1)],
}


def _knn64(points, query, k):
    """Exact neighbours: the FP32 distance keys in order, ties by index."""
    n, D = points.shape
    out = []
    ids = torch.arange(n, device=points.device)
    for q in query.split(max(1, int(1e8 / n))):
        d2 = (q[:, None, 0] - points[None, :, 0]) ** 2
        for d in range(1, D):
            d2 = (q[:, None, d] - points[None, :, d]) ** 2 + d2
        key = (d2.view(torch.int32).long() << 32) | ids
        out.append(torch.topk(key, k, dim=1, largest=False, sorted=True).values)
    key = torch.cat(out)
    return (key >> 32).int().view(torch.float32).double(), key & 0xFFFFFFFF


def _phi(r2, rbf, spacing):
    return r2 * r2.sqrt() if rbf == 1 else (r2 + (0.1 * spacing) ** 2).sqrt()


def _rbf_system(x, rbf, spacing):
    """[[Phi, P], [P^T, 0]] for stencils x [n, k, D] relative to their query."""
    n, k, D = x.shape
    A = torch.zeros(n, k + D + 1, k + D + 1, dtype=torch.float64, device=x.device)
    A[:, :k, :k] = _phi(((x[:, :, None] - x[:, None]) ** 2).sum(-1), rbf, spacing[:, None, None])
    A[:, :k, k] = A[:, k, :k] = 1.0
    A[:, :k, k + 1:] = x
    A[:, k + 1:, :k] = x.transpose(1, 2)
    return A


def _rbf_rhs(x, xq, rbf, spacing):
    """Basis values at xq [n, q, D]: [n, q, k + D + 1]."""
    r2 = ((x[:, None] - xq[:, :, None]) ** 2).sum(-1)
    return torch.cat([_phi(r2, rbf, spacing[:, None, None]), torch.ones_like(xq[:, :, :1]), xq], 2)


def _quadrature(D, device):
    """Points and weights of the ball's product rule (unit radius): four
    radial Gauss-Legendre nodes, four equal steps of each angle."""
    xr, wr = [0.339981, -0.339981, 0.861136, -0.861136], [0.652145, 0.652145, 0.347855, 0.347855]
    pts, wts = [], []
    for q in range(4 ** D):
        r, th = (xr[q % 4] + 1) / 2, (q // 4 % 4) * math.pi / 2
        ph = (q // 16) * math.pi / 4 + math.pi / 8
        pts.append([r * math.cos(th), r * math.sin(th)] if D == 2 else
                   [r * math.sin(ph) * math.cos(th), r * math.sin(ph) * math.sin(th),
                    r * math.cos(ph)])
        wts.append(wr[q % 4] / 2 * (math.pi / 2) * (math.pi / 4 if D == 3 else 1.0))
    return (torch.tensor(pts, dtype=torch.float64, device=device),
            torch.tensor(wts, dtype=torch.float64, device=device))


def _divergence_weights64(points, idx, d2, rbf):
    """W [n, k, D]: the kernel-weighted quadrature of the RBF interpolant."""
    n, k = idx.shape
    D = points.shape[1]
    p = points.double()
    unit, qw = _quadrature(D, points.device)
    near = d2[:, 1].sqrt()
    hbar = torch.cat([b.mean().expand(b.numel()) for b in near.split(16384)])
    out = []
    for i in torch.arange(n, device=points.device).split(16384):
        # relative to the query and in units of its nearest distance
        scale = near[i]
        x = (p[idx[i]] - p[i][:, None]) / scale[:, None, None]
        spacing = hbar[i] / scale if rbf == 0 else torch.ones_like(scale)
        delta = 0.05
        xq = (unit * delta).expand(len(i), -1, -1)
        r = xq.norm(dim=2)
        g = torch.where(2 * r / delta < 1, r * (2 * delta - 3 * r), (delta - r) ** 2)
        c = (240 / 7 if D == 2 else 48) / (math.pi * delta ** (3 + D))
        jac = r if D == 2 else r * xq[:, :, :2].norm(dim=2)
        aw = (c * g * jac / r * qw * delta)[:, :, None] * xq
        b = (aw[:, :, None] * _rbf_rhs(x, xq, rbf, spacing)[:, :, :, None]).sum(1)
        w = torch.linalg.solve(_rbf_system(x, rbf, spacing), b)[:, :k]
        w[:, 0] += aw.sum(1)
        out.append(w / scale[:, None, None])
    return torch.cat(out)


_Q2 = lambda t: 3 * t * t - 2  # noqa: E731


def _basis27(x, y, z):
    """The cascade's lattice polynomials, conserved moments first."""
    qx, qy, qz = _Q2(x), _Q2(y), _Q2(z)
    return torch.stack([
        torch.ones_like(x), x, y, z, x * y, x * z, y * z, x * x - y * y,
        x * x + y * y - 2 * z * z, x * x + y * y + z * z - 2, x * (3 * (y * y + z * z) - 4),
        y * (3 * (x * x + z * z) - 4), z * (3 * (x * x + y * y) - 4), x * (y * y - z * z),
        y * (x * x - z * z), z * (x * x - y * y), x * y * z, (qx * qy + qx * qz + qy * qz) / 3,
        (qx * qy + qx * qz - 2 * qy * qz) / 3, qx * (y * y - z * z), y * z * qx, x * z * qy,
        x * y * qz, x * qy * qz, y * qx * qz, z * qx * qy, qx * qy * qz], -1)


class _Exact:
    """One scene of the method in 64 bits."""

    def __init__(self, case, nodes, pulse):
        dev, Q = torch.device("cuda"), case["lattice"]
        D = 2 if Q == 9 else 3
        k, rbf, h = case["k"], case["rbf"], case["h"]
        f64 = dict(dtype=torch.float64, device=dev)
        pts = torch.from_numpy(np.ascontiguousarray(nodes.points, np.float32)).to(dev)
        self.Q, self.D = Q, D
        self.nb, self.nl = nodes.num_bulk_points, nodes.num_layer_points
        self.nf = self.nb + self.nl
        self.c = torch.tensor(_VEL[Q], **f64)
        n2 = (self.c ** 2).sum(1)
        self.w = (4 / 9 if D == 2 else 8 / 27) / torch.tensor([1.0, 4.0, 16.0, 64.0], **f64)[n2.long()]
        self.opp = torch.tensor([_VEL[Q].index(tuple(-v for v in c)) for c in _VEL[Q]], device=dev)
        p = naga_amd.problem_parameters(Q, TAU, _time_step(case))
        self.dt, self.nu = p["dt"], p["nu"]
        d2, idx = _knn64(pts, pts, k)
        W = _divergence_weights64(pts, idx, d2, rbf)[: self.nf]
        self.idx = idx[: self.nf]
        self.cw = (W.reshape(-1, D) @ self.c.T).reshape(self.nf, k, Q)
        p64 = pts.double()
        r2 = ((p64[self.idx] - p64[: self.nf, None]) ** 2).sum(2)
        wf = torch.exp(-0.5 * r2 / (h / 2.5) ** 2)
        self.wf = 0.75 * wf / wf.sum(1, keepdim=True)
        _, self.bidx = _knn64(pts[: self.nf], pts[self.nf:], k)
        x = p64[self.bidx] - p64[self.nf:, None]
        sp = torch.full((len(x),), h, **f64) / h
        b = _rbf_rhs(x / h, torch.zeros_like(x[:, :1]), rbf, sp)
        self.bw = torch.linalg.solve(_rbf_system(x / h, rbf, sp), b.transpose(1, 2))[:, :k]
        nrm = torch.from_numpy(np.ascontiguousarray(nodes.boundary_normals)).to(dev).double()
        into = nrm @ self.c.T > 0
        self.bounce = torch.where(into, self.opp, torch.arange(Q, device=dev))
        self.sigma = torch.from_numpy(np.ascontiguousarray(nodes.layer_absorption)).to(dev).double()
        centre, amp, width = pulse
        r2 = ((p64 - torch.tensor(centre, **f64)) ** 2).sum(1)
        self.g = (amp * torch.exp(-r2 / (2 * width ** 2)))[:, None] * self.w
        self.prev = torch.zeros(len(pts), Q, **f64)
        self.q1 = torch.zeros(len(pts), Q, **f64)
        if Q == 27:
            self.K = _basis27(*self.c.T)
            monos = list(itertools.product(range(3), repeat=3))
            V = torch.stack([(self.c ** torch.tensor(m, **f64)).prod(1) for m in monos], 1)
            mean = [math.prod((1.0, 0.0, 1 / 3)[e] for e in m) for m in monos]
            self.eq = torch.tensor(mean, **f64) @ torch.linalg.solve(V, self.K)
            rate = [0.0] * 4 + [1 / (3 * self.nu + 0.5)] * 6 + [
                float(np.float32(v)) for v, m in ((1.5, 3), (1.83, 3), (1.4, 1), (1.61, 1),
                                                  (1.98, 5), (1.74, 4)) for _ in range(m)]
            self.rate = torch.tensor(rate, **f64) / self.dt

    def moments(self, g):
        rt = g.sum(1)
        return rt, (g @ self.c) / (1 + rt)[:, None]

    def collide(self, f, rho, u):
        if self.Q == 27:
            P = _basis27(*(self.c[None] - u[:, None]).unbind(-1))  # [n, a, j]
            C = (f[:, :, None] * P).sum(1)
            B = (P.transpose(1, 2).reshape(-1, 27) @ self.K).reshape(-1, 27, 27)
            rhs = rho[:, None] * self.eq - C
            k = torch.zeros_like(C)
            for j in range(4, 27):
                k[:, j] = (rhs[:, j] - (B[:, j, 4:j] * k[:, 4:j]).sum(1)) / B[:, j, j]
            return self.dt * (k * self.rate) @ self.K.T
        r0, nw, we, sw, so, se, ea, ne, no = f.unbind(1)
        ux, uy = u.unbind(1)
        xx, yy, i, om = ux * ux, uy * uy, 1 / self.dt, 1 / (3 * self.nu + 0.5 * self.dt)
        axis, diag = ea + no + so + we, se + sw + ne + nw
        k3 = i * (rho * (xx + yy) - axis - 2 * (diag - rho / 3)) / 12
        k4 = om * (no + so - ea - we + rho * (xx - yy)) / 4
        k5 = om * (ne + sw - nw - se + rho * ux * uy) / 4
        k6 = (-i * ((se + sw - ne - nw - 2 * xx * uy * rho + uy * (rho - no - so - r0)) / 4
                    + ux / 2 * (ne - nw - se + sw)) - uy / 2 * (-3 * k3 - k4) - 2 * ux * k5)
        k7 = (-i * ((sw + nw - se - ne - 2 * ux * yy * rho + ux * (rho - we - ea - r0)) / 4
                    + uy / 2 * (ne + sw - se - nw)) - ux / 2 * (-3 * k3 + k4) - 2 * uy * k5)
        k8 = (i / 4 * (rho / 9 - diag + 2 * (ux * (ne - nw + se - sw) + uy * (ne + nw - se - sw))
                       + 4 * ux * uy * (nw - ne + se - sw) - xx * (no + ne + nw + so + se + sw)
                       + yy * (3 * xx * rho - ea - ne - nw - se - sw - we))
              - 2 * k3 - 2 * ux * k7 - 2 * uy * k6 + 4 * ux * uy * k5
              - (1.5 * k3 - k4 / 2) * (xx + yy))
        x, y = self.c.T
        cols = torch.stack([_Q2(x) + _Q2(y), x * x - y * y, -x * y, -y * _Q2(x), -x * _Q2(y),
                            _Q2(x) * _Q2(y)])
        return self.dt * torch.stack([k3, k4, k5, k6, k7, k8], 1) @ cols

    def rate_of(self, g):
        return -(self.cw * g[self.idx]).sum(1)

    def boundary(self, g):
        return (self.bw * g[self.bidx]).sum(1)

    def step(self):
        nf, nb, nl, hdt = self.nf, self.nb, self.nl, self.dt / 2
        g = self.g
        rt, u = self.moments(g)
        df = self.collide(self.w + g, 1 + rt, u)
        uc, uu = u @ self.c.T, (u * u).sum(1, keepdim=True)
        eq = self.w * (rt[:, None] + (1 + rt)[:, None] * (3 * uc + 4.5 * uc * uc - uu))
        # absorbing layer
        q1 = (eq + self.prev) * hdt
        q2 = (q1 + self.q1) * hdt
        self.prev, self.q1 = eq, q1
        s = g.clone()
        s[:nf] += df[:nf]
        if nl:
            sig, lay = self.sigma[:, None], slice(nb, nf)
            s[lay] -= sig * (3 * eq[lay] + 3 * sig * q1[lay] + sig * sig * q2[lay])
            field = torch.zeros_like(g)
            field[lay] = (-2 * sig * (q1[:nl] - q1[lay].mean(0))
                          + sig * sig * (q2[:nl] - q2[lay].mean(0)))
            s[:nf] -= self.rate_of(field)
        # boundary: interpolated before the collision, its own increment added
        s[nf:] = df[nf:] + self.boundary(s[:nf] - df[:nf])
        # selective filter, bounce-back
        y = torch.empty_like(g)
        y[:nf] = s[:nf] + (self.wf[:, :, None] * (s[self.idx] - s[:nf, None])).sum(1)
        y[nf:] = s[nf:].gather(1, self.bounce)
        # classic RK4 of the streaming equation
        rates, t = [], y
        for a in (0.5, 0.5, 1.0, None):
            rates.append(self.rate_of(t))
            if a:
                t = y.clone()
                t[:nf] += a * self.dt * rates[-1]
        y[:nf] += self.dt / 6 * (rates[0] + 2 * rates[1] + 2 * rates[2] + rates[3])
        y[nf:] = self.boundary(y)
        self.g = y

    def fields(self):
        rt, u = self.moments(self.g)
        return dict(rho=1 + rt, drho=rt, u=u.T.contiguous())


def exact(case, seed):
    """The pass's results in 64 bits; None where they would take too long
    (batches, variable stencil widths, clouds too large to compare by pairs)."""
    if case["kind"] == "weights":
        pts = torch.from_numpy(_cloud(case, case["n"], seed)).cuda()
        d2, idx = _knn64(pts, pts, case["k"])
        return dict(weights=_divergence_weights64(pts, idx, d2, case["rbf"]), indices=None)
    if case["kind"] == "knn":
        if case["n"] * case["queries"] > 2e10:
            return None
        ref = _cloud(case, case["n"], seed)
        query = ref if case["queries"] == case["n"] else _cloud(case, case["queries"], seed + 1)
        ref, query = torch.from_numpy(ref).cuda(), torch.from_numpy(query).cuda()
        _, idx = _knn64(ref, query, case["k"])
        d2 = ((query.double()[:, None] - ref.double()[idx]) ** 2).sum(2)
        return dict(d2=d2, idx=None)
    if case["kind"] == "batch" or case["k_min"] or _node_count(case) > 1.5e5:
        return None
    scene = _Exact(case, _nodes(case, seed), _pulse(case, seed))
    for _ in range(case["steps"]):
        scene.step()
    return scene.fields()
