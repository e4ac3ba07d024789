"""Workloads of the EIT framework for timing and comparing builds.

A case is one call a program makes through the public Python mirror or the C ABI: a
forward solve (``EIT.solve``), a Gauss-Newton step (``Solver.solve_absolute``), a batch
of uneven jobs (``BatchSolver.solve_absolute``), a differential reconstruction
(``Solver.solve_differential``), a gradient or an evaluation of the learned start's
network (``Mlp``), and a Krylov solve on a caller's matrix (``mpf_pcg_solve``).

Meshes are the ring meshes of the benchmark, electrodes cover about a quarter of the
circumference, the drive and measurement patterns are adjacent, conductivities are
seeded ellipse phantoms and measured voltages carry 60 dB noise.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from mpflow_amd import capi
from mpflow_amd.eit import EIT, Batch, BatchSolver, Context, SolveOptions, Solver, circular_ports
from mpflow_amd.learned import Mlp
from mpflow_amd.mesh import boundary_edges, promote_p2, ring_mesh
from mpflow_amd.phantom import ellipse_phantom

LAMBDA = 1e-3
CURRENT = 1e-3
NET_SEED = 5
CONTACT = 0.01        # contact impedance of the coupled complete electrode model


# ------------------------------------------------------------------------------------
# cases
# ------------------------------------------------------------------------------------
def _eit(kind, rings, ports, harmonics, frames, p2=False, contact=0.0, two_level=True):
    return dict(kind=kind, rings=rings, ports=ports, harmonics=harmonics, frames=frames, p2=p2,
                contact=contact, two_level=two_level)


def listed():
    return [
        # the smallest call: one 2D forward solve as the reference runs it (diagonal
        # preconditioner, FP32, reference stop rule), e.g. inside somebody's own optimiser
        dict(_eit("forward", 16, 16, 1, 1, two_level=False), name="forward_2d_1"),
        # training data and simulated measurements: many phantoms per launch
        dict(_eit("forward", 40, 32, 5, 64, contact=CONTACT), name="forward_p1_64"),
        # complex conductivity (multi-frequency EIT), 2.5D
        dict(_eit("complex", 20, 16, 3, 2, two_level=False), name="complex_p1_2"),
        # one frame arrives and is reconstructed: latency of one Gauss-Newton step
        dict(_eit("step", 40, 32, 5, 1), name="step_p1_1"),
        # batched reconstruction on the small mesh (offline processing of a recording)
        dict(_eit("step", 40, 32, 5, 64, contact=CONTACT), name="step_p1_64"),
        # the fine quadratic mesh, one frame at a time
        dict(_eit("step", 82, 32, 5, 1, p2=True, contact=CONTACT), name="step_p2_1"),
        # the headline workload: the fine quadratic mesh, frames batched
        dict(_eit("step", 82, 32, 5, 32, p2=True, contact=CONTACT), name="step_p2_32"),
        # independent jobs with their own meshes, electrode and harmonic counts
        dict(kind="batch", jobs=16, first=0, name="batch_16"),
        # time-difference imaging: every frame against one prepared linearisation
        dict(_eit("differential", 40, 32, 5, 64), name="differential_64"),
        # the learned start: the gradient of a large batch (forward, backward, the gradients
        # read back for the caller's own optimiser) and the evaluation of a batch of frames
        dict(kind="gradient", inputs=1024, hidden=2048, layers=3, outputs=9600, batch=4096, name="gradient_4096"),
        dict(kind="infer", inputs=1024, hidden=2048, layers=3, outputs=9600, batch=64, name="infer_64"),
        # ConjugateGradient::solve on a caller's SparseMatrix
        dict(kind="pcg", rings=40, ports=32, columns=32, name="pcg_p1_32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "complex", "step", "step", "step", "batch", "differential",
                       "gradient", "infer", "pcg"])
    ports = rng.choice([8, 12, 16, 16, 20, 24, 32, 32])
    lo = max(12, int(0.7 * ports) + 3)
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 20), first=rng.randint(0, 200))
    if kind in ("gradient", "infer"):
        return dict(kind=kind, inputs=16 * rng.randint(4, 64), hidden=_log(rng, 128, 2048), layers=rng.randint(1, 3),
                    outputs=_log(rng, 600, 9600), batch=_log(rng, 1, 256) if kind == "infer" else _log(rng, 32, 4096))
    if kind == "pcg":
        return dict(kind=kind, rings=_log(rng, lo, 60), ports=ports, columns=rng.randint(1, ports))
    if kind == "complex":
        return _eit(kind, _log(rng, lo, 32), ports, rng.randint(1, 4), rng.randint(1, 4), two_level=False)
    p2 = kind == "step" and rng.random() < 0.4
    rings = _log(rng, lo, 82 if p2 or kind == "forward" else 60)
    harmonics = rng.randint(1, 5)
    # frames up to 64 or what keeps the case below the largest listed one
    nodes = (12 if p2 else 3) * rings * (rings + 1)
    most = int(min(64, 81180 * 5 * 32 * 0.8 / (nodes * harmonics)))
    two_level = kind != "forward" or rings > 40 or rng.random() < 0.7
    if not two_level:
        most = min(most, 4)
    contact = CONTACT if harmonics > 1 and kind != "differential" and rng.random() < 0.6 else 0.0
    return _eit(kind, rings, ports, harmonics, _log(rng, 1, max(1, most)), p2, contact, two_level)


# ------------------------------------------------------------------------------------
# problems
# ------------------------------------------------------------------------------------
def _width(ports):
    return 1.6 / ports


@functools.lru_cache(maxsize=None)
def _mesh(rings, ports, p2):
    """nodes, elements, boundary edges, electrode edges and the adjacent pattern."""
    nodes, el = ring_mesh(rings, ports, _width(ports))
    if p2:
        nodes, el = promote_p2(nodes, el)
    bd = boundary_edges(el)
    pt = circular_ports(nodes, el, bd, ports, _width(ports))
    pat = np.eye(ports) - np.roll(np.eye(ports), 1, axis=0)
    return nodes, el, bd, pt, pat


def _height(harmonics):
    return (1.0, 1.0) if harmonics == 1 else (0.4, 0.1)


def _job(j):
    """Job j of the uneven multi-job workload: 2000 to 40000 elements, 16 or 32
    electrodes, 1 to 5 harmonics."""
    g = np.random.default_rng(1000003 * 4 + j)
    rings = int(round(math.sqrt((2000 + 38000 * g.random()) / 6.0)))
    return _eit("step", rings, 16 if g.random() < 0.5 else 32, int(g.integers(1, 6)), 1)


def _model(case, ctx):
    nodes, el, bd, pt, pat = _mesh(case["rings"], case["ports"], case["p2"])
    h, hp = _height(case["harmonics"])
    step = case["kind"] in ("step", "differential")
    return EIT(nodes, el, bd, pt, pat, pat, CURRENT, 1.0, case["harmonics"], h, hp,
               jacobian_exact=step or case["contact"] > 0.0, frames=case["frames"], ctx=ctx,
               contact_impedance=case["contact"], cem="coupled", complex_gamma=case["kind"] == "complex")


def _phantoms(case, seed, frames=None):
    """frames x elements conductivities."""
    nodes, el, _, _, _ = _mesh(case["rings"], case["ports"], case["p2"])
    return np.stack([ellipse_phantom(nodes, el, 1000003 * (seed + 1) + f)
                     for f in range(frames or case["frames"])]).astype(np.float32)


def _gamma(case, seed):
    g = _phantoms(case, seed)
    if case["kind"] != "complex":
        return g
    im = _phantoms(case, seed + 7919)
    return (g + 0.1j * im).astype(np.complex64)


def _options(case):
    """The settings the benchmark and the learned start use: reference defaults without a
    coarse level, else FP32 to 1e-6 for a forward solve and mixed precision for a step."""
    if not case["two_level"]:
        return SolveOptions()
    if case["kind"] == "forward":
        return SolveOptions(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-6, preconditioner=capi.MPF_PRECOND_TWO_LEVEL)
    return SolveOptions(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-4, precision=capi.MPF_PREC_MIXED, refine_steps=1,
                        refine_tol=1e-2, preconditioner=capi.MPF_PRECOND_TWO_LEVEL, graphs=case["kind"] == "batch")


def _measure(model, gamma, seed):
    """Measured voltages of the phantoms (frames x m, FP64): an accurate forward solve plus
    60 dB noise."""
    opts = SolveOptions(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-5, precision=capi.MPF_PREC_MIXED, refine_steps=2,
                        refine_tol=1e-3, preconditioner=capi.MPF_PRECOND_TWO_LEVEL)
    model.solve(torch.tensor(gamma, device="cuda"), opts)
    U = model.result64.cpu().numpy()
    rng = np.random.default_rng(seed)
    s = np.sqrt(np.mean(U ** 2, axis=1, keepdims=True)) * 1e-3
    keep = (U != 0.0)
    return torch.tensor(U + keep * s * rng.standard_normal(U.shape), device="cuda")


def _net_dims(case):
    return [case["inputs"]] + [case["hidden"]] * case["layers"] + [case["outputs"]]


def _net_data(case, seed):
    """Standardised voltage features and ln sigma targets (few modes per frame)."""
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(case["batch"], case["inputs"], generator=g)
    T = torch.randn(case["batch"], 8, generator=g) @ torch.randn(8, case["outputs"], generator=g) * 0.15
    return X, T


def _pcg_system(case, seed):
    """A 2.5D system matrix (harmonic 1) in the SparseMatrix layout and boundary sources."""
    one = _eit("forward", case["rings"], case["ports"], 2, 1)
    g = _phantoms(one, seed)[0]
    alpha = (2.0 * math.pi / 0.4) ** 2
    _, _, _, _, pat = _mesh(case["rings"], case["ports"], False)
    B = _excitation(case) @ pat
    return one, g, alpha, B[:, :case["columns"]]


# ------------------------------------------------------------------------------------
# prepare / run
# ------------------------------------------------------------------------------------
def prepare(case, seed):
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        state = _prepare(case, seed, Context())
    stream.synchronize()
    state.update(case=case, stream=stream)
    return state


def _prepare(case, seed, ctx):
    kind = case["kind"]
    if kind in ("gradient", "infer"):
        net = Mlp(_net_dims(case), seed=NET_SEED, ctx=ctx)
        X, T = _net_data(case, seed)
        return dict(net=net, X=X.cuda(), T=T.cuda() if kind == "gradient" else None)
    if kind == "pcg":
        one, g, alpha, B = _pcg_system(case, seed)
        model = _model(one, ctx)
        ids, values = model.update(torch.tensor(g), alpha)
        B = torch.tensor(B.T.copy(), dtype=torch.float32, device="cuda")
        density = int((ids != -1).sum(dim=1).max())
        return dict(ctx=ctx, n=model.N, ids=ids, values=values, density=density, B=B, X=torch.zeros_like(B),
                    options=SolveOptions())
    if kind == "batch":
        jobs = [_job(case["first"] + i) for i in range(case["jobs"])]
        models = [_model(j, ctx) for j in jobs]
        solvers = []
        for i, (j, m) in enumerate(zip(jobs, models)):
            s = Solver(m, LAMBDA, gn_refine=4, options=_options(case | dict(two_level=True)))
            s.measurement.copy_(_measure(m, _phantoms(j, seed + 31 * i), seed + i))
            solvers.append(s)
        batch = Batch(models)
        return dict(models=models, solvers=solvers, batch=batch, driver=BatchSolver(batch, solvers))
    model = _model(case, ctx)
    gamma = _gamma(case, seed)
    if kind in ("forward", "complex"):
        return dict(model=model, gamma=torch.tensor(gamma, device="cuda"), options=_options(case))
    solver = Solver(model, LAMBDA, gn_refine=4, options=_options(case))
    solver.measurement.copy_(_measure(model, gamma, seed))
    if kind == "differential":
        solver.pre_solve()
    return dict(model=model, solver=solver)


def run(state):
    with torch.cuda.stream(state["stream"]):
        return _run(state, state["case"]["kind"])


def _run(state, kind):
    if kind in ("forward", "complex"):
        return state["model"].solve(state["gamma"], state["options"])
    if kind == "step":
        s = state["solver"]
        s.material_distribution.fill_(1.0)
        return s.solve_absolute()
    if kind == "differential":
        return state["solver"].solve_differential()
    if kind == "batch":
        for s in state["solvers"]:
            s.material_distribution.fill_(1.0)
        return state["driver"].solve_absolute()
    if kind == "infer":
        return state["net"].forward(state["X"])
    if kind == "gradient":
        net = state["net"]
        net.forward(state["X"])
        net.backward(state["T"])
        return net.params(grads=True)
    X, B = state["X"], state["B"]
    X.zero_()
    st = capi.SolveStats()
    ptr = lambda t: C.c_void_p(t.data_ptr())
    rc = capi.lib().mpf_pcg_solve(state["ctx"].h, state["n"], state["density"], ptr(state["ids"]), ptr(state["values"]),
                                  B.shape[0], ptr(B), B.shape[1], ptr(X), X.shape[1], 0, C.byref(state["options"].s),
                                  C.byref(st))
    capi.check(rc, allow=(capi.MPF_OK, capi.MPF_ENOCONV))
    return X


# ------------------------------------------------------------------------------------
# the same results in 64 bits: dense matrices and direct solves
# ------------------------------------------------------------------------------------
def _f64(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to("cuda", torch.float64)


def _excitation(case):
    """nodes x electrodes: each electrode's unit current spread evenly over its edges
    (linear edges: half of an edge to either end)."""
    nodes, _, bd, pt, _ = _mesh(case["rings"], case["ports"], False)
    B = np.zeros((nodes.shape[0], case["ports"]))
    for p, edges in enumerate(pt):
        ends = bd[edges[edges >= 0]]
        length = np.linalg.norm(nodes[ends[:, 1]] - nodes[ends[:, 0]], axis=1)
        for k in (0, 1):
            np.add.at(B[:, p], ends[:, k], 0.5 * length / length.sum())
    return B


class _Exact:
    """Linear elements: dense harmonic systems, fields, voltages and Jacobian."""

    def __init__(self, case):
        nodes, el, bd, pt, pat = _mesh(case["rings"], case["ports"], False)
        self.case, self.N, self.E, self.L = case, nodes.shape[0], el.shape[0], case["ports"]
        self.h, self.hp = _height(case["harmonics"])
        self.el, self.pat = torch.as_tensor(el).long().cuda(), _f64(pat)
        xy = nodes[el]                                               # E x 3 x 2
        e1, e2 = xy[:, 1] - xy[:, 0], xy[:, 2] - xy[:, 0]
        area = 0.5 * np.abs(e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0])
        opp = xy[:, [2, 0, 1]] - xy[:, [1, 2, 0]]                    # edge opposite to each node
        self.K = _f64(np.einsum("eik,ejk->eij", opp, opp) / (4.0 * area[:, None, None]))
        self.M = _f64(area[:, None, None] / 12.0 * (np.ones((3, 3)) + np.eye(3)))
        self.B = _f64(_excitation(case))
        self.length = np.zeros(self.L)
        self.Zb = torch.zeros(self.N, self.N, dtype=torch.float64, device="cuda") if case["contact"] else None
        for p, edges in enumerate(pt):
            for a, b in bd[edges[edges >= 0]]:
                s = float(np.linalg.norm(nodes[b] - nodes[a]))
                self.length[p] += s
                if self.Zb is not None:
                    for i, j in ((a, a), (a, b), (b, a), (b, b)):
                        self.Zb[i, j] += s / (3.0 if i == j else 6.0)
        up = lambda n: n if n % 16 == 0 else (n // 16 + 1) * 16
        self.pad = up(self.L)

    def constants(self, c):
        if c == 0:
            return 0.0, 1.0 / self.h
        return (2.0 * c * math.pi / self.h) ** 2, 2.0 * math.sin(c * math.pi * self.hp / self.h) / (c * math.pi * self.hp)

    def system(self, sigma, c):
        alpha, _ = self.constants(c)
        A = torch.zeros(self.N * self.N, dtype=sigma.dtype, device="cuda")
        at = self.el[:, :, None] * self.N + self.el[:, None, :]
        A.index_add_(0, at.reshape(-1), ((self.K + alpha * self.M) * sigma[:, None, None]).reshape(-1))
        return A.reshape(self.N, self.N)

    def fields(self, sigma):
        """Per harmonic the fields of the drive and of the measurement patterns, and the
        voltages (measurement x drive)."""
        harmonics, cplx = range(self.case["harmonics"]), sigma.is_complex()
        solve = torch.linalg.solve if cplx else lambda A, F: torch.cholesky_solve(F, torch.linalg.cholesky(A))
        if not self.case["contact"]:
            Bp = self.B @ self.pat
            F = torch.cat([CURRENT * Bp, Bp], dim=1).to(sigma.dtype)
            phi, U = [], 0.0
            for c in harmonics:
                A = self.system(sigma, c)
                if c == 0:
                    A += 1.0           # the constant mode, which the sources do not excite
                phi.append(solve(A, self.constants(c)[1] * F))
                U = U + Bp.to(sigma.dtype).T @ phi[-1][:, :self.L]
            return phi, U
        # coupled complete electrode model: unit electrode sources per harmonic, then the
        # Schur complement on the electrode potentials
        zp = CONTACT * self.h / self.hp
        length = _f64(self.length)
        Bc = self.B * length
        S = torch.zeros(self.L, self.L, dtype=torch.float64, device="cuda")
        Y, scale = [], []
        for c in harmonics:
            hb, n = self.h * self.constants(c)[1], self.h * (1.0 if c == 0 else 0.5)
            Y.append(solve(self.system(sigma, c) + self.Zb / zp, Bc))
            S += n * hb * hb / zp * (torch.diag(length) - Bc.T @ Y[-1] / zp)
            scale.append(hb / zp)
        V = torch.linalg.solve(S, torch.cat([CURRENT * self.pat, self.pat], dim=1))
        return [s * (y @ V) for s, y in zip(scale, Y)], self.pat.T @ V[:, :self.L]

    def rows(self, U):
        """Measurement x drive -> the padded result vector (drive-major)."""
        out = torch.zeros(self.pad, self.pad, dtype=U.dtype, device="cuda")
        out[:self.L, :self.L] = U.T
        return out.reshape(-1)

    def jacobian(self, phi):
        """Exact derivative of the voltages at unit sigma-derivative: (drive x measurement) x E."""
        J = torch.zeros(self.L, self.L, self.E, dtype=torch.float64, device="cuda")
        for c, X in enumerate(phi):
            alpha, beta = self.constants(c)
            w = self.h * (1.0 if c == 0 else 0.5) if self.case["contact"] else 1.0 / beta
            P = X[self.el]                                            # E x 3 x 2L
            T = (self.K + alpha * self.M) @ P[:, :, self.L:]
            for k in range(3):
                J -= w * P[:, k, :self.L].T[:, None, :] * T[:, k, :].T[None]
        return J.reshape(self.L * self.L, self.E)

    def step(self, measured):
        """One Tikhonov step from the homogeneous start for every measured frame."""
        phi, U = self.fields(torch.ones(self.E, dtype=torch.float64, device="cuda"))
        J = self.jacobian(phi)
        keep = torch.as_tensor(measured).reshape(-1, self.pad, self.pad)[:, :self.L, :self.L].reshape(-1, self.L * self.L)
        r = keep.cuda() - U.T.reshape(-1)
        G = J @ J.T + LAMBDA ** 2 * torch.eye(J.shape[0], dtype=torch.float64, device="cuda")
        return 1.0 + (J.T @ torch.linalg.solve(G, r.T)).T


def _exact_net(case, seed):
    """Weights (uniform within sqrt(6 / (in + out)) from SplitMix64, zero biases) and data."""
    dims, W, state = _net_dims(case), [], np.uint64(NET_SEED)
    with np.errstate(over="ignore"):
        for a, b in zip(dims[:-1], dims[1:]):
            z = state + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, a * b + 1, dtype=np.uint64)
            state = z[-1]
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            u = ((z ^ (z >> np.uint64(31))) >> np.uint64(11)).astype(np.float64) / 2.0 ** 53
            W.append(_f64((math.sqrt(6.0 / (a + b)) * (2.0 * u - 1.0)).astype(np.float32).reshape(a, b)))
    X, T = (t.double().cuda() for t in _net_data(case, seed))
    return W, [torch.zeros(w.shape[1], dtype=torch.float64, device="cuda") for w in W], X, T


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gradient", "infer"):
        W, b, Y, T = _exact_net(case, seed)
        leaves = [p.requires_grad_(kind == "gradient") for pair in zip(W, b) for p in pair]
        for k in range(len(W)):
            Y = Y @ W[k] + b[k]
            if k + 1 < len(W):
                Y = torch.nn.functional.gelu(Y)
        if kind == "infer":
            return Y
        grads = torch.autograd.grad(((Y - T) ** 2).mean(), leaves)
        return torch.cat([g.reshape(-1) for g in grads]).cpu().numpy()
    if kind == "pcg":
        one, g, alpha, B = _pcg_system(case, seed)
        A = _Exact(one).system(_f64(g), 1)
        return torch.cholesky_solve(_f64(B), torch.linalg.cholesky(A)).T.contiguous()
    if kind == "batch":
        jobs = [_job(case["first"] + i) for i in range(case["jobs"])]
        if sum(j["harmonics"] * (3 * j["rings"] ** 2) ** 3 for j in jobs) > 4e13:
            return None
        return [_Exact(j).step(s.measurement.cpu()).contiguous() for j, s in zip(jobs, prepare(case, seed)["solvers"])]
    solves = case["harmonics"] * (case["frames"] if kind in ("forward", "complex") else 1)
    if case["p2"] or solves * (3 * case["rings"] ** 2) ** 3 > 1e13:
        return None
    if kind in ("step", "differential"):
        return _Exact(case).step(prepare(case, seed)["solver"].measurement.cpu())
    ex = _Exact(case)
    gamma = torch.as_tensor(_gamma(case, seed)).to("cuda", torch.complex128 if kind == "complex" else torch.float64)
    return torch.stack([ex.rows(ex.fields(g)[1]) for g in gamma])


# ------------------------------------------------------------------------------------
# work a pass cannot do without
# ------------------------------------------------------------------------------------
def work(case):
    """Bytes: each input read and each output written once; a forward solve also reads the
    system of every frame and harmonic and writes its fields, a step also forms the
    Jacobian.  Flops: one product with each system, the Jacobian's Gram matrix and its
    factorisation, the network's products."""
    kind = case["kind"]
    if kind in ("gradient", "infer"):
        dims, n = _net_dims(case), case["batch"]
        params = sum(a * b + b for a, b in zip(dims[:-1], dims[1:]))
        both = kind == "gradient"
        first = dims[0] * dims[1]
        return dict(bytes=4.0 * (params * (2 if both else 1) + n * (dims[0] + dims[-1])),
                    flops=2.0 * n * ((3 * params - first) if both else params))
    if kind == "batch":
        jobs = [work(_job(case["first"] + i)) for i in range(case["jobs"])]
        return {k: sum(j[k] for j in jobs) for k in ("bytes", "flops")}
    if kind == "pcg":
        n = 3 * case["rings"] * (case["rings"] + 1) + 1
        return dict(bytes=n * (7 * 8.0 + 8.0 * case["columns"]), flops=2.0 * 7 * n * case["columns"])
    rings, L, C_, F = case["rings"], case["ports"], case["harmonics"], case["frames"]
    elements = 6 * rings * rings
    n = (12 if case["p2"] else 3) * rings * (rings + 1) + 1
    nnz = n * (11.5 if case["p2"] else 7.0)
    scalar = 8 if kind == "complex" else 4
    rows = (-(-L // 16) * 16) ** 2
    one = dict(bytes=nnz * (4 + 2 * scalar) + C_ * n * L * scalar, flops=2.0 * C_ * nnz * L)
    if kind in ("forward", "complex"):
        return dict(bytes=F * (one["bytes"] + scalar * (elements + rows)), flops=F * one["flops"])
    dense = rows * rows * float(elements) + rows ** 3 / 3.0
    if kind == "differential":
        # the prepared Jacobian and factor are read once for all frames
        return dict(bytes=4.0 * rows * elements + 8.0 * rows * rows + F * (8.0 * rows + 4.0 * elements),
                    flops=F * (2.0 * rows * elements + 2.0 * rows * rows))
    return dict(bytes=F * (one["bytes"] + 4.0 * rows * elements + 8.0 * (rows + elements)), flops=F * (one["flops"] + dense))
