"""The work a user of adsgpu has it do, as measurable cases: time loops of the explicit and
the linearly implicit step in 2D and 3D, FP64 and FP32, their hooks called one by one, the
adjoints, and batches of small problems, each through the Python binding of the C ABI.

Sizes follow the benchmark's workloads (2D 128^2 with a diffusion field, 3D 128^3 at p = 2,
3D 192^3 at p = 3, 256 uneven 2D problems) and the tests' small and ragged meshes. States are
FP64 coefficient vectors; the FP32 handles' results are taken as float32, the precision their
arithmetic promises.
"""
import math
import os
import sys

import numpy as np
import torch  # before adsgpu: one HIP runtime in the process

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "iga-ads_amd"))
import adsgpu as ag  # noqa: E402

DEV = "cuda"
# largest generalised eigenvalue of (stiffness, mass) times h^2 per degree: an explicit step is
# stable below 2 / sum_d eig_d
MU = {1: 12.0, 2: 21.6, 3: 47.3}


def listed():
    return [
        # the smallest call that occurs: a few steps on a coarse mesh, where launches count
        {"name": "heat3d_tiny", "kind": "explicit", "dim": 3, "p": 2, "nx": 12, "ny": 10, "nz": 9,
         "f32": False, "form": "heat", "dirichlet": False, "steps": 2},
        # forward run of an inverse problem: diffusion field, Dirichlet, one small 2D mesh
        {"name": "heat2d_k_forward", "kind": "explicit", "dim": 2, "p": 2, "nx": 128, "ny": 128, "nz": 0,
         "f32": False, "form": "kfield", "dirichlet": True, "steps": 100},
        # its gradient: forward, checkpointed recompute and adjoint through torch's autograd
        {"name": "heat2d_k_gradient", "kind": "gradient", "dim": 2, "p": 2, "nx": 128, "ny": 128, "nz": 0,
         "f32": False, "form": "kfield", "dirichlet": True, "steps": 100, "every": 20},
        # a problem class that calls the hooks one by one, a large ragged 2D mesh at p = 3
        {"name": "hooks2d_p3", "kind": "hooks", "dim": 2, "p": 3, "nx": 480, "ny": 351, "nz": 0,
         "f32": False, "form": "heat", "dirichlet": True, "steps": 4},
        # the headline workload: 3D explicit heat at p = 2, FP64 and FP32
        {"name": "heat3d_p2_f64", "kind": "explicit", "dim": 3, "p": 2, "nx": 128, "ny": 128, "nz": 128,
         "f32": False, "form": "heat", "dirichlet": False, "steps": 10},
        {"name": "heat3d_p2_f32", "kind": "explicit", "dim": 3, "p": 2, "nx": 128, "ny": 128, "nz": 128,
         "f32": True, "form": "heat", "dirichlet": False, "steps": 10},
        # a nonlinear run on a ragged 3D mesh with Dirichlet boundaries and linear elements
        {"name": "react3d_p1_ragged", "kind": "explicit", "dim": 3, "p": 1, "nx": 77, "ny": 101, "nz": 61,
         "f32": False, "form": "reaction", "dirichlet": True, "steps": 10},
        # a diffusion field in 3D on a ragged mesh
        {"name": "heat3d_k_ragged", "kind": "explicit", "dim": 3, "p": 2, "nx": 70, "ny": 50, "nz": 61,
         "f32": False, "form": "kfield", "dirichlet": True, "steps": 4},
        # the large implicit solve: p = 3 with a source, FP64 and FP32 with refinement
        {"name": "implicit3d_p3_f64", "kind": "implicit", "dim": 3, "p": 3, "nx": 192, "ny": 192, "nz": 192,
         "f32": False, "refine": False, "kron": False, "adjoint": False, "steps": 2},
        {"name": "implicit3d_p3_f32", "kind": "implicit", "dim": 3, "p": 3, "nx": 192, "ny": 192, "nz": 192,
         "f32": True, "refine": True, "kron": False, "adjoint": False, "steps": 2},
        # its separable right-hand side, forward and adjoint steps
        {"name": "implicit3d_p3_separable", "kind": "implicit", "dim": 3, "p": 3, "nx": 192, "ny": 192, "nz": 192,
         "f32": False, "refine": False, "kron": True, "adjoint": True, "steps": 4},
        # the ensemble: 256 uneven 2D reaction-diffusion problems advanced together
        {"name": "ensemble2d_f32", "kind": "batch", "count": 256, "f32": True, "steps": 200, "lo": 32, "hi": 256},
    ]


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones among them."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["explicit3", "explicit3", "explicit2", "implicit", "implicit", "gradient", "hooks", "batch"])
    p = rng.choice([1, 2, 2, 3, 3])
    if kind == "explicit3":
        return {"kind": "explicit", "dim": 3, "p": p, "nx": size(9, 140), "ny": size(9, 140), "nz": size(9, 140),
                "f32": rng.random() < 0.4, "form": rng.choice(["heat", "heat", "reaction", "kfield"]),
                "dirichlet": rng.random() < 0.4, "steps": rng.choice([1, 2, 5])}
    if kind == "explicit2":
        return {"kind": "explicit", "dim": 2, "p": p, "nx": size(16, 480), "ny": size(16, 480), "nz": 0,
                "f32": rng.random() < 0.4, "form": rng.choice(["heat", "reaction", "kfield"]),
                "dirichlet": rng.random() < 0.5, "steps": rng.choice([2, 10, 40])}
    if kind == "implicit":
        f32 = rng.random() < 0.5
        kron = rng.random() < 0.3
        return {"kind": "implicit", "dim": 3, "p": rng.choice([2, 3, 3]), "nx": size(40, 180), "ny": size(40, 180),
                "nz": size(40, 180), "f32": f32, "refine": f32 and rng.random() < 0.6, "kron": kron,
                "adjoint": not f32 and rng.random() < 0.4, "steps": rng.choice([1, 2])}
    if kind == "gradient":
        return {"kind": "gradient", "dim": 2, "p": p, "nx": size(40, 240), "ny": size(40, 240), "nz": 0, "f32": False,
                "form": "kfield", "dirichlet": True, "steps": rng.choice([20, 30, 60]), "every": rng.choice([6, 10])}
    if kind == "hooks":
        d3 = rng.random() < 0.5
        lo, hi = (10, 100) if d3 else (30, 480)
        return {"kind": "hooks", "dim": 3 if d3 else 2, "p": p, "nx": size(lo, hi), "ny": size(lo, hi),
                "nz": size(lo, hi) if d3 else 0, "f32": False, "form": rng.choice(["heat", "reaction"]),
                "dirichlet": rng.random() < 0.5, "steps": 2}
    return {"kind": "batch", "count": rng.choice([24, 48, 96]), "f32": rng.random() < 0.5, "steps": rng.choice([20, 50]),
            "lo": 32, "hi": size(90, 256)}


# ---- the cases' problems --------------------------------------------------------------

def _mesh(case):
    return [case["nx"], case["ny"], case["nz"]][: case["dim"]]


def _dt(case):
    """A stable explicit step (half the limit), or the implicit workload's."""
    if case["kind"] == "implicit":
        return 1e-4
    ne = _mesh(case)
    top = MU[case["p"]] * sum(n * n for n in ne) * (2.0 if case["form"] == "kfield" else 1.0)
    return min(1e-4, 1.0 / top)


def _form(case):
    dt = _dt(case)
    if case["kind"] == "implicit":
        return ag.rhs_form(dt, mass=0.0, source=True)
    if case["form"] == "reaction":
        return ag.rhs_form(dt, grad=(1e-2, 1e-2, 1e-2), reaction=1.0)
    return ag.rhs_form(dt, kfield=case["form"] == "kfield")


def _greville(p, ne):
    kn = np.concatenate([np.zeros(p), np.arange(ne + 1) / ne, np.ones(p)])
    return torch.tensor([kn[i + 1:i + p + 1].mean() for i in range(ne + p)], dtype=torch.float64, device=DEV)


def _bumps(case, gen, count=4):
    """A sum of Gaussians, 1e-3 of noise on it: coefficients at the Greville abscissae, x fastest."""
    ne = _mesh(case)
    g = [_greville(case["p"], n) for n in ne][::-1]
    u = torch.zeros([len(x) for x in g], dtype=torch.float64, device=DEV)
    par = torch.rand(count, len(g) + 1, generator=gen, dtype=torch.float64).tolist()
    for row in par:
        s = 0.05 + 0.1 * row[-1]
        term = 1.0
        for d, x in enumerate(g):
            ax = [1] * len(g)
            ax[d] = -1
            term = term * torch.exp(-((x - (0.2 + 0.6 * row[d])) ** 2) / (2 * s * s)).reshape(ax)
        u += term
    noise = torch.Generator(device=DEV)
    noise.manual_seed(int(torch.randint(1 << 30, (1,), generator=gen)))
    return u + 1e-3 * (2 * torch.rand(u.shape, generator=noise, dtype=torch.float64, device=DEV) - 1)


def _waves(case, gen, terms=4):
    """A smooth field: a few separable sines."""
    g = [_greville(case["p"], n) for n in _mesh(case)][::-1]
    f = torch.zeros([len(x) for x in g], dtype=torch.float64, device=DEV)
    for _ in range(terms):
        par = torch.rand(len(g) + 1, generator=gen, dtype=torch.float64).tolist()
        term = 2 * par[-1] - 1
        for d, x in enumerate(g):
            ax = [1] * len(g)
            ax[d] = -1
            term = term * torch.sin((1 + int(3 * par[d])) * math.pi * x).reshape(ax)
        f += term
    return f


def _zero_faces(u):
    for d in range(u.dim()):
        u.select(d, 0).zero_()
        u.select(d, u.shape[d] - 1).zero_()
    return u


def _inputs(case, seed):
    """u(0) and, where the form has one, the diffusion field in [1/2, 2] or the source."""
    gen = torch.Generator()
    gen.manual_seed(seed)
    u0 = _bumps(case, gen)
    if case.get("form") == "reaction":
        u0 = (u0 - u0.min()) / (u0.max() - u0.min())
    if case.get("dirichlet"):
        _zero_faces(u0)
    k = f = None
    if case.get("form") == "kfield":
        w = _waves(case, gen)
        k = torch.exp(w / w.abs().max() * math.log(2.0))
    if case["kind"] == "implicit":
        f = _waves(case, gen)
    return u0.contiguous(), k, f


def _problems(case, seed):
    """Degrees, sizes and diffusivities of the ensemble are the workload's own; the states and
    diffusivities come from the seed."""
    shape = np.random.default_rng(2028 + case["count"] + case["hi"])
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        p, ne = int(shape.integers(1, 4)), int(shape.integers(case["lo"], case["hi"] + 1))
        eps = float(10.0 ** rng.uniform(-4, -2))
        x = (np.arange(ne + p) + 0.5) / (ne + p)
        u = 0.0
        for _ in range(3):
            cx, cy = rng.uniform(0.2, 0.8, 2)
            s = rng.uniform(0.1, 0.3)
            u = u + np.exp(-((x - cy) ** 2) / (2 * s * s))[:, None] * np.exp(-((x - cx) ** 2) / (2 * s * s))
        out.append((p, ne, eps, (u - u.min()) / (u.max() - u.min())))
    return out


BATCH_DT = 2e-5
GROUP = 8  # problems of the ensemble per returned array


def prepare(case, seed):
    if case["kind"] == "batch":
        probs = _problems(case, seed)
        b = ag.Batch([(p, ne) for p, ne, _, _ in probs], precision=ag.FP32 if case["f32"] else ag.FP64)
        b.prepare()
        b.set_forms([ag.rhs_form(BATCH_DT, grad=(e, e, 0.0), reaction=1.0) for _, _, e, _ in probs])
        for i, q in enumerate(probs):
            b.set(i, q[3])
        return {"case": case, "batch": b}
    u0, k, f = _inputs(case, seed)
    sim = ag.Simulation(case["dim"], [case["p"]] * case["dim"], _mesh(case),
                        precision=ag.FP32 if case["f32"] else ag.FP64)
    state = {"case": case, "sim": sim, "form": _form(case), "slots": None, "flags": 0}
    if case.get("dirichlet"):
        sim.fix_all_boundaries()
        state["flags"] |= ag.STEP_DIRICHLET
    if case["kind"] == "implicit":
        for d in range(case["dim"]):
            sim.set_matrix(d, 1, 1.0, 0.5 * _dt(case))
        state["slots"] = [1] * case["dim"]
        sim.set_tuning(ag.TUNE_RHS_KRONECKER, int(case["kron"]))
        state["flags"] |= ag.STEP_REFINE if case["refine"] else 0
    sim.prepare_matrices()
    torch.cuda.synchronize()
    if case["kind"] == "gradient":
        state["k"] = k.reshape(-1).requires_grad_()
        state["u0"] = u0.reshape(-1).requires_grad_()
        state["target"] = 0.9 * u0.reshape(-1).detach()
        return state
    sim.set_device(ag.U, u0.data_ptr())
    for which, field in ((ag.KFIELD, k), (ag.SOURCE, f)):
        if field is not None and case["f32"]:  # FP32 handles take their fields from the host
            sim.set(which, field.cpu().numpy())
        elif field is not None:
            sim.set_device(which, field.data_ptr())
    state["out"] = torch.empty_like(u0)
    return state


def run(state):
    case = state["case"]
    n = case["steps"]
    if case["kind"] == "batch":  # advance the ensemble and fetch every problem's state
        b = state["batch"]
        b.step(n)
        got = [b.get(i) for i in range(b.count)]
        kind = np.float32 if case["f32"] else np.float64
        return [np.concatenate(got[i:i + GROUP]).astype(kind) for i in range(0, b.count, GROUP)]
    sim, form, flags = state["sim"], state["form"], state["flags"]
    if case["kind"] == "gradient":  # one evaluation of a loss and its gradients
        k, u0 = state["k"], state["u0"]
        k.grad = u0.grad = None
        u = ag.heat_k(sim, k, u0, n, case["every"], _dt(case), bool(case["dirichlet"]))
        loss = ((u - state["target"]) ** 2).sum()
        loss.backward()
        return {"u": u.detach(), "dk": k.grad, "du0": u0.grad}
    # a stretch of the time loop, then the state as a tensor; the next pass goes on from it
    if case["kind"] == "implicit":
        sim.step_delta(n, form, state["slots"], flags)
        if case["adjoint"]:
            sim.adjoint_step_delta(n, form, state["slots"], flags)
    elif case["kind"] == "hooks":
        for _ in range(n):
            sim.swap()
            sim.compute_rhs(form)
            if case["dirichlet"]:
                sim.zero_boundary()
            sim.ads_solve()
    else:
        sim.step(n, form, flags)
    sim.get_device(ag.U, state["out"].data_ptr())
    return state["out"].float() if case["f32"] else state["out"]


# ---- what a pass cannot do without ----------------------------------------------------

def _step_work(ne, p, extra_fields, adjoint=False):
    """One step on a mesh: the state read and written once (and each field read), the element
    integrals by sum factorisation over the whole tensor grid (each 1D contraction done once
    per line of the grid, values and gradients forward, test functions backward) and the
    banded substitution of every line in every direction."""
    d = len(ne)
    n = [e + p for e in ne]
    q = [e * (p + 1) for e in ne]
    dofs = math.prod(n)
    flops = 0
    fields_in = 2  # value and derivative along x; then one more combination per direction
    for k in range(d):
        lines = math.prod(q[:k + 1]) * math.prod(n[k + 1:])
        flops += 2 * 2 * (p + 1) * lines * (fields_in + k)
        if extra_fields:
            flops += 2 * (p + 1) * lines * extra_fields
    flops += 8 * math.prod(q)
    flops += 2 * dofs * d * (2 * p * 2 + 1) // 2
    return dofs, flops


def work(case):
    f = 4 if case["f32"] else 8
    if case["kind"] == "batch":
        shape = np.random.default_rng(2028 + case["count"] + case["hi"])
        nb = nf = 0
        for _ in range(case["count"]):
            p, ne = int(shape.integers(1, 4)), int(shape.integers(case["lo"], case["hi"] + 1))
            dofs, flops = _step_work([ne, ne], p, 0)
            nb, nf = nb + 2 * dofs * f, nf + flops
        return {"bytes": nb * case["steps"], "flops": nf * case["steps"]}
    fields = 1 if case.get("form") == "kfield" else 0
    dofs, flops = _step_work(_mesh(case), case["p"], fields)
    if case.get("kron"):  # the 1D Gram and stiffness products instead of the element integrals
        flops = dofs * (2 * (2 * case["p"] + 1) * 8 + 3 * (4 * case["p"] + 1))
    per = 2 + fields + (1 if case["kind"] == "implicit" else 0)
    runs = 1
    if case.get("adjoint"):
        runs = 2
    if case["kind"] == "gradient":
        runs = 3  # forward, recompute, adjoint with the field's gradient
    return {"bytes": dofs * f * per * case["steps"] * runs, "flops": flops * case["steps"] * runs}


# ---- the same in 64 bits with plain torch ---------------------------------------------

class _Line:
    """One direction: B-spline values and derivatives at the Gauss points, the weights, and
    the Gram and stiffness matrices, dense."""

    def __init__(self, p, ne, fixed=False):
        t = np.concatenate([np.zeros(p), np.arange(ne + 1) / ne, np.ones(p)])
        g, w = np.polynomial.legendre.leggauss(p + 1)
        x = ((np.arange(ne)[:, None] + 0.5 * (g + 1)) / ne).ravel()
        span = np.repeat(np.arange(ne) + p, p + 1)
        low = np.ones((len(x), 1))  # the basis functions of rising degree that are nonzero at x
        for k in range(1, p + 1):
            prev, low = low, np.zeros((len(x), k + 1))
            for j in range(k):
                i = span - k + 1 + j
                width = t[i + k] - t[i]
                low[:, j] += (t[i + k] - x) / width * prev[:, j]
                low[:, j + 1] += (x - t[i]) / width * prev[:, j]
        der = np.zeros((len(x), p + 1))
        for j in range(p):
            i = span - p + 1 + j
            der[:, j] -= p / (t[i + p] - t[i]) * prev[:, j]
            der[:, j + 1] += p / (t[i + p] - t[i]) * prev[:, j]
        n = ne + p
        B, D = np.zeros((len(x), n)), np.zeros((len(x), n))
        for j in range(p + 1):
            B[np.arange(len(x)), span - p + j] = low[:, j]
            D[np.arange(len(x)), span - p + j] = der[:, j]
        W = np.tile(w / (2 * ne), ne)
        self.mass, self.stiff = B.T @ (W[:, None] * B), D.T @ (W[:, None] * D)
        self.B, self.D, self.w, self.M, self.K = (torch.tensor(a, device=DEV) for a in (B, D, W, self.mass, self.stiff))
        self.fixed = fixed

    def inverse(self, c=0.0):
        A = self.mass + c * self.stiff
        if self.fixed:
            A[0], A[-1] = 0.0, 0.0
            A[0, 0] = A[-1, -1] = 1.0
        return torch.tensor(np.linalg.inv(A), device=DEV)


def _along(mats, u):
    """mats[d] applied along direction d (x is the last axis); None leaves a direction alone."""
    nd = u.dim()
    for d, m in enumerate(mats):
        if m is not None:
            ax = nd - 1 - d
            u = torch.movedim(torch.tensordot(m, u, dims=([1], [ax])), 0, ax)
    return u


class _Exact:
    def __init__(self, case, ne, p, form, dt, c=0.0, grad=1.0, mass=1.0, reaction=0.0):
        self.L = [_Line(p, n, bool(case.get("dirichlet"))) for n in ne]
        self.inv = [a.inverse(c) for a in self.L]
        self.dt, self.grad, self.mass, self.reaction = dt, grad, mass, reaction
        self.zero = bool(case.get("dirichlet"))

    def mask(self, u):
        if not self.zero:
            return u
        m = _zero_faces(torch.ones_like(u))
        return u * m

    def kron(self, u):
        M, K = [a.M for a in self.L], [a.K for a in self.L]
        r = self.mass * _along(M, u) if self.mass else 0.0
        for d in range(u.dim()):
            r = r - self.dt * self.grad * _along(M[:d] + [K[d]] + M[d + 1:], u)
        return r

    def rhs(self, u, k=None):
        if k is None and not self.reaction:
            return self.kron(u)
        B, D = [a.B for a in self.L], [a.D for a in self.L]
        nd = u.dim()
        w = self.L[0].w.reshape([-1])
        for a in self.L[1:]:
            w = a.w.reshape([-1] + [1] * w.dim()) * w
        v = _along(B, u)
        kv = _along(B, k) if k is not None else 1.0
        g = self.mass * v + (self.dt * self.reaction * v * (1 - v) if self.reaction else 0.0)
        r = _along([b.T for b in B], w * g)
        for d in range(nd):
            du = _along(B[:d] + [D[d]] + B[d + 1:], u)
            T = [b.T for b in B[:d]] + [D[d].T] + [b.T for b in B[d + 1:]]
            r = r - _along(T, (self.dt * self.grad) * w * kv * du)
        return r

    def step(self, u, k=None):
        return _along(self.inv, self.mask(self.rhs(u, k)))


def exact(case, seed):
    if case["kind"] == "batch":
        out = [None] * (-(-case["count"] // GROUP))
        probs = _problems(case, seed)
        for j in range(min(2, len(out))):  # the first problems stand for the rest
            group = []
            for p, ne, eps, u in probs[j * GROUP:(j + 1) * GROUP]:
                e = _Exact({}, [ne, ne], p, None, BATCH_DT, grad=eps, reaction=1.0)
                u = torch.tensor(u, device=DEV)
                for _ in range(case["steps"]):
                    u = e.step(u)
                group.append(u.reshape(-1))
            out[j] = torch.cat(group)
        return out
    u, k, f = _inputs(case, seed)
    dt, ne, p = _dt(case), _mesh(case), case["p"]
    if case["kind"] == "implicit":
        e = _Exact(case, ne, p, None, dt, c=0.5 * dt, mass=0.0)
        load = dt * _along([a.M for a in e.L], f)
        for _ in range(case["steps"]):
            u = u + _along(e.inv, load + e.kron(u))
        if case["adjoint"]:  # A and the form's operator are symmetric
            for _ in range(case["steps"]):
                u = u + e.kron(_along(e.inv, u))
        return u
    react = case["form"] == "reaction"
    e = _Exact(case, ne, p, None, dt, grad=1e-2 if react else 1.0, reaction=1.0 if react else 0.0)
    if case["kind"] == "gradient":
        k = k.clone().requires_grad_()
        u0 = u.clone().requires_grad_()
        u = u0
        for _ in range(case["steps"]):
            u = e.step(u, k)
        ((u - 0.9 * u0.detach()) ** 2).sum().backward()
        return {"u": u.detach().reshape(-1), "dk": k.grad.reshape(-1), "du0": u0.grad.reshape(-1)}
    for _ in range(case["steps"]):
        u = e.step(u, k)
    return u
