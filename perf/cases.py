"""Performance cases of the solve path: what a program that uses the library
asks of it, from the smallest static plate to the 823,875-DOF cube, through
the public entry points (Context and autograd.ElasticProblem; device vectors
through the C-ABI of include/femgpu.h).

Meshes are the structured plates and boxes of cudafemproject_amd.problem, the
sizes those of the repository's benchmark and tests and odd ones between
them; loads, materials and densities come from the seed.  Solves ask for a
relative residual of 1e-10, the default of the autograd binding, at which two
correct solvers return the same displacements.
Results of FP32 arithmetic arrive in float64 arrays that hold 32-bit numbers;
they are handed on as float32, which loses nothing.

listed() are the cases, draw(rng) more of the same ranges, prepare() what a
program holds before the call (a context with the planned mesh), run() one
call, exact() the same results in plain 64-bit torch, work() the bytes and
operations a case cannot do without.
"""
import math

import numpy as np
import torch

import cudafemproject_amd as F
from cudafemproject_amd.autograd import ElasticProblem
from cudafemproject_amd.problem import (BatchInstance, Problem, box_face_tris, box_tet, load_batch,
                                        nodes_on_plane, outward_normals, plate_tri)

PRECISION = {"fp64": F.FP64, "fp32": F.FP32, "mixed": F.MIXED}
RHO = 2400.0
N_CASES = 4          # load cases of a batch instance


def listed():
    return [
        # A small plate as in the reference's own tests: one short solve, its
        # stresses; launches and fixed costs count.
        {"name": "plate_tiny", "kind": "static", "nx": 12, "ny": 7, "nz": 0,
         "precision": "fp64", "tol": 1e-10, "stress": True},
        # The reference-sized 2D plate (4,290 DOF): a solve and its stresses.
        {"name": "plate_64x32", "kind": "static", "nx": 64, "ny": 32, "nz": 0,
         "precision": "fp64", "tol": 1e-10, "stress": True},
        # An ordinary 3D part of ragged size in mixed precision.
        {"name": "block_odd", "kind": "static", "nx": 23, "ny": 17, "nz": 19,
         "precision": "mixed", "tol": 1e-10, "stress": True},
        # The headline cube in FP64, with the stresses for the results file.
        {"name": "cube_fp64", "kind": "static", "nx": 64, "ny": 64, "nz": 64,
         "precision": "fp64", "tol": 1e-10, "stress": True},
        # The headline cube in mixed precision, displacements only.
        {"name": "cube_mixed", "kind": "static", "nx": 64, "ny": 64, "nz": 64,
         "precision": "mixed", "tol": 1e-10, "stress": False},
        # One step of a compliance optimisation: value and gradient of a
        # cantilever with its own modulus in every element.
        {"name": "cantilever_grad", "kind": "compliance", "nx": 48, "ny": 16, "nz": 16,
         "precision": "fp64", "tol": 1e-10},
        # Forward and backward of a general loss through torch.autograd.
        {"name": "adjoint", "kind": "adjoint", "nx": 25, "ny": 9, "nz": 9,
         "precision": "fp64", "tol": 1e-10},
        # Wave propagation along the 393,216-element column, explicit steps.
        {"name": "column_explicit", "kind": "explicit", "nx": 16, "ny": 16, "nz": 256,
         "precision": "fp64", "steps": 1000, "receivers": 0},
        # A small 2D wave run in FP32 with receiver traces for a SEG-Y file.
        {"name": "plate_traces", "kind": "explicit", "nx": 63, "ny": 31, "nz": 0,
         "precision": "fp32", "steps": 400, "receivers": 24},
        # Implicit steps at several times the explicit step, a nested solve each.
        {"name": "column_implicit", "kind": "implicit", "nx": 11, "ny": 11, "nz": 80,
         "precision": "fp64", "steps": 20, "receivers": 0},
        # Many uneven plates with four load cases each, solved together.
        {"name": "plates_batch", "kind": "batch", "n": 60, "nx": 80, "ny": 40, "nz": 0,
         "precision": "fp64", "tol": 1e-10},
        # One product of a caller's own Krylov loop on device vectors.
        {"name": "matvec_cube", "kind": "matvec", "nx": 64, "ny": 64, "nz": 64,
         "precision": "fp64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["static", "static", "static", "compliance", "adjoint", "explicit",
                       "explicit", "implicit", "batch", "matvec"])
    c = {"kind": kind, "nx": 0, "ny": 0, "nz": 0, "precision": rng.choice(["fp64", "mixed"])}
    if kind == "batch":
        c.update(n=_log_int(rng, 3, 60), nx=rng.randint(10, 80), ny=rng.randint(6, 40), tol=1e-10)
        return c
    if kind in ("compliance", "adjoint"):
        n = _log_int(rng, 5, 16)
        c.update(nx=rng.randint(n, 3 * n), ny=n, nz=max(4, n + rng.randint(-2, 2)), tol=1e-10,
                 precision="fp64")
        return c
    if kind == "static" and rng.random() < 0.4:
        ny = _log_int(rng, 5, 48)
        c.update(nx=rng.randint(ny, 2 * ny), ny=ny, precision="fp64", tol=1e-10, stress=True)
        return c
    if kind == "explicit" and rng.random() < 0.4:
        ny = _log_int(rng, 8, 80)
        c.update(nx=rng.randint(ny, 2 * ny), ny=ny, receivers=rng.choice([0, 5, 24]))
    elif kind in ("explicit", "implicit"):
        n = rng.randint(5, 16 if kind == "explicit" else 11)
        c.update(nx=n, ny=max(4, n + rng.randint(-2, 2)), nz=_log_int(rng, n, 16 * n if kind == "explicit" else 80),
                 receivers=rng.choice([0, 0, 9]))
    if kind == "explicit":
        c.update(steps=rng.randint(150, 900), precision=rng.choice(["fp64", "fp32"]))
    elif kind == "implicit":
        c.update(steps=rng.randint(6, 20), precision="fp64")
    else:
        n = _log_int(rng, 6, 60)
        c.update(nx=n, ny=max(4, n + rng.randint(-3, 3)), nz=max(4, n + rng.randint(-3, 3)))
        if kind == "matvec":
            c.update(precision="fp64")
        else:
            c.update(tol=1e-10, stress=rng.random() < 0.5)
    return c


# ---------------------------------------------------------------------------
# inputs

def _box(case):
    """Edge lengths: cells of 1/64 of a metre."""
    h = 1.0 / 64.0
    return case["nx"] * h, case["ny"] * h, case["nz"] * h


def _problem(case, seed):
    """The seeded problem: mesh, clamped face, uneven pressure on the opposite
    one, Poisson ratio; element scales for the optimisation cases."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    lx, ly, lz = _box(case)
    nu = float(rng.uniform(0.2, 0.3))
    if nz == 0:
        nodes, elems = plate_tri(nx, ny, lx, ly)
        fixed, code = nodes_on_plane(nodes, 0, 0.0), 3
        j = np.arange(ny)
        a = nx + (nx + 1) * j
        fn = np.stack([a, a + nx + 1], 1).astype(np.int32)
        fa = (2 * (nx - 1 + nx * j)).astype(np.int32)
        fi = (a - 1).astype(np.int32)
        normals = outward_normals(nodes, fn, fi)
    else:
        nodes, elems = box_tet(nx, ny, nz, lx, ly, lz)
        bend = case["kind"] in ("compliance", "adjoint")
        axis = 0 if bend else 2
        fixed, code = nodes_on_plane(nodes, axis, 0.0), 7
        fn, fa, fi = box_face_tris(nx, ny, nz, axis, 1)
        normals = (np.tile([[0.0, 0.0, 1.0]], (len(fa), 1)) if bend
                   else outward_normals(nodes, fn, fi))
    p = 1e3 * (1.0 + 0.3 * rng.standard_normal(len(fa)))
    pb = Problem(nodes=nodes, elems=elems, constr_node=fixed,
                 constr_code=np.full(len(fixed), code, np.int32), face_nodes=fn, face_adj=fa,
                 face_normal=normals, face_p=p, face_interior=fi, E=2e7, nu=nu,
                 convention=F.LOADS_PHYSICAL)
    if case["kind"] in ("compliance", "adjoint"):
        pb.elem_scale = rng.uniform(0.3, 1.0, size=len(elems)) ** 3
    return pb, rng


def _time_options(case, pb):
    """Explicit step well inside the stability limit of the smallest cell
    (implicit: 12 times that), a Ricker pulse over the run."""
    lam, mu = _lame(pb.E, pb.nu, pb.dim)
    dt = 0.2 / 64.0 / math.sqrt((lam + 2 * mu) / RHO)
    implicit = case["kind"] == "implicit"
    if implicit:
        dt *= 12.0
    o = dict(rho=RHO, beta1=0.5, beta2=0.5 if implicit else 0.0, dt=dt,
             endtime=(case["steps"] + 0.5) * dt, wavelet_type=F.WAVELET_RICKER,
             freq=3.0 / (case["steps"] * dt), timeshift=0.0, ampl=1e3,
             precision=PRECISION[case["precision"]], mass_convention=F.MASS_PHYSICAL)
    if implicit:
        o.update(implicit_mode=F.IMPLICIT_PHYSICAL, pcg_eps=1e-22)
    return o


def _plates(case, seed):
    """Uneven plates (each its own grid, modulus, Poisson ratio) with four
    load cases: end tractions in x and y, top shear, body force."""
    sizes = np.random.default_rng(17)       # the plates' grids: the mesh of the batch
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["n"]):
        nx = int(sizes.integers(case["nx"] // 2, case["nx"] + 1))
        ny = int(sizes.integers(case["ny"] // 2, case["ny"] + 1))
        nodes, elems = plate_tri(nx, ny, nx / 64.0, ny / 64.0)
        f = np.zeros((len(nodes), N_CASES, 2))
        t = 1e3 * rng.uniform(0.5, 1.5, size=N_CASES) / 64.0
        right = nodes_on_plane(nodes, 0, nx / 64.0)
        top = nodes_on_plane(nodes, 1, ny / 64.0)
        f[right, 0, 0] = t[0]
        f[right, 1, 1] = t[1]
        f[top, 2, 0] = t[2]
        f[:, 3, 1] = -t[3] / 64.0
        left = nodes_on_plane(nodes, 0, 0.0)
        f[left] = 0.0
        out.append(BatchInstance(nodes=nodes, elems=elems, E=float(rng.lognormal(math.log(2e7), 0.5)),
                                 nu=float(rng.uniform(0.2, 0.35)), constr_node=left,
                                 constr_code=np.full(len(left), 3, np.int32), f=f))
    return out


_stream = None


def _shared_stream():
    """Device-vector calls on one GPU share its scratch: one stream for all."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _receivers(case, pb):
    return np.linspace(0, pb.n_nodes - 1, case["receivers"]).astype(np.int32)


# ---------------------------------------------------------------------------
# what is measured

def prepare(case, seed):
    kind = case["kind"]
    ctx = F.Context(0)
    s = {"case": case, "ctx": ctx}
    if kind == "batch":
        insts = _plates(case, seed)
        load_batch(ctx, insts)
        s["f"] = [b.f for b in insts]
        return s
    pb, rng = _problem(case, seed)
    ctx.set_problem(pb)
    if kind in ("explicit", "implicit"):
        s["options"] = _time_options(case, pb)
        if case["receivers"]:
            ctx.set_receivers(_receivers(case, pb), F.RECV_VELOCITY, 4)
    elif kind == "adjoint":
        s["problem"] = ElasticProblem(ctx, pb.E, pb.nu, precision=PRECISION[case["precision"]],
                                      tol=case["tol"])
        s["scale"] = torch.from_numpy(pb.elem_scale).requires_grad_()
        s["f"] = torch.from_numpy(ctx.rhs()).requires_grad_()
        s["target"] = torch.from_numpy(_target(pb, rng))
    elif kind == "matvec":
        ctx.diag()                          # prepares the operator
        ctx.set_stream(_shared_stream().cuda_stream)
        x = torch.from_numpy(rng.standard_normal((pb.n_nodes, pb.dim))).cuda()
        s["x"], s["y"] = x, torch.zeros_like(x)
        torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind, prec = case["kind"], PRECISION[case["precision"]]
    if kind == "static":
        u, _ = ctx.solve(prec, tol=case["tol"], tol_kind=F.TOL_REL_RES)
        return {"u": u, "stress": ctx.stress(u)} if case["stress"] else {"u": u}
    if kind == "compliance":
        c, g, u, _ = ctx.compliance_grad(prec, tol=case["tol"])
        return {"compliance": c, "gradient": g, "u": u}
    if kind == "adjoint":
        s["scale"].grad = s["f"].grad = None
        u = s["problem"].solve(s["scale"], s["f"])
        (u * s["target"]).sum().backward()
        return {"u": u.detach(), "d_scale": s["scale"].grad, "d_f": s["f"].grad}
    if kind in ("explicit", "implicit"):
        u, _ = ctx.dyn_run(**s["options"])
        out = {"u": u}
        if case["receivers"]:
            out["traces"] = ctx.traces()
        return {k: v.astype(np.float32) for k, v in out.items()} if prec == F.FP32 else out
    if kind == "batch":
        return ctx.batch_solve(s["f"], prec, tol=case["tol"])[0]
    ctx._check(ctx.lib.femgpu_matvec_noalloc(ctx.h, prec, s["x"].data_ptr(), s["y"].data_ptr()),
               "matvec_noalloc")
    return s["y"]


# ---------------------------------------------------------------------------
# the least a case needs

def work(case):
    """Compulsory bytes (mesh and inputs in, results out, once each) and
    operations (element products and vector updates of the iterations or
    steps a Jacobi-preconditioned conjugate gradient or the scheme takes)."""
    nx, ny, nz, kind = case["nx"], case["ny"], case["nz"], case["kind"]
    dim = 3 if nz else 2
    if kind == "batch":
        sx, sy = 0.75 * nx, 0.75 * ny
        nn, ne, rhs = case["n"] * (sx + 1) * (sy + 1), case["n"] * 2 * sx * sy, N_CASES
    else:
        nn = (nx + 1) * (ny + 1) * ((nz + 1) if nz else 1)
        ne, rhs = (6 * nx * ny * nz if nz else 2 * nx * ny), 1
    per_elem = 230.0 if dim == 3 else 70.0
    s = 4 if case["precision"] == "fp32" else 8
    nd = dim * nn
    mesh = 4 * (dim + 1) * ne + s * nd
    out_in = 2 * s * nd * rhs
    if kind == "matvec":
        return {"bytes": mesh + 2 * 8 * nd, "flops": per_elem * ne}
    if kind == "explicit":
        return {"bytes": mesh + out_in, "flops": case["steps"] * (per_elem * ne + 10 * nd)}
    if kind == "implicit":
        return {"bytes": mesh + out_in, "flops": case["steps"] * 30 * (per_elem * ne + 10 * nd)}
    digits = -math.log10(case["tol"])
    its = 1.7 * digits * max(nx, ny, nz) * (1.0 if dim == 3 else 0.6) * (2 if kind == "adjoint" else 1)
    bytes_ = mesh + out_in
    if case.get("stress"):
        bytes_ += 8 * 3 * (dim - 1) * ne
    if kind in ("compliance", "adjoint"):
        bytes_ += 16 * ne
    return {"bytes": bytes_, "flops": its * rhs * (per_elem * ne + 10 * nd)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, plain torch

def _lame(E, nu, dim):
    mu = E / (2.0 * (1.0 + nu))
    return (E * nu / ((1.0 + nu) * (1.0 - 2.0 * nu)) if dim == 3 else E * nu / (1.0 - nu * nu)), mu


class _Operator:
    """Element stiffnesses from barycentric gradients; fixed DOFs keep only
    their diagonal."""

    def __init__(self, nodes, elems, lam, mu, fixed, scale=None):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
        self.dev, self.dim, self.nn = dev, nodes.shape[1], len(nodes)
        d = self.dim
        el = torch.as_tensor(elems.astype(np.int64), device=dev)
        X = t(nodes)[el]
        J = (X[:, 1:] - X[:, :1]).transpose(1, 2)
        det = torch.linalg.det(J)
        g = torch.linalg.inv(J)
        self.G = torch.cat([-g.sum(1, keepdim=True), g], 1)       # gradients, (ne, npe, d)
        self.V = det.abs() / math.factorial(d)
        self.el, self.lam, self.mu = el, t(lam), t(mu)
        G, lam, mu = self.G, self.lam.reshape(-1, 1, 1, 1, 1), self.mu.reshape(-1, 1, 1, 1, 1)
        eye = torch.eye(d, dtype=torch.float64, device=dev)
        # K_(a i)(b j) = V (lam g_ai g_bj + mu g_aj g_bi + mu g_a.g_b delta_ij)
        K = lam * (G[:, :, :, None, None] * G[:, None, None, :, :])
        K += mu * (G[:, :, None, None, :] * G.transpose(1, 2)[:, None, :, :, None])
        K += mu * (G @ G.transpose(1, 2).contiguous())[:, :, None, :, None] * eye[None, None, :, None, :]
        n = d * (d + 1)
        K = K.reshape(-1, n, n) * self.V[:, None, None]
        self.dofs = (el[:, :, None] * d + torch.arange(d, device=dev)).reshape(-1, n)
        self.fixed = torch.as_tensor(fixed.reshape(-1), device=dev)
        fe = self.fixed[self.dofs]
        diag = torch.diagonal(K, dim1=1, dim2=2).clone()
        K[fe[:, :, None] | fe[:, None, :]] = 0.0
        torch.diagonal(K, dim1=1, dim2=2).copy_(diag)
        self.K0 = K
        self.K = K if scale is None else K * t(scale)[:, None, None]
        self.diag = self.assemble(torch.diagonal(self.K, dim1=1, dim2=2))

    def assemble(self, fe):
        out = torch.zeros(self.nn * self.dim, dtype=torch.float64, device=self.dev)
        return out.index_add_(0, self.dofs.reshape(-1), fe.reshape(-1))

    def __call__(self, u):
        return self.assemble((self.K * u[self.dofs][:, None, :]).sum(2))

    def solve(self, f, shift=None, factor=1.0, tol=1e-14, x0=None):
        """(factor K + diag(shift)) x = f by Jacobi-PCG, restarted on the
        true residual."""
        sh = 0.0 if shift is None else shift
        op = lambda v: factor * self(v) + sh * v  # noqa: E731
        D = factor * self.diag + sh
        D = torch.where(D != 0, D, torch.ones_like(D))
        x = torch.zeros_like(f) if x0 is None else x0.clone()
        stop = (tol * torch.linalg.norm(f)).item() ** 2
        for _ in range(3):
            r = f - op(x)
            p, gam = None, None
            for it in range(20000):
                z = r / D
                g = torch.dot(r, z)
                p = z if p is None else z + (g / gam) * p
                gam = g
                q = op(p)
                a = g / torch.dot(p, q)
                x = x + a * p
                r = r - a * q
                if it % 20 == 19 and torch.dot(r, r).item() <= stop:
                    break
                if it % 20 == 19 and not g.item() > 0:
                    break
        return x

    def stress(self, u):
        """(xx, yy, xy | xx, yy, zz, xy, yz, xz) per element."""
        ue = u.reshape(-1, self.dim)[self.el]
        H = torch.einsum("eai,eaj->eij", ue, self.G)
        e = H + H.transpose(1, 2)
        s = self.mu * e + self.lam * torch.diagonal(H, dim1=1, dim2=2).sum(1)[:, None, None] * torch.eye(
            self.dim, dtype=torch.float64, device=self.dev)
        idx = ((0, 0), (1, 1), (0, 1)) if self.dim == 2 else ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))
        return torch.stack([s[:, i, j] for i, j in idx], 1)


def _fixed(nodes, constr_node):
    fx = np.zeros(nodes.shape, bool)
    fx[constr_node] = True
    return fx


def _load(pb, pressure):
    """F = -p A / d n on the nodes of every face, zero on fixed DOFs."""
    d = pb.dim
    P = pb.nodes[pb.face_nodes]
    if d == 2:
        A = np.linalg.norm(P[:, 1] - P[:, 0], axis=1)
    else:
        A = 0.5 * np.linalg.norm(np.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0]), axis=1)
    n = pb.face_normal / np.linalg.norm(pb.face_normal, axis=1, keepdims=True)
    f = np.zeros_like(pb.nodes)
    np.add.at(f, pb.face_nodes.reshape(-1), np.repeat(-pressure[:, None] * A[:, None] / d * n, d, axis=0))
    f[_fixed(pb.nodes, pb.constr_node)] = 0.0
    return f


def _target(pb, rng):
    """Upstream gradient of a loss u . target: a smooth weight."""
    w = np.cos(pb.nodes @ rng.uniform(1.0, 6.0, size=(pb.dim, pb.dim)))
    w[pb.constr_node] = 0.0
    return w


def _ricker(t, freq, ampl):
    a = (math.pi * freq * t - math.pi) ** 2
    return ampl * (1.0 - 2.0 * a) * math.exp(-a)


def exact(case, seed):
    kind = case["kind"]
    out = lambda v: v.cpu().numpy()  # noqa: E731
    if kind == "batch":
        return _exact_batch(case, seed)
    pb, rng = _problem(case, seed)
    lam, mu = _lame(pb.E, pb.nu, pb.dim)
    A = _Operator(pb.nodes, pb.elems, lam, mu, _fixed(pb.nodes, pb.constr_node), pb.elem_scale)
    shape = pb.nodes.shape
    t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=A.dev).reshape(-1)  # noqa: E731
    if kind == "matvec":
        return out(A(t(rng.standard_normal(shape)))).reshape(shape)
    if kind in ("explicit", "implicit"):
        return _exact_time(case, pb, A, t)
    f = t(_load(pb, pb.face_p))
    u = A.solve(f)
    res = {"u": out(u).reshape(shape)}
    if kind == "static":
        if case["stress"]:
            res["stress"] = out(A.stress(u))
        return res
    ue = u[A.dofs]
    if kind == "compliance":
        g = -(ue * (A.K0 * ue[:, None, :]).sum(2)).sum(1)
        return dict(res, compliance=float(torch.dot(f, u)), gradient=out(g))
    w = A.solve(t(_target(pb, rng)))
    g = -(w[A.dofs] * (A.K0 * ue[:, None, :]).sum(2)).sum(1)
    return dict(res, d_scale=out(g), d_f=out(w).reshape(shape))


def _exact_time(case, pb, A, t):
    o = _time_options(case, pb)
    dt, b1, b2 = o["dt"], o["beta1"], o["beta2"]
    F1 = t(_load(pb, np.ones(len(pb.face_p))))
    m = A.assemble((RHO * A.V / (pb.dim + 1))[:, None].expand(-1, A.dofs.shape[1]))
    d, v, a = (torch.zeros_like(F1) for _ in range(3))
    rec = torch.as_tensor(_receivers(case, pb).astype(np.int64), device=A.dev) if case["receivers"] else None
    traces = []
    for n in range(1, case["steps"] + 1):
        d = d + dt * v + 0.5 * (1.0 - b2) * dt * dt * a
        v = v + (1.0 - b1) * dt * a
        r = _ricker(n * dt, o["freq"], o["ampl"]) * F1 - A(d)
        if b2 == 0.0:
            a = r / m
        else:
            a = A.solve(r, shift=m, factor=0.5 * b2 * dt * dt, tol=1e-15)
            d = d + 0.5 * b2 * dt * dt * a
        v = v + b1 * dt * a
        if rec is not None and n % 4 == 0:
            traces.append(v.reshape(pb.nodes.shape)[rec])
    res = {"u": d.cpu().numpy().reshape(pb.nodes.shape)}
    if rec is not None:
        res["traces"] = torch.stack(traces).cpu().numpy()
    return res


def _exact_batch(case, seed):
    """All plates as one block-diagonal system, one load case at a time."""
    insts = _plates(case, seed)
    off = np.cumsum([0] + [len(b.nodes) for b in insts])
    nodes = np.concatenate([b.nodes for b in insts])
    elems = np.concatenate([b.elems + o for b, o in zip(insts, off)])
    fixed = np.concatenate([_fixed(b.nodes, b.constr_node) for b in insts])
    lm = np.concatenate([np.tile(_lame(b.E, b.nu, 2), (len(b.elems), 1)) for b in insts])
    A = _Operator(nodes, elems, lm[:, 0], lm[:, 1], fixed)
    f = np.concatenate([b.f for b in insts])
    us = []
    for k in range(N_CASES):
        fk = torch.as_tensor(np.ascontiguousarray(f[:, k]).reshape(-1), device=A.dev)
        us.append(A.solve(fk).reshape(-1, 2).cpu().numpy())
    u = np.stack(us, 1)
    return [u[off[i]:off[i + 1]] for i in range(len(insts))]
