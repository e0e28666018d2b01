"""GPU: solves whose iterations run in one launch (a workgroup per patch on a
compute unit of its own) against dense FP64 solves of the oracle's operator,
and against the launch-per-kernel form, which plans of more than 256 patches
take."""
import threading

import numpy as np
import pytest

import cudafemproject_amd as F
from cudafemproject_amd.problem import cube_problem, plate_problem
from helpers import dense_K

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - b) / np.linalg.norm(b)


def _isolated():
    pb = cube_problem(3, convention=F.LOADS_PHYSICAL)
    pb.nodes = np.vstack([pb.nodes, [[2.0, 2.0, 2.0]]])
    return pb


def _scaled():
    pb = cube_problem(4, convention=F.LOADS_PHYSICAL)
    pb.elem_scale = np.random.default_rng(1).uniform(0.2, 1.0, pb.n_elems)
    return pb


CASES = {
    "plate-1": (lambda: plate_problem(12, 7), (0, 0)),               # one workgroup, no exchange
    "plate-2": (lambda: plate_problem(12, 7), (96, 256)),
    "plate-11": (lambda: plate_problem(12, 7), (16, 256)),
    "cube-1": (lambda: cube_problem(4), (0, 0)),
    "cube-8": (lambda: cube_problem(4), (48, 256)),
    "cube-24": (lambda: cube_problem(4), (16, 256)),                 # nodes of up to 24 patches
    "cube-ref-loads": (lambda: cube_problem(4, convention=F.LOADS_REFERENCE), (32, 256)),
    "isolated": (_isolated, (20, 256)),
    "scaled": (_scaled, (40, 256)),
}


@pytest.mark.parametrize("name", CASES)
def test_resident_solve_matches_dense(ctx, name):
    """FP64 to 1e-12 and mixed to 1e-9 on the residual; the meshes' condition
    numbers stay below 1e3, so 1e-9 and 1e-6 on the displacements."""
    make, tuning = CASES[name]
    pb = make()
    ctx.set_tuning(*tuning)
    try:
        ctx.set_problem(pb)
    finally:
        ctx.set_tuning(0, 0)
    f = ctx.rhs()
    live = np.zeros(pb.n_nodes, bool)
    live[pb.elems.ravel()] = True
    if live.all():
        u_ref = np.linalg.solve(dense_K(pb), f.ravel()).reshape(f.shape)
    else:
        sub = cube_problem(3, convention=F.LOADS_PHYSICAL)
        u_ref = np.zeros_like(f)
        u_ref[live] = np.linalg.solve(dense_K(sub), f[live].ravel()).reshape(-1, 3)
    print(f"[resident] {name}: {pb.n_elems} elements, tuning {tuning}", flush=True)
    for prec, tol, bound in ((F.FP64, 1e-12, 1e-9), (F.MIXED, 1e-9, 1e-6)):
        u, st = ctx.solve(prec, tol=tol, tol_kind=F.TOL_REL_RES)
        assert st["status"] == 0 and st["rel_res"] <= 1.01 * tol
        assert rel(u, u_ref) <= bound, (prec, rel(u, u_ref))
        assert np.all(u[~live] == 0.0)
        u2, st2 = ctx.solve(prec, tol=tol, tol_kind=F.TOL_REL_RES)
        assert np.array_equal(u, u2) and st2["iterations"] == st["iterations"]


@pytest.mark.parametrize("kind", [F.TOL_REF_GAMMA, F.TOL_REL_RES])
def test_resident_follows_the_launch_form(ctx, kind):
    """The same recurrence: the 9^3-hex cube in 6 patches (resident) and in 274
    (a launch per kernel) stops within one iteration, with the same result."""
    pb = cube_problem(9)
    out = []
    for tuning in ((0, 0), (16, 256)):
        ctx.set_tuning(*tuning)
        try:
            ctx.set_problem(pb)
        finally:
            ctx.set_tuning(0, 0)
        out.append(ctx.solve(F.FP64, tol=1e-20 if kind == F.TOL_REF_GAMMA else 1e-10, tol_kind=kind))
    (ua, sa), (ub, sb) = out
    assert abs(sa["iterations"] - sb["iterations"]) <= 1
    assert rel(ua, ub) <= 1e-8


@pytest.mark.parametrize("cap", [1, 7, 5000])
def test_resident_iteration_cap(ctx, cap):
    """The iteration cap stops the solve exactly, also past the iterations of
    one launch; 5000 iterations leave the converged solution."""
    pb = plate_problem(40, 20, convention=F.LOADS_PHYSICAL)
    ctx.set_problem(pb)
    f = ctx.rhs()
    u, st = ctx.solve_rhs(f, F.FP64, tol=0.0, max_iter=cap, raise_on_error=False)
    assert st["iterations"] == cap and st["status"] == -4
    if cap == 5000:
        v, _ = ctx.solve_rhs(f, F.FP64, tol=1e-11)
        assert rel(u, v) <= 1e-8


def test_resident_contexts_on_threads():
    """Two contexts of some 200 workgroups each solve at once: each gets the
    result it gets alone."""
    pbs = [cube_problem(28), cube_problem(29)]
    ctxs = [F.Context(0) for _ in pbs]
    try:
        want = []
        for c, pb in zip(ctxs, pbs):
            c.set_problem(pb)
            want.append(c.solve(F.FP64, tol=1e-9, tol_kind=F.TOL_REL_RES)[0])
        got = [[], []]

        def work(i):
            for _ in range(4):
                got[i].append(ctxs[i].solve(F.FP64, tol=1e-9, tol_kind=F.TOL_REL_RES)[0])

        ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for i in range(2):
            assert len(got[i]) == 4 and all(np.array_equal(u, want[i]) for u in got[i])
    finally:
        for c in ctxs:
            c.close()


def _run_with(ctx, pb, tuning, fn):
    ctx.set_tuning(*tuning)
    try:
        ctx.set_problem(pb)
    finally:
        ctx.set_tuning(0, 0)
    return fn()


# patches of more than 256 nodes (a strip per thread where every patch has at most
# 512 strips, else two elements), small ones, and more than 256 patches (a launch
# per kernel)
FORMS = [(1536, 512), (64, 256), (16, 256)]


@pytest.mark.parametrize("make", [lambda: cube_problem(9), lambda: plate_problem(70, 45)],
                         ids=["cube9", "plate70x45"])
def test_resident_wide_patches_solve(ctx, make):
    pb = make()
    u = [_run_with(ctx, pb, t, lambda: ctx.solve(F.FP64, tol=1e-11, tol_kind=F.TOL_REL_RES)[0])
         for t in FORMS]
    m = _run_with(ctx, pb, FORMS[0], lambda: ctx.solve(F.MIXED, tol=1e-9, tol_kind=F.TOL_REL_RES)[0])
    assert rel(u[0], u[2]) <= 1e-9 and rel(u[1], u[2]) <= 1e-9
    assert rel(m, u[2]) <= 1e-6


@pytest.mark.parametrize("precision,bound", [(F.FP64, 1e-11), (F.FP32, 2e-5)])
@pytest.mark.parametrize("quantity", [F.RECV_DISPLACEMENT, F.RECV_VELOCITY, F.RECV_ACCELERATION])
@pytest.mark.parametrize("make", [lambda: cube_problem(9), lambda: plate_problem(100, 60)],
                         ids=["cube9", "plate100x60"])
def test_resident_steps_match_launches(ctx, make, quantity, precision, bound):
    """Explicit steps in one launch against a launch per kernel, with damping,
    an odd number of steps, receivers on interface nodes and one node twice;
    twice in a row (the exchange words keep counting)."""
    pb = make()
    h = 1.0 / 9 if pb.dim == 3 else 1.0 / 100
    dt = 0.1 * h / np.sqrt(3 * 2e7 / 2400.0)
    opts = dict(rho=2400.0, dt=dt, endtime=61.5 * dt, wavelet_type=F.WAVELET_RICKER,
                freq=1.0 / (20 * dt), ampl=1e3, precision=precision,
                mass_convention=F.MASS_PHYSICAL, damping_alpha=0.3 / dt / 61)
    nodes = np.append(np.linspace(0, pb.n_nodes - 1, 40).astype(np.int32), 3).astype(np.int32)
    nodes[7] = 3

    def go():
        ctx.set_receivers(nodes, quantity, 3)
        ctx.dyn_run(**opts)
        u, st = ctx.dyn_run(**opts)
        assert st["steps"] == 61
        tr = ctx.traces()
        assert tr.shape[0] == 20 and np.array_equal(tr[:, 7], tr[:, -1])
        return u, tr

    res = [_run_with(ctx, pb, t, go) for t in FORMS]
    for u, tr in res[:2]:
        assert rel(u, res[2][0]) <= bound and rel(tr, res[2][1]) <= bound


def test_resident_steps_past_one_launch(ctx):
    """More steps than one launch holds (16384) equal, bitwise, two thirds of
    them continued: displacements after n steps do not depend on the launches."""
    pb = plate_problem(6, 4, convention=F.LOADS_PHYSICAL)
    ctx.set_problem(pb)
    dt = 1e-4
    opts = dict(rho=2400.0, dt=dt, precision=F.FP64, mass_convention=F.MASS_PHYSICAL)
    ctx.set_receivers(np.arange(pb.n_nodes, dtype=np.int32), F.RECV_DISPLACEMENT, 100)
    u1, st = ctx.dyn_run(endtime=20000.5 * dt, **opts)
    tr = ctx.traces()
    assert st["steps"] == 20000 and tr.shape[0] == 200
    assert np.array_equal(tr[-1], u1)
    u2, _ = ctx.dyn_run(endtime=16000.5 * dt, **opts)
    assert np.array_equal(tr[159], u2) and np.isfinite(u1).all()


@pytest.mark.parametrize("mode", [F.IMPLICIT_PHYSICAL, F.IMPLICIT_REFERENCE])
@pytest.mark.parametrize("make", [lambda: cube_problem(9), lambda: plate_problem(70, 45)],
                         ids=["cube9", "plate70x45"])
def test_resident_implicit_matches_launches(ctx, make, mode):
    """Implicit steps in one launch against a launch per kernel: Rayleigh
    damping (physical operator), receivers, nested solves to 1e-24 on gamma."""
    pb = make()
    h = 1.0 / 9 if pb.dim == 3 else 1.0 / 70
    dt = h / np.sqrt(3 * 2e7 / 2400.0)
    opts = dict(rho=2400.0, beta2=0.5, dt=dt, endtime=7.5 * dt, wavelet_type=F.WAVELET_RICKER,
                freq=1.0 / (3 * dt), ampl=1e3, mass_convention=F.MASS_PHYSICAL, implicit_mode=mode,
                pcg_eps=1e-24)
    if mode == F.IMPLICIT_PHYSICAL:
        opts.update(damping_alpha=0.1 / dt, damping_beta=0.2 * dt)
    nodes = np.linspace(0, pb.n_nodes - 1, 30).astype(np.int32)

    def go():
        ctx.set_receivers(nodes, F.RECV_VELOCITY, 2)
        u, st = ctx.dyn_run(**opts)
        assert st["steps"] == 7 and st["pcg_iterations"] > 7
        return u, ctx.traces()

    res = [_run_with(ctx, pb, t, go) for t in FORMS]
    for u, tr in res[:2]:
        assert rel(u, res[2][0]) <= 1e-9 and rel(tr, res[2][1]) <= 1e-9
