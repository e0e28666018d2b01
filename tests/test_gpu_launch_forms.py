"""GPU: the launch-per-kernel forms on meshes that otherwise run resident
(Context.set_resident): solves against the resident form, the explicit step in
one launch against the two-launch step, time steps and solves from captured
graphs against direct launches, the release of step graphs."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
from scipy.spatial import Delaunay

import cudafemproject_amd as F
from conftest import ROOT
from cudafemproject_amd import problem as P

pytestmark = pytest.mark.gpu

KW = dict(rho=1000.0, beta1=0.5, beta2=0.0, dt=2e-5, wavelet_type=F.WAVELET_RICKER, freq=500.0,
          ampl=1e3, mass_convention=F.MASS_PHYSICAL)


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - b) / np.linalg.norm(b)


@pytest.fixture
def launches(ctx):
    """The session's context in the launch form; no resident launch may run."""
    ctx.set_resident(F.RESIDENT_OFF)
    before = ctx.resident_info()
    yield ctx
    assert ctx.resident_info() == before
    ctx.set_resident(F.RESIDENT_AUTO)


def tuned(ctx, pb, tuning):
    ctx.set_tuning(*tuning)
    try:
        ctx.set_problem(pb)
    finally:
        ctx.set_tuning(0, 0)


def ragged(n=14):
    """Delaunay tetrahedra of a jittered grid: more strips than a third of the
    elements, and so in FP64 single elements per thread."""
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(float)
    x = g + rng.uniform(-0.25, 0.25, g.shape)
    t = Delaunay(x).simplices
    det = np.linalg.det(x[t][:, 1:] - x[t][:, :1])
    t = t[np.abs(det) > 0.05]
    ids = np.unique(t)
    new = np.full(len(x), -1)
    new[ids] = np.arange(len(ids))
    x, t = x[ids] / n, new[t].astype(np.int32)
    fixed = np.flatnonzero(x[:, 0] < 0.2).astype(np.int32)
    return P.Problem(nodes=x, elems=t, constr_node=fixed, constr_code=np.full(len(fixed), 7, np.int32),
                     E=2e7, nu=0.3)


@pytest.mark.parametrize("tuning", [(0, 0), (64, 256), (1536, 512), (3072, 1024)])
@pytest.mark.parametrize("make", [lambda: P.cube_problem(9), lambda: P.plate_problem(70, 45), ragged],
                         ids=["cube9", "plate70x45", "ragged"])
def test_launch_solves_match_resident(launches, make, tuning):
    """Condition numbers below 1e4: 1e-5 on the displacements at FP64 residuals
    of 1e-11 (1e-7) and 1e-9 (mixed), and twice in a row the same bits."""
    ctx, pb = launches, make()
    tuned(ctx, pb, tuning)
    f = np.random.default_rng(1).standard_normal((pb.n_nodes, pb.dim))
    opts = dict(tol_kind=F.TOL_REL_RES)
    got = [ctx.solve_rhs(f, p, tol=t, **opts)[0] for p, t in ((F.FP64, 1e-11), (F.MIXED, 1e-9)) * 2]
    assert np.array_equal(got[0], got[2]) and np.array_equal(got[1], got[3])
    with F.Context(0) as c:
        c.set_problem(pb)
        ref, _ = c.solve_rhs(f, F.FP64, tol=1e-11, **opts)
        assert c.resident_info() == (1, 0)
    assert rel(got[0], ref) <= 1e-7 and rel(got[1], ref) <= 1e-5


@pytest.mark.parametrize("alpha", [0.0, 30.0])
@pytest.mark.parametrize("precision", [F.FP64, F.FP32])
@pytest.mark.parametrize("tuning", [(0, 0), (1536, 512), (3072, 1024)])
@pytest.mark.parametrize("shape", ["column", "plate"])
def test_one_launch_step_matches_two_launch_step(launches, shape, tuning, precision, alpha):
    """Without receivers an explicit step is one patch launch whose interface
    nodes are corrected one launch late; with receivers it is the predictor
    launch plus the corrector launch (150 steps: two graph replays and single
    launches).  Both, and the resident steps, give the same displacements."""
    ctx = launches
    pb = (P.column_problem(8, 8, 24, 0.4, 0.4, 1.2, convention=F.LOADS_PHYSICAL, pressure=1.0)
          if shape == "column" else P.plate_problem(64, 32, convention=F.LOADS_PHYSICAL))
    tuned(ctx, pb, tuning)
    n = 150
    kw = dict(KW, precision=precision, damping_alpha=alpha, endtime=(n + 0.5) * KW["dt"])
    u1, st1 = ctx.dyn_run(**kw)
    ctx.set_receivers(np.array([0], np.int32), F.RECV_VELOCITY, 1)
    try:
        u2, st2 = ctx.dyn_run(**kw)
    finally:
        ctx.set_receivers([], F.RECV_DISPLACEMENT, 1)
    assert st1["steps"] == st2["steps"] == n and np.linalg.norm(u2) > 0
    bound = 1e-12 if precision == F.FP64 else 1e-5
    assert rel(u1, u2) <= bound
    with F.Context(0) as c:
        c.set_problem(pb)
        u3, _ = c.dyn_run(**kw)
        assert c.resident_info() == (1, 0)
    assert rel(u1, u3) <= bound


@pytest.mark.parametrize("receivers", [[], [5]])
@pytest.mark.parametrize("graph_steps", [1, 7, 64])
def test_explicit_graph_replays_match_eager(launches, graph_steps, receivers):
    """Steps captured in HIP graphs of several lengths (plus an eager tail)
    give bitwise the same trajectory as single launches."""
    ctx = launches
    ctx.set_problem(P.column_problem(2, 2, 12, 0.1, 0.1, 1.2, convention=F.LOADS_PHYSICAL, pressure=1e3))
    kw = dict(rho=1000.0, dt=5e-6, endtime=5e-4, wavelet_type=F.WAVELET_RICKER, freq=500.0, ampl=1.0)
    ctx.set_receivers(receivers, F.RECV_DISPLACEMENT, 1)
    try:
        a, _ = ctx.dyn_run(steps_per_graph=graph_steps, **kw)
        b, _ = ctx.dyn_run(steps_per_graph=100000, **kw)   # all steps eager
    finally:
        ctx.set_receivers([], F.RECV_DISPLACEMENT, 1)
    assert np.array_equal(a, b)


def test_implicit_step_graph_release(launches):
    """Implicit runs under many option sets (one dt each) leave their step
    graphs cached until more than 256 belong to other option sets; the run
    that releases them, and every run after, gives bitwise the results of the
    same options in a fresh context."""
    ctx = launches
    pb = P.column_problem(2, 2, 8, 0.1, 0.1, 0.4, convention=F.LOADS_PHYSICAL, pressure=1.0)
    ctx.set_problem(pb)
    kw = dict(KW, beta2=0.5, implicit_mode=F.IMPLICIT_PHYSICAL, pcg_eps=1e-8)

    def run(c, dt):
        u, st = c.dyn_run(**dict(kw, dt=dt, endtime=3.5 * dt))
        assert st["steps"] == 3
        return u

    u_first = run(ctx, 4e-5)
    for k in range(140):                         # 2 to 3 step graphs each
        run(ctx, 4e-5 * (1.0 + 0.001 * (k + 1)))
    u_again = run(ctx, 4e-5)
    u_other = run(ctx, 4e-5 * 1.0005)
    with F.Context(0) as c2:
        c2.set_resident(F.RESIDENT_OFF)
        c2.set_problem(pb)
        u_ref = run(c2, 4e-5)
        u_ref_other = run(c2, 4e-5 * 1.0005)
    assert np.array_equal(u_first, u_ref)
    assert np.array_equal(u_again, u_ref)
    assert np.array_equal(u_other, u_ref_other)


CHILD = r'''
import json, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import cudafemproject_amd as F
from cudafemproject_amd.problem import column_problem, cube_problem
out = {}
with F.Context(0) as c:
    c.set_resident(F.RESIDENT_OFF)
    c.set_problem(cube_problem(10, convention=F.LOADS_REFERENCE))
    for name, prec in (("fp64", F.FP64), ("mixed", F.MIXED)):
        u, s = c.solve(prec, tol=1e-10, tol_kind=F.TOL_REL_RES)
        out[name] = [u.ravel().tolist(), s["iterations"]]
    c.set_problem(column_problem(4, 4, 64, 0.025, 0.025, 0.4, convention=F.LOADS_PHYSICAL))
    for beta2, steps in ((0.0, 150), (0.5, 40)):
        for prec in (F.FP64, F.FP32):
            dt = 2e-6 if beta2 == 0 else 8e-6
            u, s = c.dyn_run(rho=1000.0, beta1=0.5, beta2=beta2, dt=dt, endtime=(steps + 0.5) * dt,
                             wavelet_type=F.WAVELET_RICKER, freq=2000.0, ampl=1e3, precision=prec,
                             mass_convention=F.MASS_PHYSICAL, implicit_mode=F.IMPLICIT_PHYSICAL,
                             pcg_eps=1e-8)
            out[f"dyn{beta2}/{prec}"] = [u.ravel().tolist(), s["steps"] * 100000 + s["pcg_iterations"]]
    assert c.resident_info() == (0, 0)
print(json.dumps(out))
'''


def test_no_graphs_matches_graphs():
    """Direct launches run the same kernels in the same order as the captured
    graphs: bitwise the same displacements and the same iterations."""
    def run(no_graphs):
        env = dict(os.environ)
        env.pop("FEMGPU_NO_GRAPHS", None)
        if no_graphs:
            env["FEMGPU_NO_GRAPHS"] = "1"
        r = subprocess.run([sys.executable, "-c", CHILD, ROOT], capture_output=True, text=True,
                           env=env, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.strip().splitlines()[-1])

    a, b = run(False), run(True)
    for k in a:
        assert a[k][1] == b[k][1], k
        assert np.array_equal(np.array(a[k][0]), np.array(b[k][0])), k


def test_launch_batch_matches_resident(launches):
    """FP64 lockstep batch, launch per iteration against resident: systems to
    1e-10 of plates whose condition numbers stay below 1e4."""
    insts = P.plate_batch(6, seed=3, nx_range=(20, 40), ny_range=(10, 20))
    rhs = [b.f for b in insts]
    P.load_batch(launches, insts)
    us, st, _ = launches.batch_solve(rhs, precision=F.FP64, tol=1e-10)
    assert np.all(st["status"] == 0)
    with F.Context(0) as c:
        P.load_batch(c, insts)
        ur, sr, _ = c.batch_solve(rhs, precision=F.FP64, tol=1e-10)
        assert np.all(sr["status"] == 0) and c.resident_info() == (1, 0)
    for a, b in zip(us, ur):
        assert rel(a, b) <= 1e-6


def test_modes_are_checked(ctx):
    with pytest.raises(F.FemGpuError):
        ctx.set_resident(17)
