"""GPU: resident launches that do not complete.  The host leaves a workgroup out
of a launch, the others give up waiting for it (after 2 ms), every kernel ends,
and the call goes on in launches: the results are the launch form's, bit for
bit, also where the launch that failed continued earlier ones."""
import numpy as np
import pytest

import cudafemproject_amd as F
from cudafemproject_amd.problem import cube_problem, load_batch, plate_batch, plate_problem

pytestmark = pytest.mark.gpu

STEP = dict(rho=2400.0, wavelet_type=F.WAVELET_RICKER, ampl=1e3, mass_convention=F.MASS_PHYSICAL)


def _solve(precision, **kw):
    def run(c):
        c.set_problem(cube_problem(9))
        u, st = c.solve(precision, raise_on_error=False, **kw)
        return [u, st["status"], st["iterations"], st["outer_iterations"]]
    return run


def _steps(beta2, steps, precision=F.FP64, receivers=(), make=lambda: plate_problem(70, 45), dt=1e-5,
           tuning=(0, 0), **kw):
    def run(c):
        c.set_tuning(*tuning)
        c.set_problem(make())
        c.set_tuning(0, 0)
        c.set_receivers(list(receivers), F.RECV_VELOCITY, 3)
        u, st = c.dyn_run(beta2=beta2, dt=dt, endtime=(steps + 0.5) * dt if steps > 0 else -1e-30,
                          freq=1.0 / (20 * dt), precision=precision, raise_on_error=False,
                          **dict(STEP, **kw))
        tr = c.traces() if len(receivers) else 0
        c.set_receivers([], F.RECV_VELOCITY, 1)
        return [u, st["status"], st["steps"], st["pcg_iterations"], tr]
    return run


def _batch(precision):
    insts = plate_batch(3, seed=3, nx_range=(30, 40), ny_range=(20, 30))

    def run(c):
        load_batch(c, insts)
        us, st, _ = c.batch_solve([b.f for b in insts], precision=precision, tol=1e-9)
        return us + [st["status"], st["iterations"]]
    return run


IMPL = dict(implicit_mode=F.IMPLICIT_PHYSICAL, pcg_eps=1e-20)
REL = dict(tol=1e-9, tol_kind=F.TOL_REL_RES)
FIRST = {
    "fp64": _solve(F.FP64, **REL),
    "fp32": _solve(F.FP32, tol=1e-4, tol_kind=F.TOL_REL_RES),
    "mixed": _solve(F.MIXED, **REL),
    "explicit": _steps(0.0, 60),
    "explicit-traces": _steps(0.0, 60, F.FP32, receivers=(0, 700, 3000)),
    "implicit": _steps(0.5, 5, **IMPL),
    "implicit-traces": _steps(0.5, 6, receivers=(0, 700, 3000), **IMPL),
    "batch": _batch(F.FP64),
    "batch-mixed": _batch(F.MIXED),
}
# in the third launch
LATER = {
    "fp32-capped": _solve(F.FP32, tol=0.0, max_iter=12500),
    "mixed": _solve(F.MIXED, tol=1e-12, tol_kind=F.TOL_REL_RES),
    "explicit": _steps(0.0, 40000, make=lambda: plate_problem(6, 4), tuning=(16, 256)),
    "implicit-relaxation": _steps(0.5, 0, make=lambda: plate_problem(12, 7), tuning=(16, 256), dt=1e-4,
                                  relax_reference=0, max_steps=8, **IMPL),
}


@pytest.mark.parametrize("mode,name", [(F.RESIDENT_TEST_LOSE, n) for n in FIRST] +
                         [(F.RESIDENT_TEST_LOSE_LATER, n) for n in LATER])
def test_lost_workgroup(mode, name):
    run = (FIRST if mode == F.RESIDENT_TEST_LOSE else LATER)[name]
    print(f"[lost] {name}", flush=True)
    with F.Context(0) as c:
        c.set_resident(F.RESIDENT_OFF)
        want = run(c)
        assert c.resident_info() == (0, 0)
    with F.Context(0) as c:
        c.set_resident(mode)
        for _ in range(2):
            got = run(c)
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
        done, lost = c.resident_info()
        assert lost >= 1 and done == (0 if mode == F.RESIDENT_TEST_LOSE else 2)
        c.set_resident(F.RESIDENT_AUTO)
        again = run(c)
        assert c.resident_info()[0] > done and c.resident_info()[1] == lost
        assert all(np.all(np.isfinite(np.asarray(a, float))) for a in again)


@pytest.mark.parametrize("name", ["fp64", "fp32", "mixed", "implicit", "implicit-traces"])
def test_late_abort(name):
    """A workgroup that gives up in the last exchange, when the one that reports
    the scalars has them all and has ended: its part of the result is missing,
    and the host is told."""
    run = FIRST[name]
    print(f"[late] {name}", flush=True)
    with F.Context(0) as c:
        c.set_resident(F.RESIDENT_OFF)
        want = run(c)
    with F.Context(0) as c:
        c.set_resident(F.RESIDENT_TEST_LATE)
        got = run(c)
        assert c.resident_info() == (0, 1)
        assert all(np.array_equal(a, b) for a, b in zip(got, want))


def test_small_launches_side_by_side():
    """Four contexts whose launches take some 60 units each are admitted together:
    solves, explicit and implicit steps in four threads give the bits that each
    gives alone, and no launch is given up."""
    import threading
    jobs = [("fp64", lambda: cube_problem(17)), ("mixed", lambda: cube_problem(18)),
            ("explicit", lambda: cube_problem(16)), ("implicit", lambda: cube_problem(15))]

    def run(c, kind):
        if kind in ("fp64", "mixed"):
            return c.solve(F.FP64 if kind == "fp64" else F.MIXED, **REL)[0]
        dt = 2e-5
        return c.dyn_run(beta2=0.5 if kind == "implicit" else 0.0, dt=dt, freq=1.0 / (20 * dt),
                         endtime=(8 if kind == "implicit" else 400.5) * dt, **dict(STEP, **IMPL))[0]

    ctxs = [F.Context(0) for _ in jobs]
    try:
        for c, (_, make) in zip(ctxs, jobs):
            c.set_problem(make())
        want = [run(c, k) for c, (k, _) in zip(ctxs, jobs)]
        got = [[] for _ in jobs]

        def work(i):
            for _ in range(6):
                got[i].append(run(ctxs[i], jobs[i][0]))

        ts = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for i, c in enumerate(ctxs):
            assert len(got[i]) == 6 and all(np.array_equal(u, want[i]) for u in got[i])
            assert c.resident_info()[1] == 0
    finally:
        for c in ctxs:
            c.close()


def test_way_back():
    """After a launch that was given up 64 calls of any kind go in launches, then
    one tries again; after the second 128."""
    small = plate_batch(1, seed=1, nx_range=(30, 31), ny_range=(20, 21))
    with F.Context(0) as c:
        c.set_problem(plate_problem(40, 20))
        load_batch(c, small)
        calls = [lambda: c.solve(F.FP64, **REL), lambda: c.solve(F.MIXED, **REL),
                 lambda: c.dyn_run(dt=1e-5, endtime=3.5e-5, **STEP),
                 lambda: c.dyn_run(dt=1e-5, endtime=3.5e-5, beta2=0.5, **dict(STEP, **IMPL)),
                 lambda: c.batch_solve([small[0].f], precision=F.FP64, tol=1e-6)]
        for f in calls:
            f()
        assert c.resident_info()[1] == 0
        done = c.resident_info()[0]
        c.set_resident(F.RESIDENT_TEST_LOSE)
        lost = []
        for k in range(200):
            before = c.resident_info()[1]
            calls[k % 5]()
            if c.resident_info()[1] > before:
                lost.append(k)
        assert lost == [0, 65, 194] and c.resident_info() == (done, 3)
