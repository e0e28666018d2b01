"""Resident solves and steps on patches of up to 512 nodes, by strips (every patch
of at most 512) and by two elements per thread (a 13^3-hex cube has patches of
more), with a modulus in every element, against the default plan's form with
an element per thread.  Bounds: twice the solves' relative residuals; 60
explicit steps and 4 implicit ones of nested tolerance 1e-18 differ by the
order of sums."""
import numpy as np
import pytest

import cudafemproject_amd as F
from cudafemproject_amd.problem import cube_problem, plate_problem

pytestmark = pytest.mark.gpu

MESHES = {"strips": lambda: cube_problem(16, convention=F.LOADS_PHYSICAL),
          "elements": lambda: cube_problem(13, convention=F.LOADS_PHYSICAL),
          "plate": lambda: plate_problem(70, 45, convention=F.LOADS_PHYSICAL)}


@pytest.mark.parametrize("name", list(MESHES))
def test_forms(name):
    pb = MESHES[name]()
    rng = np.random.default_rng(3)
    pb.elem_scale = rng.uniform(0.5, 2.0, pb.n_elems)
    with F.Context(0) as c, F.Context(0) as d:
        c.set_problem(pb)
        d.set_tuning(1536, 512)
        d.set_problem(pb)
        f = c.rhs()
        u, _ = c.solve(F.FP64, tol=1e-12, tol_kind=F.TOL_REL_RES)
        for prec in (F.FP64, F.MIXED):
            v, st = d.solve(prec, tol=1e-10, tol_kind=F.TOL_REL_RES)
            assert np.linalg.norm(c.matvec(v - u)) <= 2e-10 * np.linalg.norm(f)
        h = 1e-3
        for kw, bound in ((dict(beta2=0.0, dt=1e-4, endtime=60.5e-4), {F.FP64: 1e-11, F.FP32: 2e-5}),
                          (dict(beta2=0.5, dt=h, endtime=4.5 * h, pcg_eps=1e-18,
                                implicit_mode=F.IMPLICIT_PHYSICAL, damping_alpha=0.5), {F.FP64: 1e-7})):
            for prec, b in bound.items():
                x, _ = c.dyn_run(rho=2400.0, beta1=0.5, precision=prec, **kw)
                y, _ = d.dyn_run(rho=2400.0, beta1=0.5, precision=prec, **kw)
                assert np.linalg.norm(x) > 0
                assert np.linalg.norm(x - y) <= b * np.linalg.norm(x)
