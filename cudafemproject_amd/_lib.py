"""ctypes binding of the femgpu C-ABI (include/femgpu.h).

The shared library ``libfemgpu.so`` is built in-tree next to this file
(``cudafemproject_amd.build.build_library``).  Loading fails loudly when it is
missing: there is no CPU fallback anywhere in the product path.
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np

LIB_NAME = "libfemgpu.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)

# Status codes (femgpu.h)
OK = 0
E_ARG, E_HIP, E_NONFINITE, E_MAXIT, E_BREAKDOWN, E_BAD_MESH, E_STATE, E_NOMEM, E_UNSUPPORTED = (
    -1, -2, -3, -4, -5, -6, -7, -8, -9)
E_STAGNATION = -10
STATUS_NAMES = {0: "OK", -1: "E_ARG", -2: "E_HIP", -3: "E_NONFINITE", -4: "E_MAXIT",
                -5: "E_BREAKDOWN", -6: "E_BAD_MESH", -7: "E_STATE", -8: "E_NOMEM",
                -9: "E_UNSUPPORTED", -10: "E_STAGNATION"}

FP64, FP32, MIXED = 0, 1, 2
TOL_REF_GAMMA, TOL_REL_RES = 0, 1
CG_STANDARD, CG_SINGLE_REDUCTION = 0, 1
BATCH_LOCKSTEP, BATCH_PERSISTENT = 0, 1
RESIDENT_AUTO, RESIDENT_OFF = 0, 1
RESIDENT_TEST_LOSE, RESIDENT_TEST_LOSE_LATER, RESIDENT_TEST_LATE, RESIDENT_TEST_SHORT_WAITS = 2, 3, 4, 5
LOADS_REFERENCE, LOADS_PHYSICAL = 0, 1
MASS_REFERENCE, MASS_PHYSICAL = 0, 1
WAVELET_NONE, WAVELET_RICKER, WAVELET_BERLAGE = 0, 1, 2
IMPLICIT_REFERENCE, IMPLICIT_PHYSICAL = 0, 1
RECV_DISPLACEMENT, RECV_VELOCITY, RECV_ACCELERATION = 0, 1, 2


class SolveOpts(C.Structure):
    _fields_ = [("precision", C.c_int), ("tol_kind", C.c_int), ("tol", C.c_double),
                ("max_iter", C.c_int), ("inner_tol", C.c_double), ("check_every", C.c_int),
                ("recurrence", C.c_int), ("batch_schedule", C.c_int)]


class Stats(C.Structure):
    _fields_ = [("status", C.c_int), ("iterations", C.c_int), ("outer_iterations", C.c_int),
                ("rel_res", C.c_double), ("gamma_ratio", C.c_double), ("solve_ms", C.c_double)]


class DynOpts(C.Structure):
    _fields_ = [("rho", C.c_double), ("beta1", C.c_double), ("beta2", C.c_double),
                ("dt", C.c_double), ("endtime", C.c_double), ("wavelet_type", C.c_int),
                ("wavelet_freq", C.c_double), ("wavelet_timeshift", C.c_double),
                ("wavelet_ampl", C.c_double), ("precision", C.c_int),
                ("mass_convention", C.c_int), ("implicit_mode", C.c_int),
                ("pcg_eps", C.c_double), ("steps_per_graph", C.c_int),
                ("damping_alpha", C.c_double), ("damping_beta", C.c_double),
                ("relax_reference", C.c_int), ("max_steps", C.c_int)]


class DynStats(C.Structure):
    _fields_ = [("status", C.c_int), ("steps", C.c_int), ("pcg_iterations", C.c_int),
                ("run_ms", C.c_double)]


class BatchStat(C.Structure):
    _fields_ = [("status", C.c_int), ("iterations", C.c_int), ("replacements", C.c_int),
                ("pad", C.c_int), ("rel_res", C.c_double)]


_P = C.c_void_p
_D = C.POINTER(C.c_double)
_I = C.POINTER(C.c_int32)
_L = C.POINTER(C.c_int64)

# name -> (restype, argtypes); the list of exported symbols of include/femgpu.h
SIGNATURES = {
    "femgpu_create": (C.c_int, [C.POINTER(C.c_void_p), C.c_int]),
    "femgpu_destroy": (None, [_P]),
    "femgpu_last_error": (C.c_char_p, [_P]),
    "femgpu_set_stream": (C.c_int, [_P, _P]),
    "femgpu_sync": (C.c_int, [_P]),
    "femgpu_set_resident": (C.c_int, [_P, C.c_int]),
    "femgpu_resident_info": (C.c_int, [_P, _L]),
    "femgpu_set_mesh": (C.c_int, [_P, C.c_int, C.c_int64, _D, C.c_int64, _I]),
    "femgpu_set_tuning": (C.c_int, [_P, C.c_int, C.c_int]),
    "femgpu_autotune": (C.c_int, [_P, C.c_int, C.POINTER(C.c_int), C.POINTER(C.c_int),
                                  C.POINTER(C.c_double)]),
    "femgpu_plan_info": (C.c_int, [C.c_int, C.c_int64, _D, C.c_int64, _I, C.c_int, C.c_int, _L]),
    "femgpu_set_material": (C.c_int, [_P, C.c_double, C.c_double, _D]),
    "femgpu_set_constraints": (C.c_int, [_P, C.c_int64, _I, _I]),
    "femgpu_set_pressure_faces": (C.c_int, [_P, C.c_int64, _I, _I, _D, _D]),
    "femgpu_set_nodal_loads": (C.c_int, [_P, C.c_int64, _I, _D]),
    "femgpu_set_load_convention": (C.c_int, [_P, C.c_int]),
    "femgpu_set_extra_rhs": (C.c_int, [_P, _D]),
    "femgpu_matvec": (C.c_int, [_P, C.c_int, _D, _D]),
    "femgpu_matvec_noalloc": (C.c_int, [_P, C.c_int, C.c_void_p, C.c_void_p]),
    "femgpu_diag": (C.c_int, [_P, _D]),
    "femgpu_rhs": (C.c_int, [_P, _D]),
    "femgpu_matvec_repeat": (C.c_int, [_P, C.c_int, C.c_int]),
    "femgpu_time_matvec": (C.c_int, [_P, C.c_int, C.c_int, _D]),
    "femgpu_default_solve_opts": (C.c_int, [C.POINTER(SolveOpts)]),
    "femgpu_solve_static": (C.c_int, [_P, C.POINTER(SolveOpts), _D, C.POINTER(Stats)]),
    "femgpu_stress": (C.c_int, [_P, _D, _D]),
    "femgpu_strain": (C.c_int, [_P, _D, _D]),
    "femgpu_element_energy": (C.c_int, [_P, _D, _D]),
    "femgpu_batch_set_mesh": (C.c_int, [_P, C.c_int, C.c_int, _L, _D, _L, _I]),
    "femgpu_batch_set_material": (C.c_int, [_P, _D, _D]),
    "femgpu_batch_set_constraints": (C.c_int, [_P, _L, _I, _I]),
    "femgpu_batch_solve": (C.c_int, [_P, C.c_int, _D, C.POINTER(SolveOpts), _D,
                                     C.POINTER(BatchStat), _D]),
    "femgpu_set_receivers": (C.c_int, [_P, C.c_int, _I, C.c_int, C.c_int]),
    "femgpu_get_traces": (C.c_int, [_P, _D, C.c_int64, C.POINTER(C.c_int)]),
    "femgpu_write_segy": (C.c_int, [C.c_char_p, C.POINTER(C.c_float), C.c_int, C.c_int, C.c_float,
                                    C.c_int]),
    "femgpu_solve_rhs": (C.c_int, [_P, C.POINTER(SolveOpts), _D, _D, C.POINTER(Stats)]),
    "femgpu_material_grad": (C.c_int, [_P, _D, _D, _D]),
    "femgpu_compliance_grad": (C.c_int, [_P, C.POINTER(SolveOpts), _D, _D, _D, C.POINTER(Stats)]),
    "femgpu_default_dyn_opts": (C.c_int, [C.POINTER(DynOpts)]),
    "femgpu_dyn_run": (C.c_int, [_P, C.POINTER(DynOpts), _D, C.POINTER(DynStats)]),
    "femgpu_autotune_dyn": (C.c_int, [_P, C.POINTER(DynOpts), C.c_int, C.POINTER(C.c_int),
                                      C.POINTER(C.c_int), C.POINTER(C.c_double)]),
}

_lib = None


def load_library(path: str | None = None):
    """Load libfemgpu.so (raises if it is not built)."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    p = path or LIB_PATH
    if not os.path.exists(p):
        raise RuntimeError(
            f"{p} is not built: run __graft_entry__.build() (hipcc --offload-arch=gfx950); "
            "there is no CPU fallback")
    lib = C.CDLL(p)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if path is None:
        _lib = lib
    return lib


def plan_info(nodes: np.ndarray, elems: np.ndarray, elems_per_patch: int = 0,
              patch_threads: int = 0) -> dict:
    """The patch plan femgpu_set_mesh builds for a mesh at a tuning (host
    only, no device needed)."""
    lib = load_library()
    nodes = np.ascontiguousarray(nodes, dtype=np.float64)
    elems = np.ascontiguousarray(elems, dtype=np.int32)
    info = np.zeros(6, np.int64)
    st = lib.femgpu_plan_info(nodes.shape[1], nodes.shape[0], _dp(nodes), elems.shape[0],
                              _ip(elems), elems_per_patch, patch_threads,
                              info.ctypes.data_as(_L))
    if st != OK:
        raise FemGpuError(st, "femgpu_plan_info")
    keys = ("patches", "owned", "interface", "slots", "elems_per_patch", "max_patch_nodes")
    return dict(zip(keys, (int(v) for v in info)))


class FemGpuError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"femgpu error {STATUS_NAMES.get(code, code)}: {msg}")
        self.code = code


def _dp(a: np.ndarray):
    return a.ctypes.data_as(_D)


def _ip(a: np.ndarray):
    return a.ctypes.data_as(_I)


class Context:
    """One femgpu context (one device, one stream)."""

    def __init__(self, device: int = 0):
        self.lib = load_library()
        h = C.c_void_p()
        st = self.lib.femgpu_create(C.byref(h), device)
        if st != OK:
            raise FemGpuError(st, "femgpu_create failed (no HIP device?)")
        self.h = h
        self.dim = 0
        self.n_nodes = 0
        self.n_elems = 0

    def close(self):
        if getattr(self, "h", None):
            self.lib.femgpu_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.close()

    def _check(self, st: int, what: str):
        if st != OK:
            msg = self.lib.femgpu_last_error(self.h)
            raise FemGpuError(st, f"{what}: {msg.decode() if msg else ''}")

    # --- problem -----------------------------------------------------------
    def set_mesh(self, nodes: np.ndarray, elems: np.ndarray):
        nodes = np.ascontiguousarray(nodes, dtype=np.float64)
        elems = np.ascontiguousarray(elems, dtype=np.int32)
        dim = nodes.shape[1]
        self._check(self.lib.femgpu_set_mesh(self.h, dim, nodes.shape[0], _dp(nodes),
                                             elems.shape[0], _ip(elems)), "set_mesh")
        self.dim, self.n_nodes, self.n_elems = dim, nodes.shape[0], elems.shape[0]

    def set_tuning(self, elems_per_patch: int = 0, patch_threads: int = 0):
        self._check(self.lib.femgpu_set_tuning(self.h, elems_per_patch, patch_threads), "set_tuning")

    def autotune(self, precision: int = MIXED) -> dict:
        """femgpu_autotune: pick and apply the fastest patch tuning for the
        current problem (cached per mesh)."""
        e, t, ms = C.c_int(0), C.c_int(0), C.c_double(0)
        self._check(self.lib.femgpu_autotune(self.h, precision, C.byref(e), C.byref(t),
                                             C.byref(ms)), "autotune")
        return {"elems_per_patch": e.value, "patch_threads": t.value,
                "ms_per_iteration": ms.value}

    def set_material(self, E: float, nu: float, elem_scale: np.ndarray | None = None):
        if elem_scale is not None:
            elem_scale = np.ascontiguousarray(elem_scale, dtype=np.float64)
            assert elem_scale.shape == (self.n_elems,)
            p = _dp(elem_scale)
        else:
            p = None
        self._check(self.lib.femgpu_set_material(self.h, E, nu, p), "set_material")

    def set_constraints(self, nodes: np.ndarray, codes: np.ndarray):
        nodes = np.ascontiguousarray(nodes, dtype=np.int32)
        codes = np.ascontiguousarray(codes, dtype=np.int32)
        self._check(self.lib.femgpu_set_constraints(self.h, len(nodes), _ip(nodes), _ip(codes)),
                    "set_constraints")

    def set_pressure_faces(self, face_nodes, adj_elem, normals, pressures):
        fn = np.ascontiguousarray(face_nodes, dtype=np.int32)
        ae = np.ascontiguousarray(adj_elem, dtype=np.int32)
        nr = np.ascontiguousarray(normals, dtype=np.float64)
        pr = np.ascontiguousarray(pressures, dtype=np.float64)
        self._check(self.lib.femgpu_set_pressure_faces(self.h, len(ae), _ip(fn), _ip(ae), _dp(nr),
                                                       _dp(pr)), "set_pressure_faces")

    def set_nodal_loads(self, nodes, vecs):
        nd = np.ascontiguousarray(nodes, dtype=np.int32)
        vc = np.ascontiguousarray(vecs, dtype=np.float64)
        self._check(self.lib.femgpu_set_nodal_loads(self.h, len(nd), _ip(nd), _dp(vc)),
                    "set_nodal_loads")

    def set_load_convention(self, conv: int):
        self._check(self.lib.femgpu_set_load_convention(self.h, conv), "set_load_convention")

    def set_extra_rhs(self, f: np.ndarray | None):
        if f is None:
            self._check(self.lib.femgpu_set_extra_rhs(self.h, None), "set_extra_rhs")
            return
        f = np.ascontiguousarray(f, dtype=np.float64).reshape(-1)
        assert f.size == self.n_nodes * self.dim
        self._check(self.lib.femgpu_set_extra_rhs(self.h, _dp(f)), "set_extra_rhs")

    def set_problem(self, pb):
        """Load a `Problem` (cudafemproject_amd.problem) into the context."""
        self.set_mesh(pb.nodes, pb.elems)
        self.set_material(pb.E, pb.nu, pb.elem_scale)
        if len(pb.constr_node):
            self.set_constraints(pb.constr_node, pb.constr_code)
        if len(pb.face_adj):
            self.set_pressure_faces(pb.face_nodes, pb.face_adj, pb.face_normal, pb.face_p)
        if len(pb.load_node):
            self.set_nodal_loads(pb.load_node, pb.load_vec)
        self.set_load_convention(pb.convention)
        if pb.extra_rhs is not None:
            self.set_extra_rhs(pb.extra_rhs)

    # --- operators -----------------------------------------------------------
    def matvec(self, x: np.ndarray, precision: int = FP64) -> np.ndarray:
        x = np.ascontiguousarray(x, dtype=np.float64).reshape(self.n_nodes, self.dim)
        y = np.zeros_like(x)
        self._check(self.lib.femgpu_matvec(self.h, precision, _dp(x), _dp(y)), "matvec")
        return y

    def diag(self) -> np.ndarray:
        d = np.zeros((self.n_nodes, self.dim))
        self._check(self.lib.femgpu_diag(self.h, _dp(d)), "diag")
        return d

    def rhs(self) -> np.ndarray:
        f = np.zeros((self.n_nodes, self.dim))
        self._check(self.lib.femgpu_rhs(self.h, _dp(f)), "rhs")
        return f

    def matvec_repeat(self, precision: int, reps: int):
        self._check(self.lib.femgpu_matvec_repeat(self.h, precision, reps), "matvec_repeat")

    def time_matvec(self, precision: int, reps: int) -> float:
        ms = C.c_double(0)
        self._check(self.lib.femgpu_time_matvec(self.h, precision, reps, C.byref(ms)), "time_matvec")
        return ms.value

    def set_stream(self, stream_ptr: int | None):
        self._check(self.lib.femgpu_set_stream(self.h, C.c_void_p(stream_ptr) if stream_ptr else None),
                    "set_stream")

    def sync(self):
        self._check(self.lib.femgpu_sync(self.h), "sync")

    def set_resident(self, mode: int = RESIDENT_AUTO):
        self._check(self.lib.femgpu_set_resident(self.h, mode), "set_resident")

    def resident_info(self) -> tuple[int, int]:
        """Launches that stayed on the chip: (completed, given up)."""
        n = (C.c_int64 * 2)()
        self._check(self.lib.femgpu_resident_info(self.h, n), "resident_info")
        return n[0], n[1]

    # --- solves ----------------------------------------------------------------
    def _opts(self, precision, tol, tol_kind, max_iter, inner_tol, check_every,
              recurrence=CG_STANDARD) -> SolveOpts:
        o = SolveOpts()
        self.lib.femgpu_default_solve_opts(C.byref(o))
        o.precision, o.tol, o.tol_kind, o.max_iter = precision, tol, tol_kind, max_iter
        o.inner_tol, o.check_every, o.recurrence = inner_tol, check_every, recurrence
        return o

    @staticmethod
    def _stats(s: Stats) -> dict:
        return {"status": s.status, "iterations": s.iterations,
                "outer_iterations": s.outer_iterations, "rel_res": s.rel_res,
                "gamma_ratio": s.gamma_ratio, "solve_ms": s.solve_ms}

    def solve(self, precision: int = FP64, tol: float = 1e-8, tol_kind: int = TOL_REF_GAMMA,
              max_iter: int = 0, inner_tol: float = 0.1, check_every: int = 64,
              raise_on_error: bool = True, recurrence: int = CG_STANDARD):
        o = self._opts(precision, tol, tol_kind, max_iter, inner_tol, check_every, recurrence)
        u = np.zeros((self.n_nodes, self.dim))
        s = Stats()
        st = self.lib.femgpu_solve_static(self.h, C.byref(o), _dp(u), C.byref(s))
        if raise_on_error:
            self._check(st, "solve_static")
        return u, self._stats(s)

    def solve_rhs(self, f: np.ndarray, precision: int = FP64, tol: float = 1e-8,
                  tol_kind: int = TOL_REL_RES, max_iter: int = 0, inner_tol: float = 0.1,
                  check_every: int = 64, recurrence: int = CG_STANDARD,
                  raise_on_error: bool = True):
        """Solve K u = f for an explicit right-hand side (n_nodes x dim).
        raise_on_error=False returns the solution and stats of a solve that
        stopped with an error status (stats["status"])."""
        f = np.ascontiguousarray(f, dtype=np.float64).reshape(self.n_nodes, self.dim)
        o = self._opts(precision, tol, tol_kind, max_iter, inner_tol, check_every, recurrence)
        u = np.zeros((self.n_nodes, self.dim))
        s = Stats()
        st = self.lib.femgpu_solve_rhs(self.h, C.byref(o), _dp(f), _dp(u), C.byref(s))
        if raise_on_error or st in (E_ARG, E_HIP, E_STATE, E_NOMEM):
            self._check(st, "solve_rhs")
        return u, self._stats(s)

    def material_grad(self, u: np.ndarray, w: np.ndarray) -> np.ndarray:
        """g_e = -w_e' K~_e^0 u_e: dL/ds_e for adjoint solution w."""
        u = np.ascontiguousarray(u, dtype=np.float64)
        w = np.ascontiguousarray(w, dtype=np.float64)
        g = np.zeros(self.n_elems)
        self._check(self.lib.femgpu_material_grad(self.h, _dp(u), _dp(w), _dp(g)), "material_grad")
        return g

    def compliance_grad(self, precision: int = FP64, tol: float = 1e-8,
                        tol_kind: int = TOL_REL_RES, max_iter: int = 0, inner_tol: float = 0.1,
                        check_every: int = 64, recurrence: int = CG_STANDARD):
        """C = f'u and dC/ds_e from one solve; returns (C, g, u, stats)."""
        o = self._opts(precision, tol, tol_kind, max_iter, inner_tol, check_every, recurrence)
        u = np.zeros((self.n_nodes, self.dim))
        g = np.zeros(self.n_elems)
        c = C.c_double(0)
        s = Stats()
        self._check(self.lib.femgpu_compliance_grad(self.h, C.byref(o), _dp(u), C.byref(c), _dp(g),
                                                    C.byref(s)), "compliance_grad")
        return c.value, g, u, self._stats(s)

    # --- batched solves ---------------------------------------------------------
    def batch_set_mesh(self, meshes):
        """meshes: list of (nodes (n_i, dim), elems (m_i, dim+1) instance-local ids)."""
        dim = int(np.asarray(meshes[0][0]).shape[1])
        noff = np.zeros(len(meshes) + 1, np.int64)
        eoff = np.zeros(len(meshes) + 1, np.int64)
        for i, (nd, el) in enumerate(meshes):
            noff[i + 1] = noff[i] + len(nd)
            eoff[i + 1] = eoff[i] + len(el)
        nodes = np.ascontiguousarray(np.concatenate([np.asarray(m[0], np.float64) for m in meshes]))
        elems = np.ascontiguousarray(np.concatenate([np.asarray(m[1], np.int32) for m in meshes]))
        self._check(self.lib.femgpu_batch_set_mesh(self.h, dim, len(meshes), noff.ctypes.data_as(_L),
                                                   _dp(nodes), eoff.ctypes.data_as(_L), _ip(elems)),
                    "batch_set_mesh")
        self._batch = (dim, noff)

    def batch_set_material(self, E, nu):
        E = np.ascontiguousarray(E, np.float64)
        nu = np.ascontiguousarray(nu, np.float64)
        self._check(self.lib.femgpu_batch_set_material(self.h, _dp(E), _dp(nu)), "batch_set_material")

    def batch_set_constraints(self, cons):
        """cons: list of (nodes, codes) per instance (instance-local node ids)."""
        off = np.zeros(len(cons) + 1, np.int64)
        for i, (n, _) in enumerate(cons):
            off[i + 1] = off[i] + len(n)
        nodes = np.ascontiguousarray(np.concatenate([np.asarray(c[0], np.int32) for c in cons]))
        codes = np.ascontiguousarray(np.concatenate([np.asarray(c[1], np.int32) for c in cons]))
        self._check(self.lib.femgpu_batch_set_constraints(self.h, off.ctypes.data_as(_L), _ip(nodes),
                                                          _ip(codes)), "batch_set_constraints")

    def batch_solve(self, rhs, precision: int = MIXED, tol: float = 1e-8, max_iter: int = 0,
                    inner_tol: float = 0.1, raise_on_error: bool = True,
                    schedule: int = BATCH_LOCKSTEP):
        """rhs: list of (n_i, n_rhs, dim) arrays.  Returns (list of u arrays of
        the same shapes, stats as a structured array (n_inst, n_rhs), device ms).
        schedule: BATCH_LOCKSTEP (every instance over the whole GPU, graph
        replays) or BATCH_PERSISTENT (one workgroup per instance, one launch)."""
        dim, noff = self._batch
        nr = int(np.asarray(rhs[0]).shape[1])
        f = np.ascontiguousarray(np.concatenate([np.asarray(r, np.float64).reshape(-1, nr, dim)
                                                 for r in rhs]))
        assert f.shape[0] == noff[-1]
        u = np.zeros_like(f)
        st = (BatchStat * (len(rhs) * nr))()
        o = self._opts(precision, tol, TOL_REL_RES, max_iter, inner_tol, 32)
        o.batch_schedule = schedule
        ms = C.c_double(0)
        code = self.lib.femgpu_batch_solve(self.h, nr, _dp(f), C.byref(o), _dp(u), st, C.byref(ms))
        if raise_on_error:
            self._check(code, "batch_solve")
        stats = np.array([(x.status, x.iterations, x.replacements, x.rel_res) for x in st],
                         dtype=[("status", "i4"), ("iterations", "i4"), ("replacements", "i4"),
                                ("rel_res", "f8")]).reshape(len(rhs), nr)
        us = [u[noff[i]:noff[i + 1]] for i in range(len(rhs))]
        return us, stats, ms.value

    def set_receivers(self, nodes, quantity: int = RECV_DISPLACEMENT, every: int = 1):
        nodes = np.ascontiguousarray(nodes, dtype=np.int32)
        self._check(self.lib.femgpu_set_receivers(self.h, len(nodes), _ip(nodes) if len(nodes) else None,
                                                  quantity, every), "set_receivers")
        self._n_recv = len(nodes)

    def traces(self) -> np.ndarray:
        """Receiver traces of the last dyn_run: (n_samples, n_receivers, dim)."""
        n = C.c_int(0)
        self._check(self.lib.femgpu_get_traces(self.h, None, 0, C.byref(n)), "get_traces")
        out = np.zeros((n.value, getattr(self, "_n_recv", 0), self.dim))
        self._check(self.lib.femgpu_get_traces(self.h, _dp(out), out.size, C.byref(n)), "get_traces")
        return out

    def stress(self, u: np.ndarray) -> np.ndarray:
        u = np.ascontiguousarray(u, dtype=np.float64)
        nv = 3 * (self.dim - 1)
        s = np.zeros((self.n_elems, nv))
        self._check(self.lib.femgpu_stress(self.h, _dp(u), _dp(s)), "stress")
        return s

    def strain(self, u: np.ndarray) -> np.ndarray:
        """Per-element engineering strain B u_e (n_elems, 3(dim-1))."""
        u = np.ascontiguousarray(u, dtype=np.float64)
        nv = 3 * (self.dim - 1)
        s = np.zeros((self.n_elems, nv))
        self._check(self.lib.femgpu_strain(self.h, _dp(u), _dp(s)), "strain")
        return s

    def element_energy(self, u: np.ndarray) -> np.ndarray:
        u = np.ascontiguousarray(u, dtype=np.float64)
        e = np.zeros(self.n_elems)
        self._check(self.lib.femgpu_element_energy(self.h, _dp(u), _dp(e)), "element_energy")
        return e

    @staticmethod
    def _dyn_opts(lib, rho, beta1, beta2, dt, endtime, wavelet_type, freq, timeshift, ampl,
                  precision, mass_convention, implicit_mode, pcg_eps, steps_per_graph,
                  damping_alpha, damping_beta, relax_reference, max_steps):
        o = DynOpts()
        lib.femgpu_default_dyn_opts(C.byref(o))
        o.damping_alpha, o.damping_beta = damping_alpha, damping_beta
        o.relax_reference, o.max_steps = int(bool(relax_reference)), max_steps
        o.rho, o.beta1, o.beta2, o.dt, o.endtime = rho, beta1, beta2, dt, endtime
        o.wavelet_type, o.wavelet_freq, o.wavelet_timeshift, o.wavelet_ampl = (
            wavelet_type, freq, timeshift, ampl)
        o.precision, o.mass_convention, o.implicit_mode = precision, mass_convention, implicit_mode
        o.pcg_eps, o.steps_per_graph = pcg_eps, steps_per_graph
        return o

    def autotune_dyn(self, n_steps=0, rho=2400.0, beta1=0.5, beta2=0.0, dt=1e-3,
                     wavelet_type=WAVELET_NONE, freq=15.0, timeshift=0.0, ampl=1.0,
                     precision=FP64, mass_convention=MASS_REFERENCE,
                     implicit_mode=IMPLICIT_REFERENCE, pcg_eps=1e-4, steps_per_graph=64,
                     damping_alpha=0.0, damping_beta=0.0) -> dict:
        """femgpu_autotune_dyn: pick and apply the fastest patch tuning for
        the time stepper these options select (timed on n_steps steps)."""
        o = self._dyn_opts(self.lib, rho, beta1, beta2, dt, 0.0, wavelet_type, freq, timeshift,
                           ampl, precision, mass_convention, implicit_mode, pcg_eps,
                           steps_per_graph, damping_alpha, damping_beta, True, 1000000)
        e, t, us = C.c_int(0), C.c_int(0), C.c_double(0)
        self._check(self.lib.femgpu_autotune_dyn(self.h, C.byref(o), int(n_steps), C.byref(e),
                                                 C.byref(t), C.byref(us)), "autotune_dyn")
        return {"elems_per_patch": e.value, "patch_threads": t.value, "us_per_step": us.value}

    def dyn_run(self, rho=2400.0, beta1=0.5, beta2=0.0, dt=1e-3, endtime=0.1,
                wavelet_type=WAVELET_NONE, freq=15.0, timeshift=0.0, ampl=1.0,
                precision=FP64, mass_convention=MASS_REFERENCE,
                implicit_mode=IMPLICIT_REFERENCE, pcg_eps=1e-4, steps_per_graph=64,
                damping_alpha=0.0, damping_beta=0.0, relax_reference=True, max_steps=1000000,
                raise_on_error=True):
        o = self._dyn_opts(self.lib, rho, beta1, beta2, dt, endtime, wavelet_type, freq,
                           timeshift, ampl, precision, mass_convention, implicit_mode, pcg_eps,
                           steps_per_graph, damping_alpha, damping_beta, relax_reference,
                           max_steps)
        u = np.zeros((self.n_nodes, self.dim))
        s = DynStats()
        st = self.lib.femgpu_dyn_run(self.h, C.byref(o), _dp(u), C.byref(s))
        if raise_on_error:
            self._check(st, "dyn_run")
        return u, {"status": s.status, "steps": s.steps, "pcg_iterations": s.pcg_iterations,
                   "run_ms": s.run_ms}


def write_segy(path: str, traces: np.ndarray, sample_interval: float, trace_id: int = 0):
    """SEG-Y file of traces (n_traces, n_samples) (femgpu_write_segy)."""
    tr = np.ascontiguousarray(traces, dtype=np.float32)
    if tr.ndim != 2:
        raise ValueError("traces must be (n_traces, n_samples)")
    st = load_library().femgpu_write_segy(path.encode(), tr.ctypes.data_as(C.POINTER(C.c_float)),
                                          tr.shape[0], tr.shape[1], sample_interval, trace_id)
    if st != OK:
        raise FemGpuError(st, f"cannot write {path}")
