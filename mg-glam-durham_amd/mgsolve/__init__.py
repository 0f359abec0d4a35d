"""Python mirror of libmgsolve's C-ABI (include/mgsolve.h).

The product is the HIP library mgsolve/libmgsolve.so; this module only loads
it with ctypes and gives its entry points the names and argument meaning of
the reference's Fortran routines:

    Solver.initialise()              initialise_extradof   PMP2extradof.f90:181
    Solver.smooth(level, red)        relaxation_iterations_fR/_DGP
    Solver.residual(level)           calculate_residual_fR/_DGP
    Solver.restrict_residual(level)  restrict_residual_fR/_DGP
    Solver.restrict_field(level)     restrict_scalar_field
    Solver.restrict_density(level)   restrict_density
    Solver.rhs(level)                calculate_physical_right_hand_side_fR/_DGP
    Solver.correct(level)            correct_solution
    Solver.vcycle(level)             V_cycle
    Solver.fcycle(level)             F_cycle               PMP2extradof.f90:563
    Solver.wcycle(level)             W_cycle               PMP2extradof.f90:867
    Solver.solve(...)                scalar_field

There is no CPU fallback: if the library is missing, or no GPU is visible,
every call raises MgsError.
"""
from __future__ import annotations

import ctypes as C
import os
from dataclasses import dataclass

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libmgsolve.so")

MODEL_FR, MODEL_DGP = 1, 2
FLAG_REFERENCE_ROOTS = 1
PREC_FP64, PREC_MIXED = 0, 1
F32, F64 = 0, 1
HOST, DEVICE = 0, 1
EXIT_REL_TOL, EXIT_REFERENCE = 0, 1
ARR_U, ARR_RHO, ARR_F, ARR_RES, ARR_RRES, ARR_RU = range(6)
KC_SMOOTH, KC_RESIDUAL, KC_RESTRICT, KC_CORRECT, KC_COARSE, KC_UPDATE = range(6)
KC_NAMES = ["smooth", "residual", "restrict", "correct", "coarse", "update", "pm"]


class MgsError(RuntimeError):
    pass


class Params(C.Structure):
    _fields_ = [
        ("ngrid", C.c_int32), ("model", C.c_int32), ("fr_n", C.c_int32), ("branch", C.c_int32),
        ("box", C.c_double), ("omega_m", C.c_double), ("omega_l", C.c_double), ("aexpn", C.c_double),
        ("fr0", C.c_double), ("h0rc", C.c_double), ("precision", C.c_int32), ("flags", C.c_int32),
    ]


class SolveOpts(C.Structure):
    _fields_ = [
        ("mode", C.c_int32), ("max_cycles", C.c_int32), ("res_conv", C.c_double), ("rel_tol", C.c_double),
        ("init_guess", C.c_int32), ("inner_cycles", C.c_int32), ("cycle", C.c_int32), ("reserved", C.c_int32),
    ]


class SolveReport(C.Structure):
    _fields_ = [
        ("cycles", C.c_int32), ("outer", C.c_int32), ("converged", C.c_int32), ("reserved", C.c_int32),
        ("res0", C.c_double), ("res_final", C.c_double), ("seconds", C.c_double), ("history", C.c_double * 128),
    ]


class ServerOpts(C.Structure):
    _fields_ = [
        ("hbm_budget", C.c_uint64), ("max_active", C.c_int32), ("queue_capacity", C.c_int32),
        ("use_graphs", C.c_int32), ("reserved", C.c_int32),
    ]


class Request(C.Structure):
    _fields_ = [
        ("params", Params), ("delta", C.c_void_p), ("dtype", C.c_int32), ("max_outer", C.c_int32),
        ("rel_tol", C.c_double), ("exit_rule", C.c_int32), ("verify_fp64", C.c_int32), ("res_conv", C.c_double),
    ]


class RequestResult(C.Structure):
    _fields_ = [
        ("status", C.c_int32), ("outer", C.c_int32), ("converged", C.c_int32), ("verified", C.c_int32),
        ("res0", C.c_double), ("res_final", C.c_double), ("queued_ms", C.c_double), ("latency_ms", C.c_double),
        ("fp64_rel_linf", C.c_double), ("fp64_rel_l2", C.c_double), ("fp64_res_final", C.c_double),
    ]


class ServerStats(C.Structure):
    _fields_ = [
        ("submitted", C.c_int64), ("completed", C.c_int64), ("rejected", C.c_int64), ("steps", C.c_int64),
        ("p50_ms", C.c_double), ("p99_ms", C.c_double), ("mean_ms", C.c_double), ("solves_per_s", C.c_double),
        ("max_batch", C.c_int32), ("reserved", C.c_int32), ("step_ms", C.c_double), ("admit_ms", C.c_double),
        ("finish_ms", C.c_double), ("spilled", C.c_int64),
    ]


_lib = None


def load():
    """Load libmgsolve.so (raises MgsError when it is not built)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise MgsError(f"{LIB_PATH} is not built (make -C mg-glam-durham_amd); there is no CPU fallback")
    L = C.CDLL(LIB_PATH)
    H = C.c_void_p
    vp = C.c_void_p
    i32 = C.c_int32
    sig = {
        "mgs_create": ([C.POINTER(Params), C.POINTER(H)], C.c_int),
        "mgs_destroy": ([H], C.c_int),
        "mgs_last_error": ([H], C.c_char_p),
        "mgs_levels": ([H, C.POINTER(i32), C.POINTER(i32), C.POINTER(i32)], C.c_int),
        "mgs_set_params": ([H, C.POINTER(Params)], C.c_int),
        "mgs_set_density": ([H, vp, i32, i32], C.c_int),
        "mgs_get_density": ([H, vp, i32, i32], C.c_int),
        "mgs_set_field": ([H, vp, i32, i32], C.c_int),
        "mgs_get_field": ([H, vp, i32, i32, C.c_double], C.c_int),
        "mgs_set_level_array": ([H, i32, i32, vp, i32, i32], C.c_int),
        "mgs_get_level_array": ([H, i32, i32, vp, i32, i32], C.c_int),
        "mgs_background": ([H, C.POINTER(C.c_double), C.POINTER(C.c_double)], C.c_int),
        "mgs_initialise": ([H], C.c_int),
        "mgs_smooth": ([H, i32, i32], C.c_int),
        "mgs_residual": ([H, i32, C.POINTER(C.c_double)], C.c_int),
        "mgs_restrict_residual": ([H, i32], C.c_int),
        "mgs_restrict_field": ([H, i32], C.c_int),
        "mgs_restrict_density": ([H, i32], C.c_int),
        "mgs_rhs": ([H, i32], C.c_int),
        "mgs_correct": ([H, i32], C.c_int),
        "mgs_vcycle": ([H, i32], C.c_int),
        "mgs_fcycle": ([H, i32], C.c_int),
        "mgs_wcycle": ([H, i32], C.c_int),
        "mgs_solve": ([H, C.POINTER(SolveOpts), C.POINTER(SolveReport)], C.c_int),
        "mgs_fifth_force": ([H, vp, vp, vp, vp, i32, i32], C.c_int),
        "mgs_power_spectrum": ([H, i32, C.POINTER(C.c_double), C.POINTER(C.c_double), C.POINTER(C.c_double)], C.c_int),
        "mgs_power_spectrum_ex": ([H, i32, i32, i32] + [C.POINTER(C.c_double)] * 6, C.c_int),
        "mgs_make_lognormal_density": ([H, C.c_uint64, C.c_double, C.c_double, C.c_double], C.c_int),
        "mgs_particles_set": ([H, vp, vp, vp, vp, vp, vp, C.c_int64, i32], C.c_int),
        "mgs_particles_get": ([H, vp, vp, vp, vp, vp, vp, i32], C.c_int),
        "mgs_cic_deposit": ([H], C.c_int),
        "mgs_potential": ([H, C.c_double], C.c_int),
        "mgs_potential_add_fifth_force": ([H], C.c_int),
        "mgs_get_potential": ([H, vp, i32, i32], C.c_int),
        "mgs_set_potential": ([H, vp, i32, i32], C.c_int),
        "mgs_move": ([H, C.c_double, C.c_double, C.POINTER(C.c_double)], C.c_int),
        "mgs_profile": ([H, i32], C.c_int),
        "mgs_profile_get": ([H, i32, C.POINTER(C.c_int64), C.POINTER(C.c_double), C.POINTER(C.c_double)], C.c_int),
        "mgs_synchronize": ([H], C.c_int),
        "mgs_use_graphs": ([H, i32], C.c_int),
        "mgs_use_fused_levels": ([H, i32], C.c_int),
        "mgs_device_field": ([H, C.POINTER(C.c_void_p), C.POINTER(C.c_size_t)], C.c_int),
        "mgs_server_create": ([C.POINTER(ServerOpts), C.POINTER(H)], C.c_int),
        "mgs_server_destroy": ([H], C.c_int),
        "mgs_server_last_error": ([H], C.c_char_p),
        "mgs_server_submit": ([H, C.POINTER(Request), C.POINTER(C.c_int64)], C.c_int),
        "mgs_server_wait": ([H, C.c_int64, vp, C.c_size_t, i32, C.c_double, C.POINTER(RequestResult)], C.c_int),
        "mgs_server_get_stats": ([H, C.POINTER(ServerStats)], C.c_int),
        "mgs_server_test": ([H, C.c_int64, C.POINTER(i32)], C.c_int),
        "mgs_solve_noalloc": ([C.POINTER(Params), C.POINTER(SolveOpts), vp, i32, vp, i32, C.POINTER(SolveReport)],
                              C.c_int),
    }
    for name, (args, res) in sig.items():
        fn = getattr(L, name)
        fn.argtypes = args
        fn.restype = res
    _lib = L
    return L


def _np_ptr(a):
    return a.ctypes.data_as(C.c_void_p)


@dataclass
class Config:
    N: int
    model: int = MODEL_FR
    fr_n: int = 1
    branch: int = 1
    box: float = 256.0
    omega_m: float = 0.3
    omega_l: float = 0.7
    aexpn: float = 1.0
    fr0: float = -1.0e-5
    h0rc: float = 1.0
    precision: int = PREC_FP64
    flags: int = 0

    def c(self):
        return Params(self.N, self.model, self.fr_n, self.branch, self.box, self.omega_m, self.omega_l,
                      self.aexpn, self.fr0, self.h0rc, self.precision, self.flags)


class Solver:
    """One device-resident multigrid hierarchy (an mgs_handle)."""

    def __init__(self, cfg: Config):
        self.L = load()
        self.cfg = cfg
        self.h = C.c_void_p()
        p = cfg.c()
        rc = self.L.mgs_create(C.byref(p), C.byref(self.h))
        if rc != 0:
            raise MgsError(f"mgs_create failed ({rc}): {self.L.mgs_last_error(None).decode()}")
        self.N = cfg.N

    # ---- lifecycle -------------------------------------------------------
    def close(self):
        if self.h:
            self.L.mgs_destroy(self.h)
            self.h = C.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.close()

    def _chk(self, rc, what):
        if rc != 0:
            raise MgsError(f"{what} failed ({rc}): {self.L.mgs_last_error(self.h).decode()}")

    def levels(self):
        a, b, c = C.c_int32(), C.c_int32(), C.c_int32()
        self._chk(self.L.mgs_levels(self.h, C.byref(a), C.byref(b), C.byref(c)), "mgs_levels")
        return a.value, b.value, c.value

    def background(self):
        f, u = C.c_double(), C.c_double()
        self._chk(self.L.mgs_background(self.h, C.byref(f), C.byref(u)), "mgs_background")
        return f.value, u.value

    def set_params(self, cfg: Config):
        p = cfg.c()
        self._chk(self.L.mgs_set_params(self.h, C.byref(p)), "mgs_set_params")
        self.cfg = cfg

    # ---- data ------------------------------------------------------------
    @staticmethod
    def _dt(a):
        if a.dtype == np.float32:
            return F32
        if a.dtype == np.float64:
            return F64
        raise MgsError("arrays must be float32 or float64")

    def set_density(self, delta):
        a = np.ascontiguousarray(delta)
        if a.size != self.N ** 3:
            raise MgsError(f"density has {a.size} values for a grid of {self.N}^3")
        self._chk(self.L.mgs_set_density(self.h, _np_ptr(a), self._dt(a), HOST), "mgs_set_density")

    def get_density(self, dtype=np.float64):
        out = np.empty((self.N,) * 3, dtype)
        self._chk(self.L.mgs_get_density(self.h, _np_ptr(out), self._dt(out), HOST), "mgs_get_density")
        return out

    def set_field(self, u):
        a = np.ascontiguousarray(u)
        if a.size != self.N ** 3:
            raise MgsError(f"field has {a.size} values for a grid of {self.N}^3")
        self._chk(self.L.mgs_set_field(self.h, _np_ptr(a), self._dt(a), HOST), "mgs_set_field")

    def get_field(self, dtype=np.float64, scale=1.0):
        out = np.empty((self.N,) * 3, dtype)
        self._chk(self.L.mgs_get_field(self.h, _np_ptr(out), self._dt(out), HOST, scale), "mgs_get_field")
        return out

    def set_level(self, level, which, arr):
        a = np.ascontiguousarray(arr)
        n = self.N >> level
        if a.size != n ** 3:
            raise MgsError(f"level {level} holds {n}^3 values, not {a.size}")
        self._chk(self.L.mgs_set_level_array(self.h, level, which, _np_ptr(a), self._dt(a), HOST),
                  "mgs_set_level_array")

    def get_level(self, level, which, dtype=np.float64):
        n = self.N >> level
        out = np.empty((n, n, n), dtype)
        self._chk(self.L.mgs_get_level_array(self.h, level, which, _np_ptr(out), self._dt(out), HOST),
                  "mgs_get_level_array")
        return out

    # ---- operators (reference routine names) -----------------------------
    def initialise(self):
        self._chk(self.L.mgs_initialise(self.h), "mgs_initialise")

    def smooth(self, level, red):
        self._chk(self.L.mgs_smooth(self.h, level, int(bool(red))), "mgs_smooth")

    def residual(self, level):
        r = C.c_double()
        self._chk(self.L.mgs_residual(self.h, level, C.byref(r)), "mgs_residual")
        return r.value

    def restrict_residual(self, level):
        self._chk(self.L.mgs_restrict_residual(self.h, level), "mgs_restrict_residual")

    def restrict_field(self, level):
        self._chk(self.L.mgs_restrict_field(self.h, level), "mgs_restrict_field")

    def restrict_density(self, level):
        self._chk(self.L.mgs_restrict_density(self.h, level), "mgs_restrict_density")

    def rhs(self, level):
        self._chk(self.L.mgs_rhs(self.h, level), "mgs_rhs")

    def correct(self, level):
        self._chk(self.L.mgs_correct(self.h, level), "mgs_correct")

    def vcycle(self, level=0):
        self._chk(self.L.mgs_vcycle(self.h, level), "mgs_vcycle")

    def fcycle(self, level=0):
        self._chk(self.L.mgs_fcycle(self.h, level), "mgs_fcycle")

    def wcycle(self, level=0):
        self._chk(self.L.mgs_wcycle(self.h, level), "mgs_wcycle")

    def solve(self, mode=1, max_cycles=60, res_conv=1.0e-8, rel_tol=1.0e-8, init_guess=True, inner_cycles=0,
              cycle=0):
        """scalar_field: cycle 0 V_cycle, 1 F_cycle, 2 W_cycle.  Mixed precision: inner_cycles FP32 cycles of
        that kind per outer FP64 iteration, 0 = chosen per outer iteration (mode 1; 1 in mode 0)."""
        o = SolveOpts(mode, max_cycles, res_conv, rel_tol, 1 if init_guess else 0, inner_cycles, int(cycle), 0)
        r = SolveReport()
        self._chk(self.L.mgs_solve(self.h, C.byref(o), C.byref(r)), "mgs_solve")
        n = r.outer if self.cfg.precision == PREC_MIXED else r.cycles
        return dict(cycles=r.cycles, outer=r.outer, converged=bool(r.converged), res0=r.res0,
                    res_final=r.res_final, seconds=r.seconds, history=np.array(r.history[:min(n, 128)]))

    # ---- fifth force, spectra, synthetic input ---------------------------
    def fifth_force(self, dtype=np.float64):
        outs = [np.empty((self.N,) * 3, dtype) for _ in range(4)]
        self._chk(self.L.mgs_fifth_force(self.h, *[_np_ptr(a) for a in outs], self._dt(outs[0]), HOST),
                  "mgs_fifth_force")
        return tuple(outs)

    def power_spectrum(self, which=2):
        nb = self.N // 2
        k = np.zeros(nb)
        p = np.zeros(nb)
        c = np.zeros(nb)
        dp = C.POINTER(C.c_double)
        self._chk(self.L.mgs_power_spectrum(self.h, which, k.ctypes.data_as(dp), p.ctypes.data_as(dp),
                                            c.ctypes.data_as(dp)), "mgs_power_spectrum")
        return k, p, c

    def power_spectrum_ex(self, which=2, ipol=0, icic=0):
        """POWERfft5(ipol, .) with k-space binning icic: (k, P, count, klog,
        Plog, countlog), N/2 bins each (mgs_power_spectrum_ex)."""
        out = [np.zeros(self.N // 2) for _ in range(6)]
        dp = C.POINTER(C.c_double)
        self._chk(self.L.mgs_power_spectrum_ex(self.h, which, ipol, icic, *[a.ctypes.data_as(dp) for a in out]),
                  "mgs_power_spectrum_ex")
        return tuple(out)

    def make_lognormal_density(self, seed, sigma_g, slope=-1.5, kcut_frac=0.5):
        self._chk(self.L.mgs_make_lognormal_density(self.h, seed, sigma_g, slope, kcut_frac),
                  "mgs_make_lognormal_density")

    # ---- PM step: particles, deposit, potential, push ----------------------
    def set_particles(self, x, y, z, vx=None, vy=None, vz=None):
        """Positions in grid units in [1, N+1) (the reference's XPAR convention)."""
        arrs = [None if a is None else np.ascontiguousarray(a, dtype=np.float32) for a in (x, y, z, vx, vy, vz)]
        n = arrs[0].size
        if any(a is not None and a.size != n for a in arrs):
            raise MgsError("particle arrays differ in length")
        ptrs = [None if a is None else _np_ptr(a) for a in arrs]
        self._chk(self.L.mgs_particles_set(self.h, *ptrs, n, HOST), "mgs_particles_set")
        self._np = n

    def get_particles(self):
        outs = [np.empty(self._np, np.float32) for _ in range(6)]
        self._chk(self.L.mgs_particles_get(self.h, *[_np_ptr(a) for a in outs], HOST), "mgs_particles_get")
        return tuple(outs)

    def cic_deposit(self):
        self._chk(self.L.mgs_cic_deposit(self.h), "mgs_cic_deposit")

    def potential(self, trfi):
        self._chk(self.L.mgs_potential(self.h, trfi), "mgs_potential")

    def potential_add_fifth_force(self):
        self._chk(self.L.mgs_potential_add_fifth_force(self.h), "mgs_potential_add_fifth_force")

    def get_potential(self, dtype=np.float64):
        out = np.empty((self.N,) * 3, dtype)
        self._chk(self.L.mgs_get_potential(self.h, _np_ptr(out), self._dt(out), HOST), "mgs_get_potential")
        return out

    def set_potential(self, phi):
        a = np.ascontiguousarray(phi)
        if a.size != self.N ** 3:
            raise MgsError(f"potential has {a.size} values for a grid of {self.N}^3")
        self._chk(self.L.mgs_set_potential(self.h, _np_ptr(a), self._dt(a), HOST), "mgs_set_potential")

    def move(self, pconst, xconst):
        s = C.c_double()
        self._chk(self.L.mgs_move(self.h, pconst, xconst, C.byref(s)), "mgs_move")
        return s.value

    # ---- profiling ---------------------------------------------------------
    def profile(self, enable=True):
        self._chk(self.L.mgs_profile(self.h, int(bool(enable))), "mgs_profile")

    def profile_get(self, kclass):
        n, ms, b = C.c_int64(), C.c_double(), C.c_double()
        self._chk(self.L.mgs_profile_get(self.h, kclass, C.byref(n), C.byref(ms), C.byref(b)), "mgs_profile_get")
        return n.value, ms.value, b.value

    def synchronize(self):
        self._chk(self.L.mgs_synchronize(self.h), "mgs_synchronize")

    def use_graphs(self, enable=True):
        self._chk(self.L.mgs_use_graphs(self.h, int(bool(enable))), "mgs_use_graphs")

    def use_fused_levels(self, enable=True):
        """Small levels in one launch per cycle or half cycle, or one per operation (same results)."""
        self._chk(self.L.mgs_use_fused_levels(self.h, int(bool(enable))), "mgs_use_fused_levels")


def exported_symbols_declared_in_header(header_path):
    """Names of the functions include/mgsolve.h declares (for ABI tests)."""
    import re
    txt = open(header_path).read()
    return sorted(set(re.findall(r"^\s*(?:int|const char\*)\s+(mgs_\w+)\s*\(", txt, re.M)))


class Server:
    """Continuous-batching solve server (mgs_server_* in include/mgsolve.h):
    f(R) requests in mixed precision, admitted by HBM footprint into
    `max_active` slots and advanced together by batched launches."""

    def __init__(self, max_active=16, hbm_budget=0, queue_capacity=0, use_graphs=True):
        self.L = load()
        self.h = C.c_void_p()
        self._n = {}  # ticket -> ngrid of the submitted request
        o = ServerOpts(int(hbm_budget), int(max_active), int(queue_capacity), 1 if use_graphs else 0, 0)
        rc = self.L.mgs_server_create(C.byref(o), C.byref(self.h))
        if rc:
            raise MgsError(f"mgs_server_create failed ({rc}): {self.L.mgs_server_last_error(None).decode()}")

    def close(self):
        if self.h:
            self.L.mgs_server_destroy(self.h)
            self.h = C.c_void_p()

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.close()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def submit(self, cfg: Config, delta, rel_tol=1e-8, max_outer=60, exit_rule=None, res_conv=0.0,
               verify_fp64=False):
        """Queue a solve of cfg (f(R) or nDGP, PREC_MIXED) on density delta;
        returns a ticket.  exit_rule EXIT_REL_TOL (the default) stops as
        solve(mode=1, rel_tol=...), EXIT_REFERENCE as solve(mode=0,
        res_conv=...).  verify_fp64: wait() also solves the request with the
        plain FP64 method and reports the difference (fp64_rel_linf/_l2)."""
        a = np.ascontiguousarray(delta)
        if a.dtype not in (np.float32, np.float64):
            raise MgsError("delta must be float32 or float64")
        if a.size != cfg.N ** 3:
            raise MgsError(f"delta has {a.size} values for a grid of {cfg.N}^3")
        dt = F32 if a.dtype == np.float32 else F64
        rule = EXIT_REL_TOL if exit_rule is None else int(exit_rule)
        r = Request(cfg.c(), _np_ptr(a), dt, int(max_outer), float(rel_tol), rule, 1 if verify_fp64 else 0,
                    float(res_conv))
        t = C.c_int64()
        rc = self.L.mgs_server_submit(self.h, C.byref(r), C.byref(t))
        if rc:
            raise MgsError(f"mgs_server_submit failed ({rc}): {self.L.mgs_server_last_error(self.h).decode()}")
        self._n[t.value] = cfg.N
        return t.value

    def wait(self, ticket, N=None, dtype=np.float64, scale=1.0, out=None):
        """Block until the ticket is done; returns (field u, result dict).
        N, when given, must be the submitted grid's; dtype float32 or
        float64.  out: an (N, N, N) C-contiguous array of dtype to fill
        (reusing one avoids first-touch page faults on every result)."""
        n_sub = self._n.get(int(ticket))
        if N is None:
            N = n_sub
        if N is None:
            raise MgsError("unknown ticket: give N")
        if n_sub is not None and N != n_sub:
            raise MgsError(f"ticket {ticket} was submitted with N = {n_sub}, not {N}")
        dtype = np.dtype(dtype)
        if dtype not in (np.float32, np.float64):
            raise MgsError("dtype must be float32 or float64")
        if out is None:
            u = np.empty((N, N, N), dtype=dtype)
        else:
            if out.shape != (N, N, N) or out.dtype != dtype or not out.flags["C_CONTIGUOUS"]:
                raise MgsError("out must be a C-contiguous (N, N, N) array of the requested dtype")
            u = out
        res = RequestResult()
        rc = self.L.mgs_server_wait(self.h, int(ticket), _np_ptr(u), u.size, F32 if dtype == np.float32 else F64,
                                    float(scale), C.byref(res))
        self._n.pop(int(ticket), None)
        out = {k: getattr(res, k) for k, _ in RequestResult._fields_}
        if rc:
            raise MgsError(f"mgs_server_wait failed ({rc}): {self.L.mgs_server_last_error(self.h).decode()}")
        return u, out

    def test(self, ticket):
        """True when the ticket's request has finished (wait() will not block on a solve)."""
        d = C.c_int32(0)
        rc = self.L.mgs_server_test(self.h, int(ticket), C.byref(d))
        if rc:
            raise MgsError(f"mgs_server_test failed ({rc}): {self.L.mgs_server_last_error(self.h).decode()}")
        return bool(d.value)

    def stats(self):
        st = ServerStats()
        rc = self.L.mgs_server_get_stats(self.h, C.byref(st))
        if rc:
            raise MgsError(f"mgs_server_get_stats failed ({rc})")
        return {k: getattr(st, k) for k, _ in ServerStats._fields_}
