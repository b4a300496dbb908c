"""Python host mirror of the reference's Stokes-path functions over the C ABI.

The functions keep the reference's names, argument meaning and error
behaviour (``error(...)`` becomes ``M3Error``):

* ``assembly_stokes_sph_3d_double_jacobian`` (mfiles_SPH/...double_jacobian.m:1-2)
* ``restrict_stiffmat`` (mfiles_M3TET/restrict_stiffmat.m:1)
* ``cholesky_factorization`` / ``cholesky_solve`` (cholesky_*.m:1)
* ``mgpcg_solver_p`` (mfiles_M3TET/mgpcg_solver_p.m:1-2)
* ``flow3d_patera_sph`` (mfiles_M3TET/flow3d_patera_sph.m:1-9)

Matrices live on the GPU inside a :class:`StokesContext`; the functions that
return MATLAB sparse matrices in the reference return SciPy sparse matrices
gathered from the device.  Every compute call goes through ``libm3stokes.so``;
if the library is missing the import of this module fails.
"""
from __future__ import annotations

import ctypes as C
import os
import time

import numpy as np
import scipy.sparse as sp

from . import mesh as meshmod

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libm3stokes.so")
MAXL = 8


class M3Error(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"[m3 error {code}] {msg}")
        self.code = code


def _load():
    if not os.path.exists(LIB_PATH):
        raise ImportError(f"{LIB_PATH} is missing: build it with `python -m m3tet_sph_amd.build`")
    return C.CDLL(LIB_PATH)


LIB = _load()
D = C.POINTER(C.c_double)
I64 = C.POINTER(C.c_int64)
I32 = C.POINTER(C.c_int32)
U32 = C.POINTER(C.c_uint32)


class MeshDesc(C.Structure):
    _fields_ = [("nmg", C.c_int32), ("nel", C.c_int64 * MAXL), ("nnod", C.c_int64 * MAXL),
                ("nVnod", C.c_int64 * MAXL), ("EL2NOD", U32 * MAXL), ("GCOORD", D),
                ("GCOORD_SPH", D), ("els_class", I32 * 4), ("nels_class", C.c_int64 * 4),
                ("EL2NOD_cubic", U32), ("GCOORD_cubic", D), ("ncubic", C.c_int64),
                ("Ic2f_ptr", I64 * MAXL), ("Ic2f_col", I32 * MAXL), ("Ic2f_val", D * MAXL)]


class Phys(C.Structure):
    _fields_ = [("g", C.c_double), ("Bscale", C.c_double), ("Dens0", C.c_double),
                ("minVisc", C.c_double), ("maxVisc", C.c_double), ("has_minVisc", C.c_int32),
                ("has_maxVisc", C.c_int32), ("nip", C.c_int32), ("type_Dmat", C.c_int32)]


class PateraOpts(C.Structure):
    _fields_ = [("rtol_Pat", C.c_double), ("rtol_U", C.c_double), ("itmax_U", C.c_int32),
                ("itmin_Pat", C.c_int32), ("itmax_Pat", C.c_int32), ("pc_Pat", C.c_int32),
                ("wght_MM", C.c_double), ("precision", C.c_int32), ("warm_U", C.c_int32),
                ("rtol_U_final", C.c_double), ("itmax_U_final", C.c_int32), ("tol_Pat_abs", C.c_double),
                ("rtol_U_first", C.c_double)]


class Info(C.Structure):
    _fields_ = [("nitP", C.c_int32), ("nitU", C.c_int32), ("nitZ", C.c_int32),
                ("norm_rP", C.c_double), ("norm_rP0", C.c_double), ("t_assemble", C.c_double),
                ("t_restrict", C.c_double), ("t_factor", C.c_double), ("t_pressure", C.c_double),
                ("t_velocity", C.c_double), ("t_total", C.c_double)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


PREC = {"fp64": 0, "mixed": 1}

LIB.m3_create.argtypes = [C.POINTER(C.c_void_p), C.c_int]
LIB.m3_destroy.argtypes = [C.c_void_p]
LIB.m3_last_error.argtypes = [C.c_void_p]
LIB.m3_last_error.restype = C.c_char_p
LIB.m3_set_mesh.argtypes = [C.c_void_p, C.POINTER(MeshDesc)]
LIB.m3_set_bc.argtypes = [C.c_void_p, I64, D, C.c_int64]
LIB.m3_assemble.argtypes = [C.c_void_p, D, D, C.POINTER(Phys)]
LIB.m3_element_matrices.argtypes = [C.c_void_p, D, D, C.POINTER(Phys), D, D, D, D]
LIB.m3_restrict_stiffmat.argtypes = [C.c_void_p]
LIB.m3_cholesky_factorization.argtypes = [C.c_void_p]
LIB.m3_cholesky_solve.argtypes = [C.c_void_p, D, D]
LIB.m3_mgpcg.argtypes = [C.c_void_p, D, D, C.c_double, C.c_int32, C.c_int32, C.c_int32, I32, D]
LIB.m3_patera.argtypes = [C.c_void_p, D, D, C.POINTER(PateraOpts), C.POINTER(Info)]
LIB.m3_flow3d_patera_sph.argtypes = [C.c_void_p, D, D, C.POINTER(Phys), D, D,
                                     C.POINTER(PateraOpts), C.POINTER(Info)]
LIB.m3_flow3d_patera_sph_dstart.argtypes = [C.c_void_p, D, D, C.POINTER(Phys), C.c_void_p, C.c_void_p, D, D,
                                            C.POINTER(PateraOpts), C.POINTER(Info)]
LIB.m3_solution_device.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.POINTER(C.c_void_p)]
LIB.m3_get_solution.argtypes = [C.c_void_p, D, D]
LIB.m3_set_fields.argtypes = [C.c_void_p, D, D]
LIB.m3_apply.argtypes = [C.c_void_p, C.c_int32, C.c_int32, D, D]
LIB.m3_get_vector.argtypes = [C.c_void_p, C.c_int32, C.c_int32, D]
LIB.m3_stats.argtypes = [C.c_void_p, I64, C.c_int32]
LIB.m3_sweep_windows.argtypes = [C.c_void_p, C.c_int64, C.c_int32, C.c_int32, C.c_int32]
LIB.m3_sl_advect.argtypes = [C.c_void_p, D, D, C.c_double, C.c_double, C.c_double, D]


class SlmOpts(C.Structure):
    _fields_ = [("method_BT", C.c_int32), ("method_interp", C.c_int32), ("monotonic", C.c_int32)]


class SlmInfo(C.Structure):
    _fields_ = [("nshift", C.c_int64), ("nunresolved", C.c_int64)]


SLM_METHOD_BT = {"EU1": 1, "PC2": 2, "RK4": 3}
SLM_METHOD_INTERP = {"linear": 1, "quadratic": 2, "cubic": 3}
LIB.m3_advect3d_slm_p_sph.argtypes = [C.c_void_p, D, D, D, D, C.c_double, C.POINTER(SlmOpts), C.POINTER(SlmInfo)]
LIB.m3_advect3d_slm_p_sph.restype = C.c_int


class RockParams(C.Structure):
    """PHYSICS fields read by rock_prop.m:31-118 (m3_rock_params)."""
    _fields_ = [(k, C.c_double) for k in ("Visc0", "Dens0", "T_ref", "alpha", "Ea", "Va", "g", "L0", "a_UM2LM",
                                          "minVisc", "maxVisc", "minDens", "maxDens")] + \
               [(k, C.c_int32) for k in ("has_minVisc", "has_maxVisc", "has_minDens", "has_maxDens")]


def rock_params(Visc0=1.0, Dens0=1.0, T_ref=0.0, alpha=0.0, Ea=0.0, Va=0.0, g=-1.0, L0=1.0, a_UM2LM=0.0,
                minVisc=None, maxVisc=None, minDens=None, maxDens=None):
    p = RockParams()
    for k, v in dict(Visc0=Visc0, Dens0=Dens0, T_ref=T_ref, alpha=alpha, Ea=Ea, Va=Va, g=g, L0=L0,
                     a_UM2LM=a_UM2LM).items():
        setattr(p, k, v)
    for k, v in dict(minVisc=minVisc, maxVisc=maxVisc, minDens=minDens, maxDens=maxDens).items():
        setattr(p, k, 0.0 if v is None else v)
        setattr(p, "has_" + k, int(v is not None))
    return p


class DiffusionOpts(C.Structure):
    """SETTINGS.OPTS_D (default_numerics_M3TET.m:95-134), m3_diffusion_opts."""
    _fields_ = [("theta", C.c_double), ("lumping", C.c_int32), ("nip", C.c_int32), ("tol", C.c_double),
                ("is_abs_tol", C.c_int32), ("itmax", C.c_int32)]


class DiffusionInfo(C.Structure):
    _fields_ = [("nit", C.c_int32), ("norm_r0", C.c_double), ("norm_r", C.c_double), ("tol", C.c_double),
                ("t_assemble", C.c_double), ("t_solve", C.c_double)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


def diffusion_opts(theta=1.0, lumping="yes", nip=4, tol=1e-8, is_abs_tol=0, itmax=500):
    """Defaults of default_numerics_M3TET.m:95-134 (eltype 'linear', pc 'diag')."""
    o = DiffusionOpts()
    o.theta, o.nip, o.tol, o.is_abs_tol, o.itmax = theta, nip, tol, int(is_abs_tol), itmax
    o.lumping = int(lumping in ("yes", True, 1))
    return o


LIB.m3_diffusion_mesh.argtypes = [C.c_void_p, U32, C.c_int64, C.c_int64, C.c_double]
LIB.m3_diffusion3d.argtypes = [C.c_void_p, D, C.c_double, C.c_double, I64, D, C.c_int64,
                               C.POINTER(DiffusionOpts), C.POINTER(DiffusionInfo)]
LIB.m3_diffusion_apply.argtypes = [C.c_void_p, C.c_int32, D, D]
for _f in ("m3_diffusion_mesh", "m3_diffusion3d", "m3_diffusion_apply"):
    getattr(LIB, _f).restype = C.c_int

LIB.m3_set_els_ref.argtypes = [C.c_void_p, I32, C.c_int64, D]
LIB.m3_set_els_ref.restype = C.c_int
LIB.m3_unique_bars.argtypes = [C.c_int32, I32, C.c_int64, I64, I64, I64]
LIB.m3_unique_bars.restype = C.c_int
# device buffers (bars, first, bar_of), host nu, hipStream_t
LIB.m3_unique_bars_noalloc.argtypes = [C.c_int32, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, I64, C.c_void_p]
LIB.m3_unique_bars_noalloc.restype = C.c_int


def unique_bars(bars, device=0):
    """find_unique_bars (tetmesh_p1_to_p2_sph.m:238-254) on the GPU: (first,
    bar_of) with first[u] the position of unique bar u's first occurrence (in
    order of appearance) and bar_of[i] the unique index of bar i."""
    b = np.ascontiguousarray(bars, dtype=np.int32)
    if b.ndim != 2 or b.shape[1] != 2:
        raise M3Error(1, "expecting a nx2 matrix")
    n = len(b)
    first = np.empty(max(n, 1), dtype=np.int64)
    bar_of = np.empty(max(n, 1), dtype=np.int64)
    nu = C.c_int64(0)
    rc = LIB.m3_unique_bars(int(device), _p(b, I32), n, _p(first, I64), _p(bar_of, I64), C.byref(nu))
    if rc:
        raise M3Error(rc, "m3_unique_bars failed")
    return first[:nu.value].copy(), bar_of[:n].copy()


LIB.m3_hier_build.argtypes = [C.POINTER(C.c_void_p), C.c_int32, D, I32, I32, C.c_int64, C.c_int64, C.c_double,
                              C.c_double, C.c_int32, C.c_double]
LIB.m3_hier_level.argtypes = [C.c_void_p, C.c_int32, I64, I64, I64, I64, C.POINTER(C.c_int8)]
LIB.m3_hier_nodes.argtypes = [C.c_void_p, D, D, I32, C.POINTER(C.c_int8)]
LIB.m3_hier_iso.argtypes = [C.c_void_p, I64, I64, D]
LIB.m3_hier_transfer.argtypes = [C.c_void_p, C.c_int32, I64, I64, I64, D]
LIB.m3_hier_time.argtypes = [C.c_void_p, D]
LIB.m3_hier_destroy.argtypes = [C.c_void_p]
LIB.m3_hier_destroy.restype = None
LIB.m3_detmath_eval.argtypes = [C.c_int32, C.c_int32, C.c_int64, D, D, D]
for _f in ("m3_hier_build", "m3_hier_level", "m3_hier_nodes", "m3_hier_iso", "m3_hier_transfer", "m3_hier_time",
           "m3_detmath_eval"):
    getattr(LIB, _f).restype = C.c_int

DETMATH_OPS = {"sin": 0, "cos": 1, "atan2": 2, "sqrt": 3, "cart2sph": 4, "sph2cart": 5}


def detmath_eval(op, x, y=None, device=0):
    """The set-up's reproducible sin / cos / atan2(y, x) / sqrt /
    cartesian2spherical / spherical2cartesian evaluated on the GPU."""
    code = DETMATH_OPS[op]
    x = np.ascontiguousarray(x, dtype=np.float64)
    n = len(x)
    out = np.empty_like(x)
    yy = np.ascontiguousarray(y, dtype=np.float64) if y is not None else None
    rc = LIB.m3_detmath_eval(int(device), code, n, _p(x, D), None if yy is None else _p(yy, D), _p(out, D))
    if rc:
        raise M3Error(rc, LIB.m3_last_error(None).decode())
    return out


def hier_build(X4, EL4, pid4, r_cmb, r_surf, nmg, theta_cone, device=0):
    """The multigrid hierarchy built on the GPU (m3_hier_build: curved P2
    promotion of tetmesh_p1_to_p2_sph.m, 8-way refinement of
    tetmesh_refine_sph.m / tetmesh_p2_to_p1.m, the 20-node geometry of
    cubic_els_in_cone_iso.m and the transfer operators of
    intermesh_transfer_matrix.m) from the coarsest vertex mesh (0-based EL4).
    Returns a dict of host arrays: levels (finest first: EL2NOD, nnod, nVnod),
    isplit[l] (split types of level l+1), GCOORD, GCOORD_SPH, PointID, cls
    (finest element classes 0..3), iso, X20_iso, transfers[l] (CSR from level
    l+1 to level l) and gpu_ms."""
    X4 = np.ascontiguousarray(X4, dtype=np.float64)
    EL4 = np.ascontiguousarray(EL4, dtype=np.int32)
    pid4 = np.ascontiguousarray(pid4, dtype=np.int32)
    h = C.c_void_p()

    def check(rc, what):
        if rc:
            raise M3Error(rc, f"{what}: {LIB.m3_last_error(None).decode()}")

    check(LIB.m3_hier_build(C.byref(h), int(device), _p(X4, D), _p(EL4, I32), _p(pid4, I32), len(X4), len(EL4),
                            float(r_cmb), float(r_surf), int(nmg), float(theta_cone)), "m3_hier_build")
    try:
        out = dict(levels=[], isplit=[], transfers=[])
        for l in range(nmg):
            nel, nnod, nv = C.c_int64(), C.c_int64(), C.c_int64()
            check(LIB.m3_hier_level(h, l, C.byref(nel), C.byref(nnod), C.byref(nv), None, None), "m3_hier_level")
            EL = np.empty((nel.value, 10), dtype=np.int64)
            sp = np.empty(nel.value, dtype=np.int8) if l > 0 else None
            check(LIB.m3_hier_level(h, l, None, None, None, _p(EL, I64),
                                    None if sp is None else sp.ctypes.data_as(C.POINTER(C.c_int8))), "m3_hier_level")
            out["levels"].append((EL, nnod.value, nv.value))
            if sp is not None:
                out["isplit"].append(sp.astype(np.int64))
        nnod, nel = out["levels"][0][1], len(out["levels"][0][0])
        X, S = np.empty((nnod, 3)), np.empty((nnod, 3))
        pid = np.empty(nnod, dtype=np.int32)
        cls = np.empty(nel, dtype=np.int8)
        check(LIB.m3_hier_nodes(h, _p(X, D), _p(S, D), _p(pid, I32), cls.ctypes.data_as(C.POINTER(C.c_int8))),
              "m3_hier_nodes")
        niso = C.c_int64()
        check(LIB.m3_hier_iso(h, C.byref(niso), None, None), "m3_hier_iso")
        iso = np.empty(niso.value, dtype=np.int64)
        X20 = np.empty((niso.value, 20, 3))
        check(LIB.m3_hier_iso(h, C.byref(niso), _p(iso, I64), _p(X20, D)), "m3_hier_iso")
        for l in range(nmg - 1):
            nnz = C.c_int64()
            check(LIB.m3_hier_transfer(h, l, C.byref(nnz), None, None, None), "m3_hier_transfer")
            ptr = np.empty(out["levels"][l][1] + 1, dtype=np.int64)
            idx = np.empty(nnz.value, dtype=np.int64)
            w = np.empty(nnz.value)
            check(LIB.m3_hier_transfer(h, l, C.byref(nnz), _p(ptr, I64), _p(idx, I64), _p(w, D)),
                  "m3_hier_transfer")
            out["transfers"].append((ptr, idx, w))
        ms = C.c_double()
        check(LIB.m3_hier_time(h, C.byref(ms)), "m3_hier_time")
        out.update(GCOORD=X, GCOORD_SPH=S, PointID=pid, cls=cls, iso=iso, X20_iso=X20, gpu_ms=ms.value)
        return out
    finally:
        LIB.m3_hier_destroy(h)


LIB.m3_rock_prop.argtypes = [C.c_void_p, D, C.POINTER(RockParams), D, D]
LIB.m3_calculate_dt.argtypes = [C.c_void_p, D, C.c_double, C.c_double, D]
LIB.m3_rock_prop.restype = C.c_int
LIB.m3_calculate_dt.restype = C.c_int
for _f in ("m3_create", "m3_set_mesh", "m3_set_bc", "m3_assemble", "m3_element_matrices",
           "m3_restrict_stiffmat", "m3_cholesky_factorization", "m3_cholesky_solve", "m3_mgpcg",
           "m3_patera", "m3_flow3d_patera_sph", "m3_flow3d_patera_sph_dstart", "m3_apply", "m3_get_vector",
           "m3_stats", "m3_sweep_windows", "m3_sl_advect", "m3_solution_device", "m3_get_solution", "m3_set_fields"):
    getattr(LIB, _f).restype = C.c_int


def _p(a, t=D):
    return a.ctypes.data_as(t)


def _fields(Visc, Dens):
    """Host pointers of the nodal fields, or NULL for the device-resident ones."""
    if Visc is None and Dens is None:
        return None, None
    V = np.ascontiguousarray(Visc, dtype=np.float64)
    R = np.ascontiguousarray(Dens, dtype=np.float64)
    _fields.keep = (V, R)
    return _p(V), _p(R)


def phys_struct(phys, nip=14, type_Dmat="23rd"):
    p = Phys()
    p.g, p.Bscale, p.Dens0 = phys["g"], phys["Bscale"], phys["Dens0"]
    p.has_minVisc = int(phys.get("minVisc") is not None)
    p.has_maxVisc = int(phys.get("maxVisc") is not None)
    p.minVisc = phys.get("minVisc") or 0.0
    p.maxVisc = phys.get("maxVisc") or 0.0
    p.nip = nip
    p.type_Dmat = {"23rd": 0, "221": 1}[type_Dmat]
    return p


def patera_opts(rtol_Pat=1e-4, rtol_U=5e-3, itmax_U=20, itmin_Pat=3, itmax_Pat=120,
                wght_MM=1.0, precision="fp64", warm_U=False, rtol_U_final=0.0, itmax_U_final=60,
                tol_Pat_abs=0.0, rtol_U_first=0.0):
    """Defaults of flow3d_patera_mg_sph_p.m:70-98 (rtol_U_final=0 keeps the
    reference's final velocity tolerance, tol_Pat_abs=0 its relative
    pressure tolerance, rtol_U_first=0 its relative initial velocity
    tolerance)."""
    o = PateraOpts()
    o.rtol_Pat, o.rtol_U, o.itmax_U = rtol_Pat, rtol_U, itmax_U
    o.itmin_Pat, o.itmax_Pat, o.pc_Pat, o.wght_MM = itmin_Pat, itmax_Pat, 3, wght_MM
    o.precision = PREC[precision]
    o.warm_U = int(warm_U)
    o.rtol_U_final, o.itmax_U_final = rtol_U_final, itmax_U_final
    o.tol_Pat_abs = tol_Pat_abs
    o.rtol_U_first = rtol_U_first
    return o


def mesh_arrays(m):
    """The arrays of m3_mesh_desc for a ShellMesh, in the reference's layout
    (1-based indices, EL2NOD as nel rows of 10, Ic2f as node-level CSR)."""
    out = {}
    for l, L in enumerate(m.levels):
        out[f"EL2NOD_{l}"] = np.ascontiguousarray(L.EL2NOD + 1, dtype=np.uint32)
    out["GCOORD"] = np.ascontiguousarray(m.GCOORD, dtype=np.float64)
    out["GCOORD_SPH"] = np.ascontiguousarray(m.GCOORD_SPH, dtype=np.float64)
    names = ("out_cone_no_cross_2pi", "out_cone_cross_2pi", "in_cone_no_iso", "in_cone_iso")
    for k, nm in enumerate(names):
        out[f"class_{k}"] = np.ascontiguousarray(m.classes[nm] + 1, dtype=np.int32)
    iso = m.classes["in_cone_iso"]
    n_iso = len(iso)
    E20 = np.zeros((max(n_iso, 1), 20), dtype=np.uint32)
    Xc = np.zeros((max(n_iso * 16, 1), 3))
    if n_iso:
        E20[:, :4] = m.levels[0].EL2NOD[iso, :4] + 1
        E20[:, 4:] = m.nnod + 1 + np.arange(n_iso * 16).reshape(n_iso, 16)
        Xc = np.ascontiguousarray(m.X20_iso[:, 4:, :].reshape(-1, 3))
    out["EL2NOD_cubic"], out["GCOORD_cubic"], out["ncubic"] = E20, Xc, n_iso * 16
    for l in range(m.nmg - 1):
        ip, ci, w = m.transfer(l)
        out[f"Ic2f_ptr_{l}"] = np.ascontiguousarray(ip, dtype=np.int64)
        out[f"Ic2f_col_{l}"] = np.ascontiguousarray(ci, dtype=np.int32)
        out[f"Ic2f_val_{l}"] = np.ascontiguousarray(w, dtype=np.float64)
    return out


def export_case(path, m, inputs):
    """Write a solve case for the C++ harness ``m3bench``: the m3_mesh_desc
    arrays, UBC.ifix / UBC.vfix (1-based), nodal Visc / Dens as .npy files and
    the sizes and PHYSICS / NUMSCALE scalars in case.txt ("key value" lines)."""
    os.makedirs(path, exist_ok=True)
    arrs = mesh_arrays(m)
    for k, v in arrs.items():
        if isinstance(v, np.ndarray):
            np.save(os.path.join(path, k + ".npy"), v)
    np.save(os.path.join(path, "ifix.npy"), np.ascontiguousarray(np.asarray(inputs["ifix"]) + 1, dtype=np.int64))
    np.save(os.path.join(path, "vfix.npy"), np.ascontiguousarray(inputs["vfix"], dtype=np.float64))
    np.save(os.path.join(path, "Visc.npy"), np.ascontiguousarray(inputs["Visc"], dtype=np.float64))
    np.save(os.path.join(path, "Dens.npy"), np.ascontiguousarray(inputs["Dens"], dtype=np.float64))
    ph = inputs["phys"]
    lines = [f"nmg {m.nmg}", f"ncubic {arrs['ncubic']}"]
    for l, L in enumerate(m.levels):
        lines += [f"nel_{l} {len(L.EL2NOD)}", f"nnod_{l} {L.nnod}", f"nVnod_{l} {L.nVnod}"]
    lines += [f"g {ph['g']!r}", f"Bscale {ph['Bscale']!r}", f"Dens0 {ph['Dens0']!r}"]
    for k in ("minVisc", "maxVisc"):
        if ph.get(k) is not None:
            lines.append(f"{k} {ph[k]!r}")
    with open(os.path.join(path, "case.txt"), "w") as f:
        f.write("\n".join(lines) + "\n")


class StokesContext:
    """Device state of one mesh (patterns, operators, hierarchy, factor)."""

    def __init__(self, mesh: meshmod.ShellMesh, device=0, sweep_windows=None):
        """sweep_windows: (rows, split, limit, per_row) of m3_sweep_windows."""
        self._h = C.c_void_p()
        rc = LIB.m3_create(C.byref(self._h), device)
        if rc:
            msg = LIB.m3_last_error(self._h).decode() if self._h else "m3_create failed"
            if self._h:
                LIB.m3_destroy(self._h)
            self._h = None
            raise M3Error(rc, msg)
        self.mesh = mesh
        self._keep = []
        if sweep_windows is not None:
            self._check(LIB.m3_sweep_windows(self._h, *sweep_windows))
        self._set_mesh(mesh)

    def close(self):
        if self._h:
            LIB.m3_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _check(self, rc):
        if rc:
            raise M3Error(rc, LIB.m3_last_error(self._h).decode())

    def _set_mesh(self, m):
        arrs = mesh_arrays(m)
        d = MeshDesc()
        d.nmg = m.nmg
        for l, L in enumerate(m.levels):
            d.nel[l], d.nnod[l], d.nVnod[l] = len(L.EL2NOD), L.nnod, L.nVnod
            d.EL2NOD[l] = _p(arrs[f"EL2NOD_{l}"], U32)
        d.GCOORD, d.GCOORD_SPH = _p(arrs["GCOORD"]), _p(arrs["GCOORD_SPH"])
        for k in range(4):
            d.els_class[k] = _p(arrs[f"class_{k}"], I32)
            d.nels_class[k] = len(arrs[f"class_{k}"])
        d.EL2NOD_cubic, d.GCOORD_cubic = _p(arrs["EL2NOD_cubic"], U32), _p(arrs["GCOORD_cubic"])
        d.ncubic = int(arrs["ncubic"])
        for l in range(m.nmg - 1):
            d.Ic2f_ptr[l] = _p(arrs[f"Ic2f_ptr_{l}"], I64)
            d.Ic2f_col[l] = _p(arrs[f"Ic2f_col_{l}"], I32)
            d.Ic2f_val[l] = _p(arrs[f"Ic2f_val_{l}"])
        self._check(LIB.m3_set_mesh(self._h, C.byref(d)))

    # ---- operations ------------------------------------------------------------
    def set_bc(self, ifix0, vfix):
        """UBC.ifix (0-based here, converted to 1-based) and UBC.vfix."""
        i = np.ascontiguousarray(np.asarray(ifix0, dtype=np.int64) + 1)
        v = np.ascontiguousarray(vfix, dtype=np.float64)
        self._check(LIB.m3_set_bc(self._h, _p(i, I64), _p(v), len(i)))
        self.ifix, self.vfix = np.asarray(ifix0), v

    def set_els_ref(self, els_ref0, Dens0_T_bary):
        """MESH.els_ref (0-based here, converted to 1-based) and
        NUMSCALE.Dens0_T_bary: buoyancy only inside the embedded refined
        region, relative to each element's reference density; an empty
        els_ref0 restores the uniform NUMSCALE.Dens0."""
        e = np.ascontiguousarray(np.asarray(els_ref0, dtype=np.int64) + 1, dtype=np.int32)
        d = np.ascontiguousarray(Dens0_T_bary if len(e) else np.zeros(0), dtype=np.float64)
        if len(d) != len(e):
            raise M3Error(1, "els_ref and Dens0_T_bary differ in length")
        self._check(LIB.m3_set_els_ref(self._h, _p(e, I32), len(e), _p(d)))

    def assemble(self, Visc, Dens, phys, type_Dmat="23rd"):
        """Visc = Dens = None: use the fields left on the device by rock_prop."""
        V, R = _fields(Visc, Dens)
        self._check(LIB.m3_assemble(self._h, V, R, C.byref(phys_struct(phys, type_Dmat=type_Dmat))))

    def element_matrices(self, Visc, Dens, phys, type_Dmat="23rd"):
        nel = self.mesh.nel
        K = np.zeros((nel, 465))
        G = np.zeros((nel, 120))
        M = np.zeros((nel, 10))
        F = np.zeros((nel, 30))
        V = np.ascontiguousarray(Visc, dtype=np.float64)
        R = np.ascontiguousarray(Dens, dtype=np.float64)
        self._check(LIB.m3_element_matrices(self._h, _p(V), _p(R),
                                            C.byref(phys_struct(phys, type_Dmat=type_Dmat)),
                                            _p(K), _p(G), _p(M), _p(F)))
        return K, G, M, F

    def restrict_stiffmat(self):
        self._check(LIB.m3_restrict_stiffmat(self._h))

    def cholesky_factorization(self):
        self._check(LIB.m3_cholesky_factorization(self._h))

    def cholesky_solve(self, rhs):
        rhs = np.ascontiguousarray(rhs, dtype=np.float64)
        x = np.zeros_like(rhs)
        self._check(LIB.m3_cholesky_solve(self._h, _p(rhs), _p(x)))
        return x

    def mgpcg(self, b, x=None, tol=1e-8, is_abs_tol=True, itmax=50, precision="fp64"):
        b = np.ascontiguousarray(b, dtype=np.float64)
        x = np.zeros_like(b) if x is None else np.ascontiguousarray(x, dtype=np.float64).copy()
        it = C.c_int32(0)
        hist = np.zeros(itmax + 1)
        self._check(LIB.m3_mgpcg(self._h, _p(b), _p(x), tol, int(is_abs_tol), itmax, PREC[precision],
                                 C.byref(it), _p(hist)))
        return x, it.value, hist[:it.value + 1]

    def patera(self, P0=None, U0=None, **opts):
        n3 = 3 * self.mesh.nnod
        U = np.zeros(n3) if U0 is None else np.ascontiguousarray(U0, dtype=np.float64).copy()
        P = np.zeros(self.mesh.nVnod) if P0 is None else np.ascontiguousarray(P0, dtype=np.float64).copy()
        info = Info()
        o = patera_opts(warm_U=U0 is not None, **opts)
        self._check(LIB.m3_patera(self._h, _p(U), _p(P), C.byref(o), C.byref(info)))
        return U, P, info.as_dict()

    def flow3d(self, Visc, Dens, phys, P0=None, U0=None, type_Dmat="23rd", start_device=None,
               keep_on_device=False, **opts):
        """start_device=(U0_dev, P0_dev): device addresses of the starting point
        (WarmStartNet.start_device()), used instead of U0 / P0.  Visc = Dens =
        None: the fields on the device (set_fields, rock_prop).  With
        start_device and keep_on_device=True the solution stays on the device
        (solution(), solution_device()) and (None, None, info) is returned."""
        n3 = 3 * self.mesh.nnod
        V, R = _fields(Visc, Dens)
        info = Info()
        ph = C.byref(phys_struct(phys, type_Dmat=type_Dmat))
        if start_device is not None:
            U, P = (None, None) if keep_on_device else (np.empty(n3), np.empty(self.mesh.nVnod))
            o = patera_opts(warm_U=True, **opts)
            self._check(LIB.m3_flow3d_patera_sph_dstart(self._h, V, R, ph, C.c_void_p(start_device[0]),
                                                        C.c_void_p(start_device[1]),
                                                        None if U is None else _p(U), None if P is None else _p(P),
                                                        C.byref(o), C.byref(info)))
            return U, P, info.as_dict()
        if keep_on_device:
            raise ValueError("keep_on_device needs start_device")
        U = np.zeros(n3) if U0 is None else np.ascontiguousarray(U0, dtype=np.float64).copy()
        P = np.zeros(self.mesh.nVnod) if P0 is None else np.ascontiguousarray(P0, dtype=np.float64).copy()
        o = patera_opts(warm_U=U0 is not None, **opts)
        self._check(LIB.m3_flow3d_patera_sph(self._h, V, R, ph, _p(U), _p(P), C.byref(o), C.byref(info)))
        return U, P, info.as_dict()

    def set_fields(self, Visc, Dens):
        """Nodal Visc, Dens to the device fields (flow3d with Visc = Dens = None)."""
        V, R = _fields(Visc, Dens)
        self._check(LIB.m3_set_fields(self._h, V, R))

    def solution(self):
        """Host copy (U, P) of the last solve's solution, kept on the device."""
        U, P = np.empty(3 * self.mesh.nnod), np.empty(self.mesh.nVnod)
        self._check(LIB.m3_get_solution(self._h, _p(U), _p(P)))
        return U, P

    def solution_device(self):
        """Device addresses (U, P) of the last solve's solution."""
        u, p = C.c_void_p(), C.c_void_p()
        self._check(LIB.m3_solution_device(self._h, C.byref(u), C.byref(p)))
        return u.value, p.value

    def rock_prop(self, T, params, download=True):
        """VAR = rock_prop(VAR,...) (rock_prop.m:31-118) on the device: nodal
        viscosity and density from the nodal temperature.  The fields stay on
        the device for the next ``assemble``/``flow3d`` called with
        Visc = Dens = None; returned to the host if ``download``."""
        T = np.ascontiguousarray(T, dtype=np.float64)
        V = np.zeros_like(T) if download else None
        R = np.zeros_like(T) if download else None
        self._check(LIB.m3_rock_prop(self._h, _p(T), C.byref(params), _p(V) if download else None,
                                     _p(R) if download else None))
        return V, R

    def calculate_dt(self, U, dt_adv_limit=0.5, dtmax=np.inf):
        """dt = calculate_dt(...) (calculate_dt.m:40-56) from the rotated-frame U."""
        U = np.ascontiguousarray(U, dtype=np.float64)
        dt = C.c_double(0.0)
        self._check(LIB.m3_calculate_dt(self._h, _p(U), float(dt_adv_limit), float(dtmax), C.byref(dt)))
        return dt.value

    def sl_advect(self, T, U, dt, T_cmb=1.0, T_surf=0.0):
        """Semi-Lagrangian update of the vertex temperatures T (nVnod) over dt
        with the rotated-frame velocity U (3*nnod), advect3d_slm_p_sph.m:1.
        Departure points are searched in two rings of elements around each
        vertex; one farther away raises M3Error (dt too large)."""
        T = np.ascontiguousarray(T, dtype=np.float64)
        U = np.ascontiguousarray(U, dtype=np.float64)
        out = np.zeros_like(T)
        self._check(LIB.m3_sl_advect(self._h, _p(T), _p(U), float(dt), float(T_cmb), float(T_surf), _p(out)))
        return out

    def advect3d_slm_p_sph(self, Ux, Uy, Uz, T, dt, method_BT="PC2", method_interp="quadratic", monotonic=1):
        """T advected over dt on the P2 nodes (advect3d_slm_p_sph.m:1-140 with
        OPTS_SLM.method_BT / method_interp / monotonic; Cartesian velocity
        Ux, Uy, Uz on the P2 nodes for 'PC2'; 'EU1' takes the three arrays as
        (v_theta, v_phi, v_r), as backtrack_EU1 does, :145-161).  Returns
        (T, info)."""
        T = np.array(T, dtype=np.float64, copy=True)
        U = [np.ascontiguousarray(u, dtype=np.float64) for u in (Ux, Uy, Uz)]
        o = SlmOpts(SLM_METHOD_BT[method_BT], SLM_METHOD_INTERP[method_interp], int(monotonic))
        info = SlmInfo()
        self._check(LIB.m3_advect3d_slm_p_sph(self._h, _p(U[0]), _p(U[1]), _p(U[2]), _p(T), float(dt), C.byref(o),
                                              C.byref(info)))
        return T, dict(nshift=info.nshift, nunresolved=info.nunresolved)

    def diffusion_mesh(self, EL4=None, nnodT=None, theta_cone=None):
        """Linear tetrahedra of the diffusion step (0-based (nel, 4) over the
        first nnodT nodes).  Default: the finest mesh's vertex tetrahedra on
        the P1 vertices, the grid the temperature lives on here."""
        m = self.mesh
        if EL4 is None:
            EL4, nnodT = m.levels[0].EL2NOD[:, :4], m.nVnod
        EL = np.ascontiguousarray(np.asarray(EL4, dtype=np.int64) + 1, dtype=np.uint32)
        tc = m.theta_cone if theta_cone is None else theta_cone
        self._check(LIB.m3_diffusion_mesh(self._h, _p(EL, U32), len(EL), int(nnodT), float(tc)))
        self._diff_n = int(nnodT)

    def diffusion3d(self, T, kappa, dt, ifix=(), vfix=(), **opts):
        """T = diffusion3d_p(T,kappa,...,TBC,dt) (diffusion3d_p.m:1-116) on the
        tetrahedra of ``diffusion_mesh``; ifix 0-based, vfix the values."""
        T = np.ascontiguousarray(T, dtype=np.float64).copy()
        ifx = np.ascontiguousarray(np.asarray(ifix, dtype=np.int64) + 1)
        vfx = np.ascontiguousarray(np.broadcast_to(np.asarray(vfix, dtype=np.float64), ifx.shape))
        o = diffusion_opts(**opts)
        info = DiffusionInfo()
        self._check(LIB.m3_diffusion3d(self._h, _p(T), float(kappa), float(dt), _p(ifx, I64), _p(vfx),
                                       len(ifx), C.byref(o), C.byref(info)))
        return T, info.as_dict()

    def diffusion_apply(self, which, x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        y = np.zeros_like(x)
        self._check(LIB.m3_diffusion_apply(self._h, int(which), _p(x), _p(y)))
        return y

    def apply(self, which, level, x):
        m = self.mesh
        sizes = {0: 3 * m.levels[level].nnod, 1: 3 * m.nnod, 2: m.nVnod, 3: m.nVnod}
        if which == 4:
            ny = 3 * m.levels[level].nnod
        elif which == 5:
            ny = 3 * m.levels[level + 1].nnod
        else:
            ny = sizes[which]
        x = np.ascontiguousarray(x, dtype=np.float64)
        y = np.zeros(ny)
        self._check(LIB.m3_apply(self._h, which, level, _p(x), _p(y)))
        return y

    def get_vector(self, which, level=0):
        m = self.mesh
        n = m.nVnod if which == 4 else 3 * (m.levels[level].nnod if which in (2, 3) else m.nnod)
        out = np.zeros(n)
        self._check(LIB.m3_get_vector(self._h, which, level, _p(out)))
        return out

    def stats(self):
        out = np.zeros(64, dtype=np.int64)
        self._check(LIB.m3_stats(self._h, _p(out, I64), 64))
        nmg = int(out[0])
        return dict(nmg=nmg, nnzb=[int(v) for v in out[1:1 + nmg]],
                    chol_n=int(out[1 + nmg]), chol_T=int(out[2 + nmg]), chol_tiles=int(out[3 + nmg]),
                    chol_levels=int(out[4 + nmg]), chol_heights=int(out[5 + nmg]),
                    nslot=[int(v) for v in out[6 + nmg:6 + 2 * nmg]],
                    windows=[int(v) for v in out[6 + 2 * nmg:6 + 3 * nmg]],
                    window_entries=[int(v) for v in out[6 + 3 * nmg:6 + 4 * nmg]])


# ---------------------------------------------------------------------------
# reference-named mirrors
# ---------------------------------------------------------------------------

def _ctx(MESH):
    ctx = getattr(MESH, "_m3ctx", None)
    if ctx is None:
        ctx = StokesContext(MESH)
        MESH._m3ctx = ctx
    return ctx


def _sync_els_ref(ctx, MESH, NUMSCALE):
    """MESH.els_ref / NUMSCALE.Dens0_T_bary into the context (set when they change)."""
    els = getattr(MESH, "els_ref", None)
    els = np.zeros(0, dtype=np.int64) if els is None else np.asarray(els)
    d0 = np.asarray(NUMSCALE.get("Dens0_T_bary", np.zeros(0)), dtype=np.float64) if len(els) else np.zeros(0)
    key = (els.tobytes(), d0.tobytes())
    if getattr(ctx, "_ref_key", (b"", b"")) != key:   # a new context has no region
        ctx.set_els_ref(els, d0)
        ctx._ref_key = key


class Csc(C.Structure):
    _fields_ = [("nrow", C.c_int64), ("ncol", C.c_int64), ("nnz", C.c_int64), ("colptr", I64),
                ("rowidx", I64), ("val", D)]


LIB.m3_assembly_stokes_sph_3d_double_jacobian.argtypes = [C.c_void_p, D, D, C.POINTER(Phys),
                                                          C.POINTER(Csc), D, C.POINTER(Csc), C.POINTER(Csc), D]
LIB.m3_assembly_stokes_sph_3d_double_jacobian.restype = C.c_int


def assembly_stokes_sph_3d_double_jacobian(VAR, MESH, PHYSICS, NUMSCALE, OPTS):
    """[KK,Fb,GG,MM,Fpdil,DensEl,ViscIP] (assembly_stokes_sph_3d_double_jacobian.m:1-2)
    through m3_assembly_stokes_sph_3d_double_jacobian: element matrices on the
    GPU, per-entry sums in the library; KK and MM lower-triangular, as the
    reference returns them (SciPy CSC).  DensEl / ViscIP are not returned
    (OPTS.return_dens_el / return_visc_ip are off on this path)."""
    if OPTS.get("nip", 14) != 14:
        raise M3Error(1, "only OPTS.nip = 14 is supported")
    phys = dict(g=PHYSICS["g"], Bscale=NUMSCALE["Bscale"], Dens0=NUMSCALE["Dens0"],
                minVisc=PHYSICS.get("minVisc"), maxVisc=PHYSICS.get("maxVisc"))
    ctx = _ctx(MESH)
    _sync_els_ref(ctx, MESH, NUMSCALE)
    V = np.ascontiguousarray(VAR["Visc"], dtype=np.float64)
    R = np.ascontiguousarray(VAR["Dens"], dtype=np.float64)
    ph = C.byref(phys_struct(phys, type_Dmat=OPTS.get("type_Dmat", "23rd")))
    mats = [Csc(), Csc(), Csc()]
    fp = np.zeros(1)
    ctx._check(LIB.m3_assembly_stokes_sph_3d_double_jacobian(ctx._h, _p(V), _p(R), ph, C.byref(mats[0]), None,
                                                             C.byref(mats[1]), C.byref(mats[2]), _p(fp)))
    arrays = []
    for m in mats:
        cp, ri, va = np.zeros(m.ncol + 1, np.int64), np.zeros(m.nnz, np.int64), np.zeros(m.nnz)
        m.colptr, m.rowidx, m.val = _p(cp, I64), _p(ri, I64), _p(va)
        arrays.append((cp, ri, va, (m.nrow, m.ncol)))
    Fb = np.zeros(3 * MESH.nnod)
    ctx._check(LIB.m3_assembly_stokes_sph_3d_double_jacobian(ctx._h, _p(V), _p(R), ph, C.byref(mats[0]), _p(Fb),
                                                             C.byref(mats[1]), C.byref(mats[2]), _p(fp)))
    KK, GG, MM = [sp.csc_matrix((va, ri, cp), shape=shape) for cp, ri, va, shape in arrays]
    return KK, Fb, GG, MM, float(fp[0]), None, None


def mgpcg_solver_p(ctx, b, x, OPTS):
    """[x,itCG,time,rrms_vec] = mgpcg_solver_p(K1,K,KbD,permKbD,b,x,Ic2f_U,nmg,COMM,OPTS)
    with the operators held by ``ctx`` (mgpcg_solver_p.m:1-2, options :704-713)."""
    t0 = time.perf_counter()
    x, it, hist = ctx.mgpcg(b, x, tol=OPTS.get("tol", 1e-8), is_abs_tol=OPTS.get("is_abs_tol", 1),
                            itmax=OPTS.get("itmax", 50), precision=OPTS.get("precision", "fp64"))
    return x, it, time.perf_counter() - t0, hist


def intermesh_transfer_matrix(MESH, l=0, ndof=3):
    """Ic2f = intermesh_transfer_matrix(GCOORD,EL2NOD,GCOORD_c,EL2NOD_c,ndof)
    (intermesh_transfer_matrix.m:1-79) between level l (fine) and level l+1
    (coarse) of MESH: the P2 interpolation of the parent element at every
    fine node, one row per fine dof (the ndof components share the weights,
    :50-55), as a SciPy CSR matrix."""
    ip, ci, w = MESH.transfer(l)
    nf, nc = MESH.levels[l].nnod, MESH.levels[l + 1].nnod
    rows = np.repeat(np.arange(nf), np.diff(ip))
    R = np.concatenate([ndof * rows + k for k in range(ndof)])
    Cc = np.concatenate([ndof * ci + k for k in range(ndof)])
    return sp.csr_matrix((np.tile(w, ndof), (R, Cc)), shape=(ndof * nf, ndof * nc))


def restrict_stiffmat(MESH, K1=None, ifree=None, fid=None):
    """[KK,Ic2f_U] = restrict_stiffmat(MESH,K1,ifree,fid) (restrict_stiffmat.m:1):
    the Galerkin operators of every multigrid level, formed on the device
    from the K1 assembled in MESH's context (K1 and ifree are held there;
    the arguments are accepted for the reference's signature), returned as
    SciPy BSR matrices (full dof numbering, identity at fixed dofs) together
    with the dof-level transfer matrices."""
    ctx = _ctx(MESH)
    ctx.restrict_stiffmat()
    KK = [get_operator(ctx, l) for l in range(MESH.nmg)]
    Ic2f_U = [intermesh_transfer_matrix(MESH, l) for l in range(MESH.nmg - 1)]
    return KK, Ic2f_U


def cholesky_factorization(MESH):
    """[L,perm] = cholesky_factorization(A) (cholesky_factorization.m:26-36)
    for the coarsest operator of MESH's context: the tile factor stays on the
    device; the returned handle is what ``cholesky_solve`` takes."""
    ctx = _ctx(MESH)
    ctx.cholesky_factorization()
    return ctx


def cholesky_solve(rhs, L):
    """x = cholesky_solve(rhs,L,perm) (cholesky_solve.m:27-43) with the handle
    of ``cholesky_factorization``; rhs and x in the coarse dof numbering
    (fixed dofs give 0)."""
    return L.cholesky_solve(rhs)


def flow3d_patera_mg_sph_p(VAR, MESH, COMM, UBC, SETTINGS, PHYSICS, NUMSCALE, dt=None, **opts):
    """[VAR,Uinfo] = flow3d_patera_mg_sph_p(...) (flow3d_patera_mg_sph_p.m:1): the
    multigrid Stokes solve that flow3d_patera_sph dispatches to."""
    return flow3d_patera_sph(VAR, MESH, COMM, UBC, SETTINGS, PHYSICS, NUMSCALE, dt, **opts)


def flow3d_patera_sph(VAR, MESH, COMM, UBC, SETTINGS, PHYSICS, NUMSCALE, dt=None, **opts):
    """[VAR,Uinfo] = flow3d_patera_sph(...) (flow3d_patera_sph.m:1-9): the MG
    branch (nmg > 1) of flow3d_patera_mg_sph_p; returns Ux,Uy,Uz (Cartesian),
    Uth,Uph,Ur (rotated) and P in VAR (flow3d_patera_mg_sph_p.m:672-681)."""
    if MESH.nmg < 2:
        raise M3Error(1, "only the multigrid branch (nmg > 1) is provided")
    ctx = _ctx(MESH)
    key = (id(UBC["ifix"]), len(UBC["ifix"]))
    if getattr(ctx, "_bc_key", None) != key:
        ctx.set_bc(UBC["ifix"], UBC["vfix"])
        ctx._bc_key = key
    phys = dict(g=PHYSICS["g"], Bscale=NUMSCALE["Bscale"], Dens0=NUMSCALE["Dens0"],
                minVisc=PHYSICS.get("minVisc"), maxVisc=PHYSICS.get("maxVisc"))
    _sync_els_ref(ctx, MESH, NUMSCALE)
    U, P, info = ctx.flow3d(VAR["Visc"], VAR["Dens"], phys, P0=VAR.get("P"), **opts)
    from .fields import rotation_frames
    R = rotation_frames(MESH.GCOORD)
    Uxyz = np.einsum("nij,nj->ni", R, U.reshape(-1, 3))
    VAR = dict(VAR)
    VAR.update(Uth=U[0::3].copy(), Uph=U[1::3].copy(), Ur=U[2::3].copy(), Ux=Uxyz[:, 0].copy(),
               Uy=Uxyz[:, 1].copy(), Uz=Uxyz[:, 2].copy(), P=P)
    return VAR, info


# ---- measurement helpers (no reference counterpart) ------------------------
LIB.m3_residual.argtypes = [C.c_void_p, D, D, D]
LIB.m3_profile.argtypes = [C.c_void_p, C.c_int32]
LIB.m3_profile_read.argtypes = [C.c_void_p, D, C.c_int32]
LIB.m3_get_operator.argtypes = [C.c_void_p, C.c_int32, I64, I32, D]
for _f in ("m3_residual", "m3_profile", "m3_profile_read", "m3_get_operator"):
    getattr(LIB, _f).restype = C.c_int


def residual(ctx, U, P):
    """(|r_U|, |f_U|, |r_P|) RMS norms for the assembled problem."""
    U = np.ascontiguousarray(U, dtype=np.float64)
    P = np.ascontiguousarray(P, dtype=np.float64)
    out = np.zeros(3)
    ctx._check(LIB.m3_residual(ctx._h, _p(U), _p(P), _p(out)))
    return out


def profile(ctx, enable):
    ctx._check(LIB.m3_profile(ctx._h, int(enable)))


LIB.m3_copy_rate.argtypes = [C.c_int32, C.c_int64, C.c_int32, D]
LIB.m3_copy_rate.restype = C.c_int


def copy_rate(nbytes=1 << 30, reps=20, device=0):
    """GB/s (read + write) of a plain device copy of nbytes (m3_copy_rate)."""
    g = C.c_double(0)
    rc = LIB.m3_copy_rate(int(device), int(nbytes), int(reps), C.byref(g))
    if rc:
        raise M3Error(rc, "m3_copy_rate failed")
    return g.value


def profile_read(ctx):
    """Kernel timings since ``profile(ctx, True)``: the fine-level fused sweeps
    (FP64 and mixed) and every other V-cycle kernel, each as launches,
    seconds (HIP events at kernel start and end) and algorithmic bytes."""
    out = np.zeros(9)
    ctx._check(LIB.m3_profile_read(ctx._h, _p(out), 9))
    return dict(n_fp64=int(out[0]), t_fp64=out[1], b_fp64=out[2], n_mixed=int(out[3]), t_mixed=out[4],
                b_mixed=out[5], n_vcycle_other=int(out[6]), t_vcycle_other=out[7], b_vcycle_other=out[8])


def get_operator(ctx, level):
    """Level operator as scipy BSR (3x3 blocks)."""
    st = ctx.stats()
    nn = ctx.mesh.levels[level].nnod
    nb = st["nnzb"][level]
    rp = np.zeros(nn + 1, dtype=np.int64)
    col = np.zeros(nb, dtype=np.int32)
    val = np.zeros(9 * nb)
    ctx._check(LIB.m3_get_operator(ctx._h, level, _p(rp, I64), _p(col, I32), _p(val)))
    return sp.bsr_matrix((val.reshape(nb, 3, 3), col, rp), shape=(3 * nn, 3 * nn))


def diffusion3d_p(T, kappa, MESH, COMM, SETTINGS, TBC, dt):
    """[T] = diffusion3d_p(T,kappa,MESH,COMM,SETTINGS,TBC,dt) (diffusion3d_p.m:1)
    on the vertex tetrahedra of MESH.  SETTINGS["OPTS_D"] holds theta,
    lumping, nip, tol, is_abs_tol, itmax; TBC["ifix"] (0-based) and
    TBC["vfix"] the fixed temperatures."""
    if np.size(np.unique(kappa)) > 1:
        raise M3Error(1, "Diffusivity kappa must be a scalar.")
    ctx = _ctx(MESH)
    if getattr(ctx, "_diff_n", None) != len(T):
        ctx.diffusion_mesh()
    o = {k: v for k, v in (SETTINGS.get("OPTS_D") or {}).items()
         if k in ("theta", "lumping", "nip", "tol", "is_abs_tol", "itmax")}
    T, _ = ctx.diffusion3d(T, float(np.ravel(kappa)[0]), dt, TBC.get("ifix", ()), TBC.get("vfix", ()), **o)
    return T


def advect3d_slm_p_sph(ctx, Ux, Uy, Uz, T, dt, OPTS_SLM=None):
    """[T] = advect3d_slm_p_sph(MESH,COMM,Ux,Uy,Uz,T,dt,OPTS_SLM,WS_SLM)
    (mfiles_SPH/advect3d_slm_p_sph.m:1-140) for a field on the P2 nodes of
    the context's finest mesh.  OPTS_SLM keys method_BT ('PC2' or 'EU1'),
    method_interp ('quadratic') and monotonic (1) default to
    default_numerics_M3TET.m:141-153.  MESH and COMM are the context; the
    search workspace WS_SLM is not needed.  Returns (T, info)."""
    o = dict(method_BT="PC2", method_interp="quadratic", monotonic=1)
    o.update(OPTS_SLM or {})
    return ctx.advect3d_slm_p_sph(Ux, Uy, Uz, T, dt, o["method_BT"], o["method_interp"], o["monotonic"])


def thermal_advdiff_3d_p(VAR, MESH, COMM, PHYSICS, SETTINGS, NUMSCALE, TBC, dt):
    """[VAR] = thermal_advdiff_3d_p(...) (thermal_advdiff_3d_p.m:1-56, 'Diffusion'
    solver, curved edges): diffusion over dt/2, semi-Lagrangian advection over
    dt with the rotated-frame velocity VAR["U"], diffusion over dt/2.  VAR["T"]
    holds the vertex temperatures.  The vertex form of the advection searches
    two rings of elements around each vertex and raises M3Error when a
    departure point lies farther (dt too large); calculate_dt.m bounds dt by
    the domain extents only, so keep dt |u| below an element there, or use
    advect3d_slm_p_sph on the P2 nodes, whose search walks any distance."""
    ctx = _ctx(MESH)
    T = diffusion3d_p(VAR["T"], PHYSICS["kappa"], MESH, COMM, SETTINGS, TBC, dt / 2)
    T = ctx.sl_advect(T, VAR["U"], dt, SETTINGS.get("T_cmb", 1.0), SETTINGS.get("T_surf", 0.0))
    T = diffusion3d_p(T, PHYSICS["kappa"], MESH, COMM, SETTINGS, TBC, dt / 2)
    VAR = dict(VAR)
    VAR["T"] = T
    return VAR
