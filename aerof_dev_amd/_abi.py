"""ctypes binding of the aerofx C ABI (include/aerofx.h).

Loads the in-tree library ``aerof_dev_amd/_lib/libaerofx.so``; raises
immediately if it is missing, so no caller can fall back to anything else.
"""
from __future__ import annotations

import ctypes as C
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
# AEROFX_LIB may point at another build of the same library (e.g. a build
# with different compiler flags); the default is the in-tree build.
LIB_PATH = os.environ.get("AEROFX_LIB") or os.path.join(_HERE, "_lib", "libaerofx.so")

AEROFX_BC_ISOTHERMAL_WALL = 1
AEROFX_BC_SLIP_WALL = 2
AEROFX_BC_ADIABATIC_WALL = 3
AEROFX_BC_INLET = 4
AEROFX_BC_OUTLET = 5
AEROFX_MVP_H1 = 0
AEROFX_MVP_FD = 1
AEROFX_MVP_H2 = 2
AEROFX_PREC_JACOBI = 0
AEROFX_PREC_RAS_ILU0 = 1
AEROFX_ERR_ARG = -1
AEROFX_ERR_HIP = -2
AEROFX_ERR_MESH = -3
AEROFX_ERR_NOMEM = -4
AEROFX_ERR_STATE = -5
AEROFX_PHYS_ROEFLUX7 = 0
AEROFX_PHYS_BOUNDFLUX5 = 1
AEROFX_PHYS_VANALBADA = 2
AEROFX_PHYS_ROEJAC6_SW1 = 3
AEROFX_PHYS_ROEJAC6_SW2 = 4
AEROFX_PHYS_INVERT5_F64 = 5
AEROFX_PHYS_INVERT5_F32 = 6
AEROFX_PHYS_ROEFLUX5 = 7
AEROFX_PHYS_ROEJAC6_LM_SW1 = 8
AEROFX_PHYS_ROEJAC6_LM_SW2 = 9
AEROFX_PHYS_ROE_FLUX = 10
AEROFX_PHYS_RECONSTRUCT = 11
AEROFX_PHYS_ROE_JAC_PAIR = 12
TIMER_NAMES = ("nodalGrad", "fvTerm", "fvTermNodes", "fvJac", "fluidPrecSetup", "jacApply",
               "precApply", "gramSchmidt", "feTerm", "feJac")

c_double_p = C.POINTER(C.c_double)
c_int_p = C.POINTER(C.c_int)


class BoxSpec(C.Structure):
    _fields_ = [
        ("nx", C.c_int), ("ny", C.c_int), ("nz", C.c_int),
        ("lo", C.c_double * 3), ("hi", C.c_double * 3),
        ("jitter", C.c_double),
        ("seed", C.c_uint64),
        ("face_code", C.c_int * 6),
        ("nbumps", C.c_int),
        ("bump_amp", c_double_p), ("bump_center", c_double_p), ("bump_width", c_double_p),
    ]


class Params(C.Structure):
    _fields_ = [
        ("gamma", C.c_double), ("pstiff", C.c_double), ("beta", C.c_double),
        ("second_order", C.c_int),
        ("rho_inf", C.c_double), ("p_inf", C.c_double), ("mach", C.c_double),
        ("alpha", C.c_double), ("yaw", C.c_double),
    ]


class Mesh(C.Structure):
    _fields_ = [
        ("num_nodes", C.c_int), ("num_tets", C.c_int), ("num_faces", C.c_int),
        ("X", c_double_p), ("tets", c_int_p), ("faces", c_int_p), ("face_codes", c_int_p),
    ]


class LowMachC(C.Structure):
    _fields_ = [("min_mach", C.c_double), ("slope", C.c_double), ("cutoff", C.c_double),
                ("shock_reducer", C.c_double), ("irey", C.c_double)]


class ViscousC(C.Structure):
    _fields_ = [("reynolds", C.c_double), ("viscosity_model", C.c_int), ("bulk_viscosity", C.c_double),
                ("sutherland_ts", C.c_double), ("conductivity_model", C.c_int), ("prandtl", C.c_double),
                ("conductivity", C.c_double), ("wall_temperature", C.c_double), ("viscous_cst", C.c_double)]


class SowerHeader(C.Structure):
    _fields_ = [("num_nodes", C.c_int), ("num_tets", C.c_int), ("num_faces", C.c_int),
                ("num_clus_nodes", C.c_int), ("num_sub_cluster", C.c_int), ("num_neighbours", C.c_int),
                ("num_bcs", C.c_int), ("version", C.c_double)]


class NewtonOpts(C.Structure):
    _fields_ = [("precision", C.c_int), ("max_steps", C.c_int), ("eps", C.c_double),
                ("cfl0", C.c_double), ("cfl_max", C.c_double), ("ser", C.c_double),
                ("cfl_coef1", C.c_double), ("cfl_coef2", C.c_double),
                ("gmres_m", C.c_int), ("gmres_maxits", C.c_int), ("gmres_eps", C.c_double),
                ("mvp", C.c_int), ("fd_order", C.c_int), ("prec", C.c_int), ("prec_subdomain", C.c_int),
                ("eps_formula", C.c_int), ("failsafe", C.c_int), ("check_final_res", C.c_int)]


class BlockStats(C.Structure):
    _fields_ = [("cycles", C.c_int), ("inner_its", C.c_int), ("converged", C.c_int), ("res_max", C.c_double),
                ("seconds", C.c_double), ("tune_waves_dots", C.c_int), ("tune_waves_update", C.c_int)]


class AdjointOpts(C.Structure):
    _fields_ = [("precision", C.c_int), ("cfl", C.c_double), ("max_its", C.c_int), ("eps", C.c_double),
                ("gmres_m", C.c_int), ("gmres_maxits", C.c_int), ("gmres_eps", C.c_double)]


class AdjointStats(C.Structure):
    _fields_ = [("its", C.c_int), ("converged", C.c_int), ("krylov_its", C.c_int), ("res0", C.c_double),
                ("res", C.c_double), ("seconds", C.c_double)]


class NewtonStats(C.Structure):
    _fields_ = [("steps", C.c_int), ("converged", C.c_int), ("krylov_its", C.c_int),
                ("res0", C.c_double), ("res", C.c_double), ("final_cfl", C.c_double),
                ("seconds", C.c_double), ("failsafe_redos", C.c_int), ("saturated", C.c_int),
                ("final_res_failures", C.c_int)]


# name -> (restype, argtypes); every symbol declared in include/aerofx.h
SIGNATURES = {
    "aerofx_last_error": (C.c_char_p, []),
    "aerofx_version": (C.c_int, []),
    "aerofx_mesh_box_sizes": (C.c_int, [C.POINTER(BoxSpec), c_int_p, c_int_p, c_int_p]),
    "aerofx_mesh_box": (C.c_int, [C.POINTER(BoxSpec), c_double_p, c_int_p, c_int_p, c_int_p]),
    "aerofx_mesh_box_bump_derivative": (C.c_int, [C.POINTER(BoxSpec), C.c_int, C.c_int, c_double_p]),
    "aerofx_mesh_edges": (C.c_int, [C.c_int, C.c_int, c_int_p, c_int_p, c_int_p]),
    "aerofx_mesh_rcm": (C.c_int, [C.c_int, C.c_int, c_int_p, c_int_p]),
    "aerofx_mesh_renumber": (C.c_int, [C.c_int, C.c_int, C.c_int, c_int_p, c_double_p, c_int_p, c_int_p]),
    "aerofx_mesh_color_edges": (C.c_int, [C.c_int, C.c_int, c_int_p, c_int_p, c_int_p]),
    "aerofx_state_init": (C.c_int, [C.POINTER(Params), C.c_int, C.c_double, C.c_uint64, C.c_int,
                                    c_double_p, c_double_p]),
    "aerofx_ctx_create": (C.c_int, [C.POINTER(Mesh), C.POINTER(Params), C.POINTER(C.c_void_p)]),
    "aerofx_ctx_destroy": (C.c_int, [C.c_void_p]),
    "aerofx_ctx_sizes": (C.c_int, [C.c_void_p, c_int_p, c_int_p, c_int_p]),
    "aerofx_ctx_set_stream": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int]),
    "aerofx_ctx_sync": (C.c_int, [C.c_void_p]),
    "aerofx_ctx_set_residual_kernels": (C.c_int, [C.c_void_p, C.c_int]),
    "aerofx_ctx_set_low_mach": (C.c_int, [C.c_void_p, C.POINTER(LowMachC)]),
    "aerofx_ctx_set_viscous": (C.c_int, [C.c_void_p, C.POINTER(ViscousC)]),
    "aerofx_ctx_node_types": (C.c_int, [C.c_void_p, c_int_p]),
    "aerofx_apply_bcs_residual": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_apply_bcs_solution": (C.c_int, [C.c_void_p, C.c_void_p]),
    "aerofx_ctx_set_failsafe": (C.c_int, [C.c_void_p, C.c_int]),
    "aerofx_ctx_set_krylov_check": (C.c_int, [C.c_void_p, C.c_int]),
    "aerofx_ctx_reset_failsafe": (C.c_int, [C.c_void_p]),
    "aerofx_ctx_failsafe_nodes": (C.c_int, [C.c_void_p, c_int_p]),
    "aerofx_ctx_profile": (C.c_int, [C.c_void_p, C.c_int]),
    "aerofx_ctx_timers": (C.c_int, [C.c_void_p, c_double_p, C.POINTER(C.c_longlong)]),
    "aerofx_ctx_tables": (C.c_int, [C.c_void_p, c_int_p, c_double_p, c_double_p, c_double_p, c_double_p]),
    "aerofx_residual": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_residual_ex": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int]),
    "aerofx_residual_noalloc": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int]),
    "aerofx_error_count": (C.c_int, [C.c_void_p, c_int_p]),
    "aerofx_gradients": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_primitive": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_timestep": (C.c_int, [C.c_void_p, C.c_void_p, C.c_double, C.c_void_p]),
    "aerofx_jacobian_setup": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int]),
    "aerofx_jacobian_blocks": (C.c_int, [C.c_void_p, c_double_p, c_double_p]),
    "aerofx_jvp": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_prec_apply": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_gmres": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_double, C.c_int,
                               c_int_p, c_double_p]),
    "aerofx_jvp_fd": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]),
    "aerofx_mvp_select": (C.c_int, [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int]),
    "aerofx_mvp_apply": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_prec_select": (C.c_int, [C.c_void_p, C.c_int, C.c_int]),
    "aerofx_jvp_transpose": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_prec_apply_transpose": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_gmres_transpose": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_double, C.c_int,
                                         c_int_p, c_double_p]),
    "aerofx_block_gmres": (C.c_int, [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_double, C.c_int,
                                     C.c_int, C.c_int, C.POINTER(BlockStats)]),
    "aerofx_mesh_color_edges_gpu": (C.c_int, [C.c_int, C.c_int, c_int_p, c_int_p]),
    "aerofx_mesh_rcm_gpu": (C.c_int, [C.c_int, C.c_int, c_int_p, c_int_p]),
    "aerofx_wall_force": (C.c_int, [C.c_void_p, C.c_void_p, c_double_p, c_double_p, C.c_void_p, C.c_void_p]),
    "aerofx_adjoint_solve": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.POINTER(AdjointOpts),
                                       C.POINTER(AdjointStats)]),
    "aerofx_adjoint_residual": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_direct_solve": (C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p,
                                      C.POINTER(AdjointOpts), C.POINTER(AdjointStats)]),
    "aerofx_residual_derivative": (C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]),
    "aerofx_steady_solve": (C.c_int, [C.c_void_p, C.c_void_p, C.POINTER(NewtonOpts), C.POINTER(NewtonStats),
                                      c_double_p, C.c_int]),
    "aerofx_sower_info": (C.c_int, [C.c_char_p, C.c_char_p, C.c_int, C.POINTER(SowerHeader)]),
    "aerofx_sower_read": (C.c_int, [C.c_char_p, C.c_char_p, C.c_int, c_double_p, c_int_p, c_int_p, c_int_p,
                                    c_int_p, c_int_p]),
    "aerofx_sower_write": (C.c_int, [C.c_char_p, C.c_char_p, C.c_int, C.c_int, C.c_int, c_double_p, c_int_p,
                                     c_int_p, c_int_p]),
    "aerofx_solution_info": (C.c_int, [C.c_char_p, c_int_p, c_int_p, c_int_p]),
    "aerofx_solution_write": (C.c_int, [C.c_char_p, C.c_int, C.c_double, C.c_int, C.c_int, c_double_p]),
    "aerofx_solution_read": (C.c_int, [C.c_char_p, C.c_int, c_double_p, C.c_int, C.c_int, c_int_p, c_double_p]),
    "aerofx_physics_eval": (C.c_int, [C.c_int, C.c_int, C.c_double, C.c_void_p, C.c_void_p, C.c_void_p,
                                      C.c_void_p, C.c_void_p]),
}

_lib = None


def lib() -> C.CDLL:
    """The loaded library with typed signatures (raises if it is not built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"aerofx native library not built: {LIB_PATH} is missing "
                "(run __graft_entry__.build() or make -C aerof_dev_amd/csrc)")
        L = C.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _lib = L
    return _lib


class AerofxError(RuntimeError):
    pass


def check(rc: int, what: str) -> int:
    """Raises AerofxError on rc < 0; returns rc (>= 0) otherwise."""
    if rc < 0:
        msg = lib().aerofx_last_error().decode(errors="replace")
        raise AerofxError(f"{what} failed ({rc}): {msg}")
    return rc
