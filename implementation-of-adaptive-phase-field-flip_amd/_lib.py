"""ctypes binding of ``libpfflip_hip.so`` (declared in ``include/pfflip.h``).

The library is required: there is no CPU fallback.  Loading works on a
machine without a GPU (the HIP runtime initialises lazily), which is what
the CPU test-suite uses to check the exported ABI.
"""

from __future__ import annotations

import ctypes
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libpfflip_hip.so")

MAX_LEVELS = 16
TILE = 8

PH_VEL_FROM_MOM, PH_PHASE, PH_ZERO, PH_STAR, PH_GRAVITY, PH_RHS, PH_TAGS_IN = 1, 2, 4, 8, 16, 32, 64
GA_G2P, GA_ADVECT, GA_REFLECT, GA_SOLIDS, GA_STATE = 1, 2, 4, 8, 16

P = ctypes.c_void_p
F3 = P * 3
PP = ctypes.POINTER(ctypes.c_void_p)  # a C `T* const x[3]` parameter


class PhaseArgs(ctypes.Structure):
    _fields_ = [
        ("nx", ctypes.c_int32), ("ny", ctypes.c_int32), ("nz", ctypes.c_int32),
        ("flags", ctypes.c_int32),
        ("mass", F3), ("mom", F3), ("vel", F3), ("vel_star", F3), ("valid", F3),
        ("cell_mass", P), ("cell_wsum", P), ("phi_cell", P), ("is_liquid", P),
        ("phi_face", F3), ("beta", F3), ("solid", P), ("rhs", P),
        ("mass_eps", ctypes.c_float), ("rho_min", ctypes.c_float),
        ("alpha_phi", ctypes.c_float), ("rho_0l", ctypes.c_float),
        ("rho_l", ctypes.c_float), ("rho_g", ctypes.c_float),
        ("gravity", ctypes.c_float * 3),
        ("dt", ctypes.c_float), ("dx", ctypes.c_float),
        ("rho_tilde_0", ctypes.c_float), ("k_div", ctypes.c_float),
    ]


MG_UNFUSED_SMOOTHER = 1
MG_SEPARATE_DOTS = 2
MG_SPLIT_LEVELS = 4


class MGLevel(ctypes.Structure):
    _fields_ = [
        ("nx", ctypes.c_int32), ("ny", ctypes.c_int32), ("nz", ctypes.c_int32),
        ("_pad", ctypes.c_int32),
        ("bx", P), ("by", P), ("bz", P), ("diag", P), ("p", P), ("b", P), ("r", P),
        ("bx_h", P), ("by_h", P), ("bz_h", P), ("p_h", P),
    ]


class MG(ctypes.Structure):
    _fields_ = [
        ("nlev", ctypes.c_int32), ("pre", ctypes.c_int32), ("post", ctypes.c_int32),
        ("coarsest", ctypes.c_int32), ("omega", ctypes.c_float),
        ("precision", ctypes.c_int32), ("small_from", ctypes.c_int32),
        ("options", ctypes.c_int32),
        ("lev", MGLevel * MAX_LEVELS),
        ("rhs", P), ("res", P), ("z", P), ("q", P), ("Ap", P), ("scalars", P),
        ("host_state", P),
    ]


class G2PArgs(ctypes.Structure):
    _fields_ = [
        ("px", P), ("pv", P), ("ptype", P), ("pstate", P), ("pflag", P),
        ("n", ctypes.c_int64),
        ("nx", ctypes.c_int32), ("ny", ctypes.c_int32), ("nz", ctypes.c_int32),
        ("flags", ctypes.c_int32),
        ("vel", F3), ("dvel", F3), ("vel_liq", F3), ("solid", P),
        ("dx", ctypes.c_float), ("dt", ctypes.c_float),
        ("alpha_liquid", ctypes.c_float), ("alpha_air", ctypes.c_float),
        ("lo", ctypes.c_float * 3), ("hi", ctypes.c_float * 3),
    ]


class DropletArgs(ctypes.Structure):
    _fields_ = [
        ("px", P), ("pv", P), ("ptype", P), ("pstate", P), ("pdrop_r", P),
        ("n", ctypes.c_int64),
        ("nx", ctypes.c_int32), ("ny", ctypes.c_int32), ("nz", ctypes.c_int32),
        ("seed", ctypes.c_int32),
        ("phi", P), ("shear", P), ("vel", F3),
        ("dx", ctypes.c_float), ("dt", ctypes.c_float), ("delta_phi", ctypes.c_float),
        ("r_mu", ctypes.c_float), ("r_sigma", ctypes.c_float),
        ("r_min", ctypes.c_float), ("r_max", ctypes.c_float),
        ("spray_threshold", ctypes.c_float), ("spray_rate", ctypes.c_float),
        ("gravity", ctypes.c_float * 3),
        ("rho_g", ctypes.c_float), ("rho_l", ctypes.c_float), ("cd", ctypes.c_float),
        ("evap_k", ctypes.c_float),
        ("lo", ctypes.c_float * 3), ("hi", ctypes.c_float * 3),
        ("max_substeps", ctypes.c_int32),
        ("counters", P),
    ]


class MsbgGrid(ctypes.Structure):
    _fields_ = [
        ("nbx", ctypes.c_int32), ("nby", ctypes.c_int32), ("nbz", ctypes.c_int32),
        ("n0", ctypes.c_int32), ("sh0", ctypes.c_int32), ("nslots", ctypes.c_int32),
        ("ncells", ctypes.c_int32), ("h0", ctypes.c_float),
        ("level", P), ("slot", P), ("blk", P), ("blev", P), ("coff", P), ("cslot", P),
    ]


class MrParams(ctypes.Structure):
    _fields_ = [
        ("r0", ctypes.c_float), ("rho_l", ctypes.c_float), ("rho_g", ctypes.c_float),
        ("rho_min", ctypes.c_float), ("alpha_phi", ctypes.c_float), ("rho_0l", ctypes.c_float),
        ("rho_tilde_0", ctypes.c_float), ("k_div", ctypes.c_float), ("gravity", ctypes.c_float * 3),
        ("dt", ctypes.c_float), ("nu_l", ctypes.c_float), ("nu_g", ctypes.c_float),
        ("alpha_cap", ctypes.c_float), ("lo", ctypes.c_float * 3), ("hi", ctypes.c_float * 3),
        ("max_level", ctypes.c_int32),
        ("mass_scale", ctypes.c_double), ("mom_scale", ctypes.c_double), ("w_scale", ctypes.c_double),
    ]


class MrParticles(ctypes.Structure):
    _fields_ = [("x", P), ("v", P), ("type", P), ("level", P), ("defer", P), ("n", ctypes.c_int64)]


class MrFields(ctypes.Structure):
    _fields_ = [(k, P) for k in ("acc", "cwsum", "phi", "is_liquid", "fmass", "fvel", "fvel_star", "fdvel",
                                 "fbeta", "rhs", "pressure")]


# name -> (restype, argtypes); mirrors include/pfflip.h
I32, I64, F32, F64, SZ = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_double, ctypes.c_size_t
SIGNATURES = {
    "pf_last_error": (ctypes.c_char_p, []),
    "pf_abi_version": (ctypes.c_int, []),
    "pf_fill_u32": (ctypes.c_int, [P, I64, ctypes.c_uint32, P]),
    "pf_read_scalars": (ctypes.c_int, [P, P, SZ, P]),
    "pf_bin_nkeys": (I64, [ctypes.c_int, ctypes.c_int, ctypes.c_int]),
    "pf_bin_scan_tmp_bytes": (SZ, [ctypes.c_int, ctypes.c_int, ctypes.c_int]),
    "pf_bin_sort": (ctypes.c_int, [P, P, I64, ctypes.c_int, ctypes.c_int, ctypes.c_int, F32,
                                   P, P, P, P, P, P, P, I32, P]),
    "pf_bin_sort_noalloc": (ctypes.c_int, [P, P, I64, ctypes.c_int, ctypes.c_int, ctypes.c_int, F32,
                                           P, P, P, P, P, P, I32, P]),
    "pf_p2g_stage_bytes": (SZ, [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int]),
    "pf_p2g": (ctypes.c_int, [P, P, P, P, P, ctypes.c_int, ctypes.c_int, ctypes.c_int, F32, F32,
                              P, P, P, P, P, P, P, P, P, P, SZ, P]),
    "pf_phase_beta_forces": (ctypes.c_int, [ctypes.POINTER(PhaseArgs), P]),
    "pf_build_rhs": (ctypes.c_int, [I32, I32, I32, PP, P, P, F32, F32, F32, F32, P]),
    "pf_mg_scalar_bytes": (SZ, []),
    "pf_mg_setup": (ctypes.c_int, [ctypes.POINTER(MG)]),
    "pf_mg_build": (ctypes.c_int, [ctypes.POINTER(MG), P, P, P, P]),
    "pf_mg_precondition": (ctypes.c_int, [ctypes.POINTER(MG), P, P, P]),
    "pf_mg_vcycle": (ctypes.c_int, [ctypes.POINTER(MG), P, P, P]),
    "pf_mgpcg_solve": (ctypes.c_int, [ctypes.POINTER(MG), P, P, F64, I32,
                                      ctypes.POINTER(I32), ctypes.POINTER(F64), P]),
    "pf_mgpcg_state_create": (ctypes.c_int, [ctypes.POINTER(P)]),
    "pf_mgpcg_state_destroy": (ctypes.c_int, [P]),
    "pf_mg_time_smoother": (ctypes.c_int, [ctypes.POINTER(MG), I32, I32, ctypes.POINTER(F32), P]),
    "pf_apply_A": (ctypes.c_int, [ctypes.c_int, ctypes.c_int, ctypes.c_int, P, P, P, P, P, P, P]),
    "pf_project": (ctypes.c_int, [P, PP, PP, PP, PP, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                  F32, F32, P, P]),
    "pf_extrapolate": (ctypes.c_int, [PP, P, PP, PP, PP, PP, ctypes.c_int, ctypes.c_int,
                                      ctypes.c_int, ctypes.c_int, P]),
    "pf_g2p_advect": (ctypes.c_int, [ctypes.POINTER(G2PArgs), P]),
    "pf_g2p_advect_binned": (ctypes.c_int, [ctypes.POINTER(G2PArgs), P, P, P, P, P, P]),
    "pf_max_speed": (ctypes.c_int, [P, P, P, I64, P, P]),
    "pf_droplets": (ctypes.c_int, [ctypes.POINTER(DropletArgs), P]),
    "pf_msbg_apply": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, I32, P]),
    "pf_msbg_residual": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P]),
    "pf_msbg_rbgs": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P, I32, F32, P]),
    "pf_msbg_rbgs_active": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P, P, I32, F32, P, P]),
    "pf_msbg_relax_update": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P, I32, F32, P, P]),
    "pf_msbg_coarsest_max_cells": (I32, []),
    "pf_msbg_coarse_op_max_cells": (I32, []),
    "pf_msbg_coarse_op": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, I32, F32, P, P]),
    "pf_msbg_coarse_apply": (ctypes.c_int, [P, P, P, I32, P]),
    "pf_msbg_coarsest_smooth": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, I32, F32, P]),
    "pf_msbg_rows_bytes": (ctypes.c_size_t, [I32]),
    "pf_msbg_rows_build": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P]),
    "pf_msbg_rows_smooth": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, I32, I32, I32, F32, P]),
    "pf_msbg_rows_apply": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P]),
    "pf_msbg_rows_apply_dot": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, P]),
    "pf_mrcg_update": (ctypes.c_int, [P, P, I32, P, P, P, P, P, P, I64, P, P]),
    "pf_mrcg_direction": (ctypes.c_int, [P, P, I32, P, P, P, P, P, I64, P, P, P, P]),
    "pf_msbg_coarsen_beta": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MsbgGrid), P, P, P]),
    "pf_msbg_restrict": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MsbgGrid), P, P, P]),
    "pf_msbg_prolong_add": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MsbgGrid), P, P, P]),
    "pf_msbg_geometry": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P]),
    "pf_msbg_cover": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P]),
    "pf_vec_reduce_bytes": (SZ, []),
    "pf_vec_reduce": (ctypes.c_int, [I32, P, P, I64, P, P]),
    "pf_vec_axpby": (ctypes.c_int, [F32, P, F32, P, I64, P]),
    "pf_vec_jacobi": (ctypes.c_int, [P, P, P, I64, P]),
    "pf_vec_axpby_dev": (ctypes.c_int, [P, I32, F32, P, I32, P, I64, P, P]),
    "pf_vec_remove_mean": (ctypes.c_int, [P, I64, P, P]),
    "pf_mrcg_scalar": (ctypes.c_int, [I32, P, P, P, P, F64, P]),
    "pf_mr_refine_map": (ctypes.c_int, [ctypes.POINTER(MrParticles), P, I32, I32, I32, F32, F32, I32, P]),
    "pf_mr_max_speed": (ctypes.c_int, [P, I64, P, P]),
    "pf_mr_p2g": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParticles), ctypes.POINTER(MrParams),
                                 ctypes.POINTER(MrFields), P]),
    "pf_mr_p2g_scratch_ints": (I64, [I64, I32]),
    "pf_mr_p2g_sorted": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParticles),
                                        ctypes.POINTER(MrParams), ctypes.POINTER(MrFields), P, P]),
    "pf_mr_finish": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParams), ctypes.POINTER(MrFields), P]),
    "pf_mr_face_prepare": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParams),
                                          ctypes.POINTER(MrFields), P]),
    "pf_mr_rhs": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParams), ctypes.POINTER(MrFields), P]),
    "pf_mr_project": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParams), ctypes.POINTER(MrFields),
                                     P]),
    "pf_mr_max_divergence": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P]),
    "pf_mr_g2p": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParticles), ctypes.POINTER(MrParams),
                                 ctypes.POINTER(MrFields), P]),
    "pf_mr_advect": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), ctypes.POINTER(MrParticles), ctypes.POINTER(MrParams),
                                    P, P]),
    "pf_mr_neighbours": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P]),
    "pf_mr_g2p_near": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, ctypes.POINTER(MrParticles),
                                      ctypes.POINTER(MrParams), ctypes.POINTER(MrFields), P]),
    "pf_mr_advect_near": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, ctypes.POINTER(MrParticles),
                                         ctypes.POINTER(MrParams), P, P]),
    "pf_mr_block_distance": (ctypes.c_int, [ctypes.POINTER(MsbgGrid), P, P, P, P, F32, P]),
    "pf_mr_scan_tmp_ints": (I64, [I64]),
    "pf_mr_classify": (ctypes.c_int, [ctypes.POINTER(MrParticles), P, I32, I32, I32, F32, F32, I32, I32, I32, P, P,
                                      P, P, P]),
    "pf_mr_emit": (ctypes.c_int, [ctypes.POINTER(MrParticles), P, P, P, I32, F32, I32, ctypes.POINTER(MrParticles),
                                  P]),
    "pf_velocity_gradient": (ctypes.c_int, [PP, P, ctypes.c_int, ctypes.c_int, ctypes.c_int, F32, P]),
    "pf_rasterize_spray": (ctypes.c_int, [P, P, P, I64, P, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                          F32, P]),
    "pf_adj_g2p_advect": (ctypes.c_int, [ctypes.POINTER(G2PArgs), P, P, P, P, PP, PP, PP, P]),
    "pf_adj_g2p_advect_binned": (ctypes.c_int, [ctypes.POINTER(G2PArgs), P, P, P, P, P, P, P, PP, PP, PP, P]),
    "pf_adj_extrapolate": (ctypes.c_int, [P, PP, PP, PP, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                          ctypes.c_int, P]),
    "pf_adj_project": (ctypes.c_int, [P, PP, PP, PP, PP, P, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                      F32, F32, P]),
    "pf_adj_solve_beta": (ctypes.c_int, [P, P, PP, ctypes.c_int, ctypes.c_int, ctypes.c_int, P]),
    "pf_adj_phase": (ctypes.c_int, [ctypes.POINTER(PhaseArgs), PP, PP, PP, P, PP, PP, P]),
    "pf_adj_p2g": (ctypes.c_int, [P, P, P, P, I64, PP, PP, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                  F32, F32, P, P, P]),
}

_LIB = None


def load() -> ctypes.CDLL:
    """Load the HIP library (raises if it has not been built)."""
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it first (python __graft_entry__.py or "
                "implementation-of-adaptive-phase-field-flip_amd/build.py)")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _LIB = lib
    return _LIB


class PFError(RuntimeError):
    """A non-zero return from the C ABI."""


def check(rc: int, name: str) -> None:
    if rc != 0:
        msg = load().pf_last_error().decode(errors="replace")
        raise PFError(f"{name} failed with code {rc}: {msg}")


def call(name: str, *args) -> None:
    check(getattr(load(), name)(*args), name)


def ptr(t) -> ctypes.c_void_p | None:
    """Device address of a torch tensor (None passes NULL)."""
    if t is None:
        return None
    return ctypes.c_void_p(t.data_ptr())


def ptr3(ts) -> ctypes.Array:
    return F3(*[None if t is None else t.data_ptr() for t in ts])


def stream():
    import torch
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
