"""ctypes binding of libmortar_hip.so (the C-ABI declared in include/mortar_hip.h) and the native call layer above it
(_mortar_native.so, csrc/mortar_torch.cpp).

There is no fallback: if a library is missing or a call fails, a RuntimeError is raised.
"""
from __future__ import annotations

import ctypes as C
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmortar_hip.so")
NATIVE_PATH = os.path.join(_HERE, "_mortar_native.so")

c_i32, c_i64, c_vp, c_f32 = C.c_int32, C.c_int64, C.c_void_p, C.c_float


class BcsrStruct(C.Structure):
    """mortar_bcsr_t"""
    _fields_ = [("codes", c_vp), ("sdup", c_vp), ("col", c_vp), ("row_ptr", c_vp), ("row_desc", c_vp),
                ("codes_o", c_vp), ("sd_o", c_vp), ("col_o", c_vp), ("codes4_o", c_vp),
                ("Rb", c_i32), ("Cb", c_i32), ("nnz", c_i32),
                ("seg_cb", c_i32), ("uniform_scale", c_f32), ("one_scale", c_i32)]


class RepackStruct(C.Structure):
    """mortar_repack_t"""
    _fields_ = [("W", c_vp), ("Wt", c_vp), ("pos", c_vp), ("pos_t", c_vp), ("src_t", c_vp), ("values", c_vp), ("scale_out", c_vp),
                ("status", c_vp), ("status_t", c_vp), ("workspace", c_vp), ("values_f32", c_i32), ("threshold", c_f32)]


_SIGS = {
    "mortar_last_error": (C.c_char_p, []),
    "mortar_abi_version": (C.c_int, []),
    "mortar_encode_blocks_host": (C.c_int, [c_vp, c_i64, c_vp, c_i64, c_vp, c_vp]),
    "mortar_uniform_scale_host": (C.c_int, [c_vp, c_i64, c_vp]),
    "mortar_decode_blocks_host": (C.c_int, [c_vp, c_i64, c_vp]),
    "mortar_octet_layout_host": (c_i64, [c_vp, c_i32, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp, c_vp, c_vp, c_vp]),
    "mortar_fp4_stream_host": (C.c_int, [c_vp, c_i64, c_vp]),
    "mortar_octet_positions_host": (C.c_int, [c_vp, c_i32, c_i32, c_i32, c_vp, c_vp]),
    "mortar_transpose_topology_host": (C.c_int, [c_vp, c_vp, c_i32, c_i32, c_vp, c_vp, c_vp]),
    "mortar_requantize_workspace_bytes": (c_i64, []),
    "mortar_requantize": (C.c_int, [c_vp, c_vp, c_i32, c_vp, c_vp, c_i32, c_i32, c_f32, c_vp, c_vp, c_vp, c_i32, c_f32,
                                  c_vp, c_vp]),
    "mortar_requantize_pairs": (C.c_int, [c_vp, c_i32, c_vp]),
    "mortar_poison_on_status": (C.c_int, [c_vp, c_i64, c_vp, c_vp]),
    "mortar_swiglu_bf16": (C.c_int, [c_vp, c_i64, c_i64, c_i32, c_vp, c_i64, c_vp]),
    "mortar_swiglu_backward_bf16": (C.c_int, [c_vp, c_i64, c_vp, c_i64, c_i64, c_i32, c_vp, c_i64, c_vp]),
    "mortar_sdd_blocks_per_wave_host": (c_i32, [c_vp, c_vp, c_i32, c_i32, c_i64]),
    "mortar_sdd_plan_host": (c_i64, [c_vp, c_vp, c_i32, c_i32, c_i32, c_vp, c_i64]),
    "mortar_sdd_workspace_bytes": (c_i64, [c_i32, c_i32, c_i32, c_i64]),
    "mortar_sdd_bf16": (C.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp, c_i64, c_vp, c_i64, c_i64, c_vp, c_vp, c_vp]),
    "mortar_prefill_max_seg_cb": (C.c_int, []),
    "mortar_prefill_form_host": (C.c_int, [c_i32, c_i64, c_i32, c_i32, c_i32, c_i32, c_vp, c_vp]),
    "mortar_decode_max_seg_cb": (C.c_int, [c_i32]),
    "mortar_validate_bcsr_host": (C.c_int, [c_vp, c_vp, c_i32, c_i32]),
    "mortar_schedule_host": (C.c_int, [c_vp, c_i32, c_i32, c_i32, c_vp, c_vp]),
    "mortar_unit_order_host": (C.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_vp]),
    "mortar_unit_order_segments_host": (C.c_int, [c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp]),
    "mortar_decode_worklist_host": (c_i64, [c_vp, c_vp, c_i32, c_i32, c_i32, c_i32, c_i32, c_vp, c_vp, c_vp]),
    "mortar_spmm_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_i64, c_vp]),
    "mortar_gateup_swiglu_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_i64, c_vp, c_i32,
                                            c_vp, c_vp, c_vp]),
    "mortar_norm_gateup_swiglu_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_f32, c_vp, c_i64, c_vp, c_i32,
                                                 c_vp, c_vp, c_vp]),
    "mortar_norm_fusable": (C.c_int, [c_i32]),
    "mortar_norm_gateup_decode_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_f32, c_vp, c_i64, c_vp]),
    "mortar_values_seg_cb": (c_i32, [c_i32]),
    "mortar_segment_ptr_host": (C.c_int, [c_vp, c_vp, c_i32, c_i32, c_i32, c_vp]),
    "mortar_dds_values_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_vp, c_i32, c_i32, c_i64, c_vp, c_i64, c_i64, c_vp, c_i64, c_vp]),
    "mortar_transpose_blocks_bf16": (C.c_int, [c_vp, c_vp, c_i64, c_vp, c_vp]),
    "mortar_mlp_hidden_bytes": (c_i64, [c_i64, c_i32]),
    "mortar_mlp_bf16": (C.c_int, [c_vp, c_vp, c_vp, c_vp, c_vp, c_i64, c_i64, c_i32, c_vp, c_f32, c_vp, c_i32, c_vp, c_vp, c_i64,
                                  c_i32, c_vp]),
    "mortar_spmm_bf16_masked": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_i64, c_vp, c_i32, c_vp]),
    "mortar_route_tile": (C.c_int, [c_i32, c_i64]),
    "mortar_remoe_gates": (C.c_int, [c_vp, c_i64, c_i32, c_i32, c_vp, c_vp, c_vp]),
    "mortar_remoe_route": (C.c_int, [c_vp, c_i64, c_i32, c_i32, c_vp, c_vp, c_vp]),
    "mortar_router_bf16": (C.c_int, [c_vp, c_i32, c_i64, c_i32, c_i64, c_vp, c_vp, c_vp, c_vp, c_f32, c_vp, c_vp, c_i32,
                                     c_vp, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp, c_vp]),
    "mortar_norm_router_bf16": (C.c_int, [c_vp, c_i64, c_i32, c_i64, c_vp, c_f32, c_vp, c_vp, c_vp, c_vp, c_vp, c_f32, c_vp, c_vp, c_i32,
                                          c_vp, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp, c_vp]),
    "mortar_router_tail_f32": (C.c_int, [c_vp, c_i64, c_i32, c_i64, c_vp, c_vp, c_vp, c_f32, c_vp, c_vp, c_i32, c_vp, c_i32,
                                         c_i32, c_vp, c_vp, c_vp, c_vp]),
    "mortar_router_project_bf16": (C.c_int, [c_vp, c_i64, c_i32, c_i64, c_vp, c_i32, c_vp, c_i64, c_vp]),
    "mortar_router_stats_workspace_bytes": (c_i64, [c_i64, c_i32]),
    "mortar_router_stats": (C.c_int, [c_vp, c_i64, c_i32, c_f32, c_f32, c_f32, c_vp, c_vp, c_vp, c_vp]),
    "mortar_route_flags": (C.c_int, [c_vp, c_i64, c_i32, c_i64, c_i32, c_vp, c_i64, c_vp, c_i64, c_vp]),
    "mortar_stack_table_bytes": (c_i64, [c_i32]),
    "mortar_stack_prepare": (C.c_int, [c_i32, c_i32, c_vp, c_vp, c_vp, c_vp, c_i64, c_i64, c_i64, c_vp, c_vp]),
    "mortar_stack_run": (C.c_int, [c_i32, c_i32, c_vp, c_i64, c_vp, c_vp]),
    "mortar_gemv_bf16": (C.c_int, [c_vp, c_vp, c_i64, c_i32, c_vp, c_i32, c_i32, c_vp, c_i32, c_i64, c_vp, c_i64,
                                   c_vp, c_vp, c_i32, c_i64, c_vp, c_i64, c_vp, c_i64, c_vp]),
    "mortar_rmsnorm_bf16": (C.c_int, [c_vp, c_i64, c_i32, c_i64, c_vp, c_f32, c_vp, c_i64, c_vp]),
    "mortar_spmm_hc_post": (C.c_int, [c_vp, c_vp, c_vp, c_i64, c_i64, c_vp, c_i32, c_i32, c_vp, c_vp, c_vp, c_vp, c_vp, c_i32, c_vp]),
    "mortar_gemv_f32_workspace_bytes": (c_i64, [c_vp, c_i32, c_i32]),
    "mortar_gemv_f32": (C.c_int, [c_vp, c_vp, c_i64, c_vp, c_vp, c_i64, c_i32, c_vp, c_i32, c_i32, c_i32, c_vp, c_i32, c_i64, c_vp, c_i64,
                                  c_vp, c_i64, c_vp, c_i32, c_i64, c_vp, c_i64, c_vp, c_i64, c_vp]),
    "mortar_gemv_f32_one_better": (C.c_int, [c_vp, c_i32, c_i32]),
    "mortar_gemv_f32_one": (C.c_int, [c_vp, c_vp, c_i32, c_i32, c_vp, c_i32, c_i64, c_vp, c_i64, c_vp, c_i32, c_i64, c_vp, c_i64, c_vp, c_i64,
                                      c_vp]),
    "mortar_gemv_noalloc_max_floats": (c_i64, []),
    "mortar_gemv_bf16_noalloc": (C.c_int, [c_vp, c_vp, c_i64, c_i32, c_vp, c_i32, c_i32, c_vp, c_i32, c_i64, c_vp, c_i64,
                                           c_vp, c_i32, c_i64, c_vp, c_i64, c_vp, c_i64, c_vp]),
}

class PackHandle(C.Structure):
    """One packed matrix for the native call layer: its mortar_bcsr_t, the schedules built so far and, once it has been re-packed,
    what a re-pack needs beside the values."""
    _fields_ = [("w", c_vp), ("sched1", c_vp), ("sched2", c_vp), ("pos", c_vp), ("src", c_vp), ("status", c_vp), ("workspace", c_vp)]


class TopologyHandle(C.Structure):
    """One pack.BcsrTopology for the native call layer."""
    _fields_ = [("row_ptr", c_vp), ("col", c_vp), ("seg_ptr", c_vp), ("src", c_vp), ("Rb", c_i32), ("Cb", c_i32), ("nnz", c_i64)]


EXPORTS = tuple(_SIGS)
_lib = None
_native = None


def lib():
    """The loaded library.  Raises if it has not been built (run `python build.py` in the package)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: the MORTAR HIP extension has not been built "
                "(run __graft_entry__.build() or `python build.py` in the package directory)")
        l = C.CDLL(LIB_PATH)
        for name, (res, args) in _SIGS.items():
            fn = getattr(l, name)
            fn.restype, fn.argtypes = res, args
        _lib = l
    return _lib


def native():
    """The native call layer.  Raises if it has not been built."""
    global _native
    if _native is None:
        lib()                                   # one copy of the library for both bindings
        if not os.path.exists(NATIVE_PATH):
            raise RuntimeError(f"{NATIVE_PATH} is missing: the native call layer has not been built "
                               "(run __graft_entry__.build() or `python build.py` in the package directory)")
        import importlib.machinery
        import importlib.util
        loader = importlib.machinery.ExtensionFileLoader("_mortar_native", NATIVE_PATH)
        mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_mortar_native", loader))
        loader.exec_module(mod)
        _native = mod
    return _native


def check(rc: int, what: str) -> int:
    if rc < 0:
        msg = lib().mortar_last_error().decode("utf-8", "replace")
        err = ValueError if rc in (-1, -2, -4) else RuntimeError
        raise err(f"{what} failed ({rc}): {msg}")
    return rc
