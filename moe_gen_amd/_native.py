"""ctypes binding of libmoe_mi355.so (the C ABI declared in include/moe_mi355.h).

The library is the only compute path of this package: if it is missing or cannot
be loaded, every operator raises.  There is no PyTorch or CPU fallback.
"""
from __future__ import annotations

import ctypes
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmoe_mi355.so")
PLACES_PATH = os.path.join(_HERE, "_places.so")

c_void_p, c_int32, c_size_t, c_float, c_int64 = (ctypes.c_void_p, ctypes.c_int32, ctypes.c_size_t,
                                                 ctypes.c_float, ctypes.c_int64)


class RouterParams(ctypes.Structure):
    """struct moe_router_params."""
    _fields_ = [
        ("n_tokens", c_int32), ("hidden", c_int32), ("n_experts", c_int32), ("top_k", c_int32),
        ("n_group", c_int32), ("topk_group", c_int32), ("scoring", c_int32), ("method", c_int32),
        ("norm_topk_prob", c_int32), ("scale_mode", c_int32), ("logits_bf16", c_int32),
        ("weights_bf16", c_int32), ("norm_eps", c_float), ("routed_scaling_factor", c_float),
    ]


class MlpGroup(ctypes.Structure):
    """struct moe_mlp_group."""
    _fields_ = [
        ("x", c_void_p), ("x_rows", c_int32), ("n_rows", c_int32), ("row_map", c_void_p),
        ("w_gate", c_void_p), ("w_up", c_void_p), ("w_down", c_void_p),
        ("s_gate", c_void_p), ("s_up", c_void_p), ("s_down", c_void_p), ("offsets", c_void_p),
        ("n_experts", c_int32), ("inter", c_int32), ("max_rows", c_int32), ("fp8", c_int32),
        ("act", c_void_p), ("y", c_void_p), ("workspace", c_void_p), ("workspace_bytes", c_size_t),
    ]


class LayerArgs(ctypes.Structure):
    """struct moe_layer_args."""
    _fields_ = [
        ("x", c_void_p), ("norm_weight", c_void_p), ("w_gate", c_void_p), ("bias", c_void_p),
        ("router", c_void_p), ("routed", c_void_p), ("shared", c_void_p),      # addresses of a RouterParams and two MlpGroup
        ("topk_idx", c_void_p), ("topk_w", c_void_p), ("counts", c_void_p), ("logits_bf16", c_void_p), ("out", c_void_p),
        ("workspace", c_void_p), ("workspace_bytes", c_size_t), ("norm_eps", c_float), ("combine_mode", c_int32),
        ("join_shared", c_int32),
    ]


# name -> (restype, argtypes); every symbol include/moe_mi355.h declares
SIGNATURES = {
    "moe_last_error": (ctypes.c_char_p, []),
    "moe_version": (ctypes.c_char_p, []),
    "moe_router": (ctypes.c_int, [c_void_p, c_void_p, c_void_p, ctypes.POINTER(RouterParams), c_void_p,
                                  c_void_p, c_void_p, c_void_p]),
    "moe_router_rmsnorm": (ctypes.c_int, [c_void_p, c_void_p, ctypes.c_float, c_void_p, c_void_p,
                                          ctypes.POINTER(RouterParams), c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "moe_dispatch_workspace_bytes": (c_size_t, [c_int32, c_int32, c_int32]),
    "moe_dispatch": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_int32, c_void_p, c_void_p, c_void_p,
                                    c_void_p, c_void_p, c_void_p, c_int32, c_void_p, c_void_p, c_size_t, c_void_p]),
    "moe_dispatch_static": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_int32, c_void_p, c_void_p, c_void_p,
                                           c_void_p, c_void_p, c_void_p, c_int32, c_void_p, c_void_p]),
    "moe_grouped_workspace_bytes": (c_size_t, [c_int32, c_int32]),
    "moe_grouped_swiglu_bf16": (ctypes.c_int, [c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                               c_int32, c_int32, c_int32, c_int32, c_void_p, c_void_p,
                                               c_int32, c_void_p, c_size_t, c_void_p]),
    "moe_grouped_swiglu_w8a16": (ctypes.c_int, [c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                                c_void_p, c_void_p, c_void_p, c_int32, c_int32, c_int32,
                                                c_int32, c_void_p, c_void_p, c_int32, c_void_p, c_size_t, c_void_p]),
    "moe_grouped_swiglu_joint": (ctypes.c_int, [ctypes.POINTER(MlpGroup), ctypes.POINTER(MlpGroup), c_int32, c_int32, c_int32,
                                                c_void_p]),
    "moe_mlp_workspace_bytes": (c_size_t, [ctypes.POINTER(MlpGroup), c_int32]),
    "moe_shared_joins": (ctypes.c_int, [ctypes.POINTER(MlpGroup), ctypes.POINTER(MlpGroup), c_int32]),
    "moe_layer_workspace_bytes": (c_size_t, [ctypes.POINTER(LayerArgs)]),
    "moe_layer_forward": (ctypes.c_int, [ctypes.POINTER(LayerArgs), c_void_p]),
    "moe_dequant_fp8_block128": (ctypes.c_int, [c_void_p, c_void_p, c_int32, c_int32, c_void_p, c_void_p]),
    "moe_combine": (ctypes.c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int32, c_int32,
                                   c_int32, c_int32, c_void_p, c_void_p]),
    "moe_combine_residual": (ctypes.c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int32,
                                            c_int32, c_int32, c_int32, c_void_p, c_void_p]),
    "moe_rmsnorm": (ctypes.c_int, [c_void_p, c_void_p, ctypes.c_float, c_int32, c_int32, c_void_p, c_void_p]),
    "moe_arena_index_create": (ctypes.c_int, [ctypes.POINTER(c_void_p)]),
    "moe_arena_index_destroy": (ctypes.c_int, [c_void_p]),
    "moe_arena_index_add": (ctypes.c_int, [c_void_p, ctypes.c_char_p, ctypes.c_char_p, ctypes.c_int64, ctypes.c_int64,
                                           ctypes.POINTER(ctypes.c_int64), c_int32]),
    "moe_arena_index_parse": (ctypes.c_int, [c_void_p, c_size_t, ctypes.POINTER(c_void_p)]),
    "moe_arena_index_wire_size": (c_size_t, [c_void_p]),
    "moe_arena_index_serialize": (ctypes.c_int, [c_void_p, c_void_p, c_size_t]),
    "moe_arena_index_n_modules": (c_int32, [c_void_p]),
    "moe_arena_index_module": (ctypes.c_int, [c_void_p, c_int32, ctypes.POINTER(ctypes.c_char_p),
                                              ctypes.POINTER(c_int32)]),
    "moe_arena_index_find": (ctypes.c_int, [c_void_p, ctypes.c_char_p]),
    "moe_arena_index_tensor": (ctypes.c_int, [c_void_p, c_int32, c_int32, ctypes.POINTER(ctypes.c_char_p),
                                              ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_int64),
                                              ctypes.POINTER(c_int32), ctypes.POINTER(ctypes.POINTER(ctypes.c_int64))]),
    "moe_stage_add_module_from_arena": (ctypes.c_int, [c_void_p, c_int32, c_void_p, ctypes.c_char_p, c_void_p, c_size_t,
                                                       c_int32, ctypes.POINTER(ctypes.c_char_p),
                                                       ctypes.POINTER(c_size_t)]),
    "moe_stage_add_module_from_segment": (ctypes.c_int, [c_void_p, c_int32, c_void_p, ctypes.c_char_p, c_void_p, c_size_t,
                                                         c_int32, ctypes.POINTER(ctypes.c_char_p),
                                                         ctypes.POINTER(c_size_t)]),
    "moe_write_words": (ctypes.c_int, [c_void_p, ctypes.POINTER(ctypes.c_uint64), c_int32, c_void_p]),
    "moe_stage_set_bounce": (ctypes.c_int, [c_void_p, c_int32, c_size_t, c_int32]),
    "moe_stage_add_module_pageable": (ctypes.c_int, [c_void_p, c_int32, c_int32, ctypes.POINTER(c_void_p),
                                                     ctypes.POINTER(c_size_t), ctypes.POINTER(c_size_t)]),
    "moe_stage_create": (ctypes.c_int, [ctypes.POINTER(c_void_p), c_int32, ctypes.POINTER(c_size_t),
                                        ctypes.POINTER(c_int32), ctypes.POINTER(c_void_p), c_int32]),
    "moe_stage_set_policy": (ctypes.c_int, [c_void_p, c_int32, c_int32]),
    "moe_stage_fetch": (ctypes.c_int, [c_void_p, ctypes.POINTER(c_int32), c_int32, ctypes.POINTER(c_int32)]),
    "moe_stage_add_module": (ctypes.c_int, [c_void_p, c_int32, c_int32, ctypes.POINTER(c_void_p),
                                            ctypes.POINTER(c_size_t), ctypes.POINTER(c_size_t)]),
    "moe_stage_pump": (ctypes.c_int, [c_void_p]),
    "moe_stage_acquire": (ctypes.c_int, [c_void_p, c_int32, c_void_p, ctypes.POINTER(c_int32)]),
    "moe_stage_release": (ctypes.c_int, [c_void_p, c_int32, c_void_p]),
    "moe_stage_resident": (ctypes.c_int, [c_void_p, c_int32]),
    "moe_stage_set_active_slots": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_int32]),
    "moe_stage_set_model": (ctypes.c_int, [c_void_p, ctypes.c_char_p, c_int32, c_int32]),
    "moe_stage_tag_module": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_int32]),
    "moe_stage_clear_expert_buffer": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_void_p]),
    "moe_stage_set_phase_slots": (ctypes.c_int, [c_void_p, c_int32, c_int32, c_int32]),
    "moe_stage_set_phase": (ctypes.c_int, [c_void_p, ctypes.c_char_p]),
    "moe_stage_reset_prefill_buffer": (ctypes.c_int, [c_void_p]),
    "moe_stage_reset_weight_copy_queue": (ctypes.c_int, [c_void_p]),
    "moe_stage_stats": (ctypes.c_int, [c_void_p, ctypes.POINTER(c_int64), ctypes.POINTER(c_int64)]),
    "moe_stage_sync": (ctypes.c_int, [c_void_p]),
    "moe_stage_destroy": (ctypes.c_int, [c_void_p]),
}

_lib = None
_places_hold = None


def places_hold(objects: list, tensors: list, addresses) -> bool:
    """Whether every object of [dict, key, object, ...] is still there and every tensor of [dict, key, ...] at its address (an
    array of 64-bit integers)."""
    global _places_hold
    if _places_hold is None:
        if not os.path.exists(PLACES_PATH):
            raise RuntimeError(f"{PLACES_PATH} is missing: build it with `make -C {os.path.join(_HERE, 'csrc')}`")
        import torch  # noqa: F401  (its libraries are what _places.so is linked against)
        f = ctypes.PyDLL(PLACES_PATH).moe_places_hold
        f.argtypes, f.restype = [ctypes.py_object, ctypes.py_object, c_void_p], ctypes.c_int
        _places_hold = f
    return bool(_places_hold(objects, tensors, addresses.buffer_info()[0]))


def lib() -> ctypes.CDLL:
    """Load libmoe_mi355.so (built by `make -C moe_gen_amd/csrc` or __graft_entry__.build())."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `make -C {os.path.join(_HERE, 'csrc')}` "
                "(hipcc --offload-arch=gfx950). This package has no other compute path.")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _lib = L
    return _lib


def last_error() -> str:
    return lib().moe_last_error().decode()


def check(rc: int, what: str) -> None:
    """Mirror of the reference's convention: native failure -> RuntimeError with the message."""
    if rc != 0:
        raise RuntimeError(f"{what} failed (status {rc}): {last_error()}")
