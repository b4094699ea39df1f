"""ctypes binding of libnatsl.so (the C ABI declared in include/natsl.h).

There is no CPU fallback: if the library has not been built the import of any operator fails
with an explicit error.
"""
from __future__ import annotations

import ctypes
import os
from ctypes import c_char_p, c_float, c_int, c_int64, c_longlong, c_size_t, c_uint64, c_void_p

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "csrc", "libnatsl.so")
STEP_CORE_PATH = os.path.join(_HERE, "_step_core.so")

F32, BF16 = 0, 1
DECAY_NON_LINEAR, QK_L2NORM, INTRA_CHUNK, QUERY_ONLY, FRESH_BLOCK_START, STATES_ONLY = 1, 2, 4, 8, 16, 32
STEP_SYNC_FAILED = 32                                    # the word of a step's shared memory that says that one has failed

_lib = _step_core = None
_entries = None

_SIGNATURES = {
    "natsl_version": (c_int, []),
    "natsl_last_error": (c_char_p, []),
    "natsl_mean_pool": (c_int, [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_hard_select": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_layer_select": (c_int, [c_void_p] * 5 + [c_int] * 4 + [c_void_p]),
    "natsl_route": (c_int, [c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p,
                            c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p]),
    "natsl_softmax_sparse_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                         c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_int, c_int,
                                         c_void_p, c_int, c_int, c_void_p]),
    "natsl_softmax_sparse_fwd_per_tile": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p,
                                         c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_int, c_int,
                                         c_void_p, c_int, c_int, c_void_p]),
    "natsl_softmax_fwd_variant": (c_int, [c_int, c_int, c_int, c_int, c_int, c_int]),
    "natsl_softmax_bwd_workspace_bytes": (c_size_t, [c_int, c_int, c_int]),
    "natsl_softmax_sparse_bwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                         c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                         c_int, c_int, c_int, c_float, c_int, c_int, c_void_p, c_size_t, c_void_p, c_int, c_int, c_int,
                                         c_void_p]),
    "natsl_linear_workspace_bytes": (c_size_t, [c_int64, c_int]),
    "natsl_gdn_chunk_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                    c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_int, c_void_p,
                                    c_size_t, c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_mamba_chunk_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                      c_void_p, c_void_p, c_int,
                                      c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_int, c_void_p, c_size_t,
                                      c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_seq_table": (c_int, [c_void_p, c_int, c_void_p, c_void_p]),
    "natsl_linear_chunk_states": (c_int, [c_int] + [c_void_p] * 10 + [c_int] * 9 + [c_float, c_int, c_void_p, c_size_t, c_int, c_void_p, c_int, c_int, c_void_p, c_void_p]),
    "natsl_linear_chunk_bwd": (c_int, [c_int] + [c_void_p] * 9 + [c_int] + [c_void_p] * 12 + [c_int] * 8 + [c_float, c_int, c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_norm_gate_bwd_workspace_bytes": (c_size_t, [c_int64, c_int]),
    "natsl_norm_gate_bwd": (c_int, [c_void_p] * 14 + [c_size_t, c_int64, c_int, c_int, c_float, c_int, c_void_p]),
    "natsl_norm_gate_logits_fwd": (c_int, [c_void_p] * 7 + [c_int64, c_int, c_int, c_float, c_int, c_void_p]),
    "natsl_norm_gate_logits_bwd": (c_int, [c_void_p] * 14 + [c_size_t, c_int64, c_int, c_int, c_float, c_int, c_void_p]),
    "natsl_row_norm_bwd_workspace_bytes": (c_size_t, [c_int64, c_int]),
    "natsl_row_norm_bwd": (c_int, [c_void_p] * 6 + [c_size_t, c_int64, c_int, c_float, c_int, c_int, c_int, c_void_p]),
    "natsl_short_conv_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                     c_int, c_int, c_void_p]),
    "natsl_short_conv_bwd_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int]),
    "natsl_short_conv_bwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_size_t,
                                     c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]),
    "natsl_row_norm_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_int64, c_int, c_float, c_int, c_int, c_int, c_void_p]),
    "natsl_norm_gate_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_int,
                                    c_float, c_int, c_void_p]),
    "natsl_gdn_recurrent_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                        c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                        c_float, c_int, c_int, c_void_p]),
    "natsl_mamba_recurrent_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                          c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                          c_float, c_int, c_int, c_void_p]),
    "natsl_attn_masked_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "natsl_attn_masked_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                      c_int, c_int, c_float, c_int, c_void_p, c_size_t, c_int64, c_int64, c_void_p]),
    "natsl_attn_masked_static_scratch_bytes": (c_size_t, []),
    "natsl_attn_masked_fwd_static": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
                                             c_int, c_int, c_float, c_int, c_void_p]),
    "natsl_decode_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "natsl_decode_fwd": (c_int, [c_int] + [c_void_p] * 5 + [c_int] * 8 + [c_float, c_int64, c_int64, c_void_p, c_size_t] + [c_void_p] * 11 +
                                [c_int, c_void_p] + [c_int] * 6 + [c_float, c_int, c_void_p]),
    "natsl_linear_chunk_bwd_steps": (c_int, [c_int, c_int, c_void_p, c_int] + [c_void_p] * 9 + [c_int] + [c_void_p] * 12 + [c_int] * 8 +
                                     [c_float, c_int, c_int, c_void_p, c_int, c_int, c_void_p]),
    "natsl_linear_block_sums": (c_int, [c_void_p] * 2 + [c_int] * 5 + [c_void_p, c_int, c_int, c_void_p]),
    "natsl_block_grads": (c_int, [c_void_p, c_int] + [c_void_p] * 3 + [c_int, c_void_p, c_void_p] + [c_int] * 8 + [c_void_p, c_int, c_void_p]),
    "natsl_block_grads_logits": (c_int, [c_void_p] * 2 + [c_int] + [c_void_p] * 3 + [c_int] + [c_void_p] * 2 + [c_int] * 7 + [c_void_p]),
    "natsl_kv_collect": (c_int, [c_void_p, c_void_p, c_longlong, c_void_p, c_void_p, c_longlong, c_void_p] + [c_int] * 12 + [c_void_p]),
    "natsl_kv_counts": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p] + [c_int] * 4 + [c_void_p]),
    "natsl_kv_flags": (c_int, [c_void_p, c_void_p] + [c_int] * 4 + [c_void_p]),
    "natsl_kv_note": (c_int, [c_void_p] * 2 + [c_int] * 4 + [c_void_p] * 2 + [c_int] * 3 + [c_void_p]),
    "natsl_block_tails": (c_int, [c_void_p] + [c_int] * 5 + [c_void_p]),
    "natsl_roll_state": (c_int, [c_void_p] * 4 + [c_int, c_int64, c_int64, c_void_p] + [c_int] * 3 + [c_int64, c_void_p]),
    "natsl_conv_norm_fwd": (c_int, [c_void_p] + [c_int] * 6 + [c_void_p]),
    "natsl_conv_norm_bwd_workspace_bytes": (c_size_t, [c_void_p] + [c_int] * 4),
    "natsl_conv_norm_bwd": (c_int, [c_void_p] + [c_int] * 6 + [c_void_p, c_size_t, c_void_p]),
    "natsl_gates_fwd": (c_int, [c_void_p] * 6 + [c_int64] + [c_int] * 4 + [c_void_p]),
    "natsl_gates_bwd_workspace_bytes": (c_size_t, [c_int64, c_int]),
    "natsl_gates_bwd": (c_int, [c_void_p] * 6 + [c_int] + [c_void_p] * 4 + [c_size_t, c_int64] + [c_int] * 4 + [c_void_p]),
    "natsl_dx_init": (c_int, [c_void_p] * 4 + [c_int] * 6 + [c_void_p]),
    "natsl_hard_select_bwd": (c_int, [c_void_p] * 3 + [c_int] * 5 + [c_void_p]),
    "natsl_project": (c_int, [c_void_p, c_int, c_void_p, c_int64, c_int, c_int, c_void_p]),
    "natsl_project_bwd": (c_int, [c_void_p, c_int, c_void_p, c_void_p] + [c_int] * 4 + [c_void_p]),
    "natsl_layer_front": (c_int, [c_void_p, c_void_p]),
    "natsl_narrow_fwd_pays": (c_int, [c_int64, c_int, c_int]),
    "natsl_narrow_linear_bwd_pays": (c_int, [c_int64, c_int, c_int, c_int]),
    "natsl_narrow_wgrad_pays": (c_int, [c_int64, c_int, c_int, c_int, c_int]),
    "natsl_project_bwd_takes": (c_int, [c_void_p, c_int, c_void_p, c_void_p]),
    "natsl_narrow_wgrad": (c_int, [c_void_p] * 3 + [c_int64, c_int, c_int, c_void_p]),
    "natsl_narrow_wgrad_workspace_bytes": (c_size_t, [c_int64, c_int, c_int]),
    "natsl_narrow_wgrad_split": (c_int, [c_void_p] * 3 + [c_int64, c_int, c_int, c_void_p, c_size_t, c_void_p]),
    "natsl_narrow_linear_bwd": (c_int, [c_void_p] * 3 + [c_int64, c_int, c_int, c_void_p]),
    "natsl_wgrad_workspace_bytes": (c_size_t, [c_void_p, c_int, c_int64, c_int]),
    "natsl_wgrad": (c_int, [c_void_p, c_int, c_void_p, c_int64, c_int, c_int, c_void_p, c_size_t, c_void_p]),
    "natsl_mixed_softmax_variant": (c_int, [c_int, c_int, c_int, c_int, c_int, c_int]),
    "natsl_mixed_workspace_bytes": (c_size_t, [c_int64, c_int]),
    "natsl_order_streams": (c_int, [c_void_p, c_void_p]),
    "natsl_mixed_fwd": (c_int, [c_void_p, c_int, c_void_p, c_void_p]),
    "natsl_layer_step_workspace_bytes": (c_size_t, [c_void_p]),
    "natsl_layer_step_fwd": (c_int, [c_void_p, c_void_p, c_size_t, c_void_p]),
    "natsl_layer_step_sync_bytes": (c_size_t, [c_void_p]),
    "natsl_layer_step_sync_fwd": (c_int, [c_void_p, c_void_p, c_size_t, c_void_p, c_size_t, c_uint64, c_void_p]),
    "natsl_layer_step_gave_up": (c_uint64, [c_int]),
    "natsl_kv_compact": (c_int, [c_void_p, c_void_p, c_longlong, c_int, c_void_p, c_void_p, c_longlong, c_void_p, c_int, c_void_p,
                                 c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]),
}


class NatslError(RuntimeError):
    pass


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise NatslError(
                f"{LIB_PATH} is missing: build it with `python -m neuralattentionsearchlinear_amd._build` "
                "(there is no CPU fallback for the NAtS-L hot path)")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            if hasattr(L, name):
                fn = getattr(L, name)
                fn.restype, fn.argtypes = res, args
        _lib = L
    return _lib


def step_core():
    """The native host side of the layers (csrc/host/step_core.cpp)."""
    global _step_core
    if _step_core is None:
        if not os.path.exists(STEP_CORE_PATH):
            raise NatslError(f"{STEP_CORE_PATH} is missing: build it with `python -m neuralattentionsearchlinear_amd._build`")
        from . import _step_core as core
        _step_core = core
    return _step_core


def entries():
    """What the native host side of the operators calls (csrc/host/mixed_core.cpp)."""
    global _entries
    if _entries is None:
        _entries = step_core().make_entries(lib()._handle)
    return _entries


def exported_symbols():
    return list(_SIGNATURES)


def check(rc: int, what: str):
    if rc == 0:
        return
    msg = lib().natsl_last_error().decode()
    if rc == -2:
        raise NotImplementedError(f"{what}: {msg}")
    if rc == -1:
        raise ValueError(f"{what}: {msg}")
    raise NatslError(f"{what} failed ({rc}): {msg}")


def dtype_code(t: torch.dtype) -> int:
    if t == torch.bfloat16:
        return BF16
    if t == torch.float32:
        return F32
    raise NotImplementedError(f"dtype {t} is not supported by the HIP path (bf16 or fp32)")


def ptr(t):
    return None if t is None else t.data_ptr()


def stream_ptr(device=None):
    """The current stream's handle as a number (the raw query: no Stream object is made)."""
    index = device.index if isinstance(device, torch.device) else device
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)
