"""The layers' generation step as one native call (natsl_layer_step_sync_fwd): a few new tokens of cached sequences, from the hidden
states to the layer's output, with the cache's new rows written in place.

A step of a layer is a few microseconds of memory traffic per kernel, so what it costs is launches and host time: the same step
as separate torch operations and operator calls is forty launches and ~0.57 ms of host time (340M geometry), this is one
launch for one token of few sequences, three for more, five for several tokens a sequence, and at most 20 us behind one call of
csrc/host/step_core.cpp, which also compares the layer with its plan, checks the cache's tensors and allocates the step's.  `layer_step` declines (returns None) whatever the call is not built for -- other dtypes,
tensors that want gradients, replaced or hooked submodules, the 'attn' mode, more than 64 new tokens in all -- and the layers'
general path runs.
"""
from __future__ import annotations

import ctypes
import weakref

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from . import _capi
from .modules import FusedMultiInputRMSNormGated, L2Norm, RMSNorm, ShortConvolution

MAX_ROWS = 64
MAX_WAIT_US = 10_000_000                                 # what a part of a step's launch waits for another before it gives up

_INTS = ("B", "T", "D", "H", "K", "V", "HQ", "HN", "block", "conv_width", "is_delta", "flags", "n_in", "n_kept", "cache_tokens", "types_dtype",
         "norm_dtype", "gate_dtype", "out_norm_dtype", "reserved")
_FLOATS = ("scale_attn", "scale_linear", "norm_eps", "l2_eps", "out_norm_eps", "reserved_f")
_WEIGHTS = ("wq", "wk", "wv", "wg", "wa", "wb", "w_mix", "wo", "conv_wq", "conv_wk", "conv_wv", "conv_bq", "conv_bk", "conv_bv", "norm_q", "norm_k",
            "a_log", "dt_bias", "out_norm1", "out_norm2")
_TENSORS = ("x", "types", "conv_state_q", "conv_state_k", "conv_state_v", "conv_out_q", "conv_out_k", "conv_out_v", "state", "g_cumsum",
            "block_start", "state_out", "g_cumsum_out", "cache_k", "cache_v", "cache_valid", "block_k", "block_v", "block_g", "block_beta",
            "block_hidden", "out")


class LayerStep(ctypes.Structure):
    """natsl_layer_step of include/natsl.h."""
    _fields_ = ([(n, ctypes.c_int32) for n in _INTS] + [(n, ctypes.c_float) for n in _FLOATS] +
                [(n, ctypes.c_void_p) for n in _WEIGHTS + _TENSORS])


DECAY, SILU, ATTN_FROM_CONV, ATTN_NORM, L2_ROWS, ATTN_OWN_BLOCK, NEG_EIGVAL, FRESH_START = (1 << i for i in range(8))

# where the weights are: (field, submodule or None, parameter, exact submodule type or None)
_PARAMS = (("wq", "q_proj", "weight", nn.Linear), ("wk", "k_proj", "weight", nn.Linear), ("wv", "v_proj", "weight", nn.Linear),
           ("wg", "g_proj", "weight", nn.Linear), ("wa", "a_proj", "weight", nn.Linear), ("wb", "b_proj", "weight", nn.Linear),
           ("w_mix", "nats_out_weights_layer", "weight", nn.Linear), ("wo", "o_proj", "weight", nn.Linear),
           ("conv_wq", "q_conv1d", "weight", ShortConvolution), ("conv_wk", "k_conv1d", "weight", ShortConvolution),
           ("conv_wv", "v_conv1d", "weight", ShortConvolution), ("conv_bq", "q_conv1d", "bias", None), ("conv_bk", "k_conv1d", "bias", None),
           ("conv_bv", "v_conv1d", "bias", None), ("norm_q", "q_norm", "weight", RMSNorm), ("norm_k", "k_norm", "weight", RMSNorm),
           ("a_log", None, "A_log", None), ("dt_bias", None, "dt_bias", None), ("out_norm1", "o_norm", "weight1", FusedMultiInputRMSNormGated),
           ("out_norm2", "o_norm", "weight2", FusedMultiInputRMSNormGated))
_OPTIONAL = {"wb", "norm_q", "norm_k", "conv_bq", "conv_bk", "conv_bv"}
_EITHER_DTYPE = {"norm_q", "norm_k", "a_log", "dt_bias", "out_norm1", "out_norm2"}       # the others are bf16


# by layer, outside of it: a copied or saved layer takes nothing of this along
_watches = weakref.WeakKeyDictionary()


# what the plans are made from besides the weights: a layer's options, and those of its submodules
_OPTIONS = ("hidden_size", "head_k_dim", "head_v_dim", "head_attn_k_dim", "head_attn_v_dim", "num_heads", "num_v_heads", "num_attn_heads",
            "num_nats_head", "nats_block_size", "ops_for_incomplete_chunks", "use_short_conv", "conv_size", "attn_with_short_conv", "attn_qk_norm",
            "allow_neg_eigval", "decay_for_non_gdn_blocks", "decay_for_non_mamba_blocks", "value_dim")
_SUB_OPTIONS = ("eps", "kernel_size", "activation")
_SUBMODULES = tuple({p[1]: p[3] for p in _PARAMS if p[1] is not None and p[3] is not None}.items()) + (("q_norm2", L2Norm), ("k_norm2", L2Norm))
_PLAIN_TENSORS = {nn.Parameter, torch.Tensor, type(None)}


def weight_shapes(layer):
    """The weights' shapes under the layer's options, by field: what the kernels address.  A layer with others (a replaced projection, a
    pruned head) is left to its submodules, which take or refuse them."""
    D, qk, vd, H, W = layer.hidden_size, layer.num_heads * layer.head_k_dim, layer.value_dim, layer.num_heads, layer.conv_size
    s = dict(wq=(qk, D), wk=(qk, D), wv=(vd, D), wg=(vd, D), wa=(H, D), wb=(H, D), w_mix=(2 * layer.num_attn_heads, qk), wo=(D, vd),
             conv_wq=(qk, 1, W), conv_wk=(qk, 1, W), conv_wv=(vd, 1, W), conv_bq=(qk,), conv_bk=(qk,), conv_bv=(vd,), a_log=(H,), dt_bias=(H,))
    s["norm_q"] = s["norm_k"] = (layer.head_attn_k_dim,)
    s["out_norm1"] = s["out_norm2"] = (layer.head_attn_v_dim,)
    return s


class _Watch:
    """What a layer's plans were made from besides its weights' values: which weights and plain submodules it has, the options, and the
    weights' addresses, types and layouts.  No tensor or module is held: a replaced weight is freed when its owner lets go of it."""

    def __init__(self, layer):
        mods = layer._modules
        absent = [n for n, _ in _SUBMODULES if mods.get(n) is None]
        parts, self.plain = [], True                       # parts: (name, type, its parameters, its options, their values)
        weights = [*layer._parameters.values()]
        for n, kind in _SUBMODULES:
            m = mods.get(n)
            if m is not None:
                options = [o for o in _SUB_OPTIONS if o in m.__dict__]
                parts.append((n, type(m), [*m._parameters], options, [m.__dict__[o] for o in options]))
                weights += m._parameters.values()
                self.plain &= type(m) is kind
        options = [o for o in _OPTIONS if o in layer.__dict__]
        self.plain &= {*map(type, weights)} <= _PLAIN_TENSORS
        self.core = _capi.step_core().make_watch(parts, [*layer._parameters], absent, options, [layer.__dict__[o] for o in options],
                                                 weights) if self.plain else None
        self.step_plan = self.front_plan = self.native_plan = None

    def weights(self, layer):
        """The weights by field, None where the layer has none."""
        mods, out = layer._modules, []
        for _, mod, name, _ in _PARAMS:
            m = layer if mod is None else mods.get(mod)
            out.append(None if m is None else m._parameters.get(name))
        return out

    def holds(self, layer):
        """0: something has changed; 1: nothing has; 2: nothing has, and a submodule has a hook or a forward of its own."""
        return _capi.step_core().holds(self.core, layer) if self.plain else 0


def watch(layer):
    """The layer's _Watch, made anew when a weight, a submodule or an option has changed; None when a submodule or a weight is not a
    plain one, when something is hooked, or under forward-mode differentiation (whose tangents only the general path's products carry)."""
    if torch.autograd.forward_ad._current_level >= 0:
        return None
    w = _watches.get(layer)
    state = 0 if w is None else w.holds(layer)
    if state == 0:
        w = _watches[layer] = _Watch(layer)
        state = w.holds(layer)
    return w if state == 1 and not _has_any_global_hook() else None


class _Plan:
    """What stays the same from step to step: the weights' addresses, the geometry and the mode."""

    def __init__(self, layer, kind, seen):
        self.built = False
        params = seen.weights(layer)
        s = self.fixed = LayerStep()
        by, shapes = dict(zip((p[0] for p in _PARAMS), params)), weight_shapes(layer)
        delta = kind == 'gdn'
        K, V, H, HQ = layer.head_k_dim, layer.head_v_dim, layer.num_heads, layer.num_attn_heads
        for n, t in by.items():
            if t is None:
                if n not in _OPTIONAL or (n == "wb" and delta) or (n in ("norm_q", "norm_k") and layer.attn_qk_norm):
                    return
                continue
            if not (t.is_cuda and t.is_contiguous() and t.device == params[0].device and t.shape == shapes[n] and
                    (t.dtype == torch.bfloat16 or (n in _EITHER_DTYPE and t.dtype == torch.float32))):
                return
            setattr(s, n, t.data_ptr())
        same = lambda a, b: by[a] is None or by[a].dtype == by[b].dtype
        if not (same("norm_q", "norm_k") and same("a_log", "dt_bias") and same("out_norm1", "out_norm2")):
            return
        if not layer.use_short_conv or layer.num_v_heads != H or layer.ops_for_incomplete_chunks == 'attn':
            return
        convs = [layer.q_conv1d, layer.k_conv1d, layer.v_conv1d]
        W, act = layer.conv_size, convs[0].activation
        if any(c.kernel_size[0] != W or (c.activation is None) != (act is None) for c in convs) or W not in (2, 3, 4):
            return
        if any(layer._modules[m].bias is not None for m in ("q_proj", "k_proj", "v_proj", "g_proj", "a_proj", "nats_out_weights_layer", "o_proj")) \
                or (delta and layer._modules["b_proj"].bias is not None):
            return
        D, KA, VA = layer.hidden_size, layer.head_attn_k_dim, layer.head_attn_v_dim
        if K not in (64, 128, 192) or KA not in (64, 128) or VA not in (64, 128) or K % KA or HQ % H or HQ % layer.num_nats_head or \
                H % layer.num_nats_head or V % 16 or D % 32 or (H * V) % 32 or layer.nats_block_size % 64:
            return
        code = lambda n: _capi.dtype_code(by[n].dtype) if by[n] is not None else _capi.BF16
        s.D, s.H, s.K, s.V, s.HQ, s.HN, s.block, s.conv_width, s.is_delta = D, H, K, V, HQ, layer.num_nats_head, layer.nats_block_size, W, int(delta)
        s.norm_dtype, s.gate_dtype, s.out_norm_dtype = code("norm_q"), code("a_log"), code("out_norm1")
        if by["norm_q"] is not None:
            if layer.q_norm.eps != layer.k_norm.eps:
                return
            s.norm_eps = layer.q_norm.eps
        s.scale_attn, s.out_norm_eps = KA ** -0.5, layer.o_norm.eps
        flags = (SILU if act is not None else 0) | (ATTN_FROM_CONV if layer.attn_with_short_conv else 0) | \
                (ATTN_NORM if layer.attn_qk_norm else 0) | (ATTN_OWN_BLOCK if layer.ops_for_incomplete_chunks == 'all' else 0)
        if delta:
            flags |= (DECAY if layer.decay_for_non_gdn_blocks else 0) | (NEG_EIGVAL if layer.allow_neg_eigval else 0)
            s.scale_linear = K ** -0.5
        else:
            flags |= (DECAY if layer.decay_for_non_mamba_blocks else 0) | L2_ROWS
            s.scale_linear = 1.0
            if layer.q_norm2.eps != layer.k_norm2.eps:
                return
            s.l2_eps = layer.q_norm2.eps
        s.flags = flags
        self.device = params[0].device
        L = _capi.lib()
        address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
        self.core = _capi.step_core().make_step(ctypes.addressof(s), ctypes.sizeof(s), address(L.natsl_layer_step_sync_fwd),
                                                address(L.natsl_layer_step_workspace_bytes), address(L.natsl_layer_step_sync_bytes), MAX_WAIT_US,
                                                self.device.index)
        self.built = True


def layer_step(layer, kind, x, cache):
    """The layer's output [B,T,D] for new tokens x on `cache` (NAtSLayerCache), which is brought up to date; None when the general
    path has to run.  Called with the cache as it is before the step and only for steps that stay inside the block."""
    B, T, D = x.shape
    if B * T > MAX_ROWS or T < 1 or x.dtype != torch.bfloat16 or torch.is_grad_enabled() and _wants_grad(layer, x) or torch.is_autocast_enabled():
        return None
    seen = watch(layer)
    if seen is None:
        return None
    plan = seen.step_plan
    if plan is None:
        plan = seen.step_plan = _Plan(layer, kind, seen)
    if not plan.built:
        return None
    bs, n_in, start = cache.nats_block_size, cache._n_tokens_in_nats_block, cache.recurrent_state_block_start
    f, core = plan.fixed, _capi.step_core()
    if (bs != f.block or n_in + T > bs or x.device != plan.device or cache.n_attn_blocks is None or cache.attn_k is None or
            (cache._linear_only == bool(f.flags & ATTN_OWN_BLOCK)) or cache.op_for_incomplete_chunk == 'attn'):
        return None
    completes = n_in + T == bs
    full = cache.attn_k.shape[1] < cache.n_attn_tokens_max + T
    tensors = lambda: (cache.conv_state, cache.recurrent_state, cache.l_attn_k, cache.l_attn_v, cache.lattn_g, cache.block_type_state,
                       cache.lattn_beta, cache.attn_k, cache.attn_v, cache.valid_attn_tokens, start, cache.g_cumsum)
    types = None
    if completes or full:
        if not core.takes(plan.core, B, *tensors()):       # (before anything of the cache changes)
            return None
        if completes:
            types, _, _ = layer.select_ops(cache.update_attn_types(input_hidden_states=x), None, force_last_block=False)
            if types.shape != (B, 1, f.HN, 2) or types.device != x.device:
                raise ValueError(f"select_ops must give types {(B, 1, f.HN, 2)} on {x.device}, got {tuple(types.shape)} on {types.device}")
            types = (types if types.dtype in (torch.bfloat16, torch.float32) else types.float()).contiguous()
        if full:
            cache._grow(cache.n_attn_tokens_max + T)
    done = core.run(plan.core, x, n_in, cache.n_attn_blocks_max, _capi.stream_ptr(x.device), types,
                    0 if types is None else _capi.dtype_code(types.dtype), *tensors(), getattr(cache, 'step_shared', None))
    if type(done) is not tuple:
        if done is None:                                   # (the cache's tensors are not what the kernels address)
            return None
        _capi.check(done, "natsl_layer_step_sync_fwd")
    out, state_out, start, new_conv, g_out, cache.step_shared = done
    if types is None:
        cache.note_step(state_out, start, new_conv, g_out, T)
    else:
        cache.update(recurrent_state=state_out, recurrent_state_block_start=start, attn_state=(cache.attn_k, cache.attn_v), conv_state=new_conv,
                     nats_block_types=types, g=cache.lattn_g, n_new_tokens=T)
    attrs = layer.__dict__
    attrs['last_recurrent_state'], attrs['last_block_start_state'] = state_out, start
    return out


def _wants_grad(layer, x):
    return x.requires_grad or any(p.requires_grad for p in layer.parameters())
