"""CPU-only: the C-ABI library builds, loads, and exports every function include/natsl.h declares;
argument validation runs on the host before any launch."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "natsl.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(natsl_[a-z_0-9]+)\s*\(", text)))


def _lib():
    from neuralattentionsearchlinear_amd import _capi
    if not os.path.exists(_capi.LIB_PATH):
        from neuralattentionsearchlinear_amd import _build
        _build.build()
    return _capi.lib()


def test_header_symbols_are_exported():
    names = _declared()
    assert len(names) >= 10
    L = _lib()
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    from neuralattentionsearchlinear_amd import _capi
    assert sorted(_capi.exported_symbols()) == names          # the ctypes table covers the whole header
    assert L.natsl_version() >= 100


def test_argument_validation_needs_no_gpu():
    L = _lib()
    # null pointers / bad shapes are rejected on the host, before any launch
    assert L.natsl_hard_select(None, None, None, 1, 4, 2, 1, 0, None, 0, 0, None) == -1
    assert b"null" in L.natsl_last_error()
    assert L.natsl_route(ctypes.c_void_p(16), 1, 1, 4, 2, 256, 32, None, None, None, None, None, None, None, 0, 0, None) == -2
    assert b"multiple of 64" in L.natsl_last_error()
    assert L.natsl_linear_workspace_bytes(16384, 16) == 16384 * 16 * (2 * 64 * 64 * 2 + 4 * 64 * 4)
    p = ctypes.c_void_p(256)
    rc = L.natsl_softmax_sparse_fwd(p, p, p, p, p, p, 1, p, p, 1, 256, 4, 4, 4, 96, 96, 4, 64, 0.1, 1, 1, None, 0, 0, None)
    assert rc == -2 and b"head dims" in L.natsl_last_error()
    rc = L.natsl_gdn_chunk_fwd(p, p, p, p, p, None, p, None, None, None, None, None, p, 1, 1, 256, 4, 4, 128, 128, 4, 64, 0.1, 7, p, 16, 1,
                               None, 0, 0, None)
    assert rc == -3 and b"workspace" in L.natsl_last_error()
    # the softmax backward's 32-bit row offsets: T * HQ * max(K, V) * 2 bytes must stay below 2^32 -- refused on the host,
    # before any kernel is launched (T = 2^20 tokens x 32 heads x 128 x 2 bytes = 2^33)
    rc = L.natsl_softmax_sparse_bwd(p, p, p, p, p, p, p, p, p, p, p, 1, p, p, 1, 1 << 20, 32, 32, 32, 128, 128, 1 << 14, 64, 0.1, 1, 1,
                                    p, ctypes.c_size_t(1 << 40), None, 0, 0, 0, None)
    assert rc == -2 and b"32-bit" in L.natsl_last_error()


def test_workspaces_stay_small():
    """Partial sums are bounded by the chip and not by the tokens: a row of 2 H sums for each of 2048 workgroups of the gates' backward; for a
    weight's gradient its own rows, in blocks of 32, for each of 128 slices."""
    L = _lib()
    for rows in (1, 4096, 32768, 1 << 20, 1 << 24):
        for H in (1, 6, 16, 33, 64, 256):
            assert 0 < L.natsl_gates_bwd_workspace_bytes(rows, H) <= 2048 * 2 * H * 4
    from neuralattentionsearchlinear_amd._front import _WgradSeg
    up = lambda n, to: -(-n // to) * to
    for rows, ns, D in ((32768, (24,), 768), (1 << 20, (8, 40), 256), (16000, (32,), 2048), (6000, (40,), 1152), (40, (8,), 8), (32768, (768, 1536, 200), 1000)):
        segs = (_WgradSeg * len(ns))(*[_WgradSeg(None, None, n, n) for n in ns])
        assert 0 < L.natsl_wgrad_workspace_bytes(segs, len(ns), rows, D) <= 128 * sum(up(n, 32) for n in ns) * up(D, 256) * 4


def test_no_cpu_fallback():
    import torch
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    x = torch.zeros(1, 64, 1, 64, dtype=torch.bfloat16)
    g = torch.zeros(1, 64, 1)
    ty = torch.ones(1, 1, 1, 2)
    with pytest.raises(_capi.NatslError):
        nats_mixed_attn_gdn(x, x, x, x, x, x, None, g, g.bfloat16(), ty, None)


def test_product_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "neuralattentionsearchlinear_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in src.replace("no CPU fallback", ""), f"{f} mentions the oracle"


def test_backward_entry_rejects_what_is_not_built():
    """Argument errors come back as codes from the host, before any launch."""
    import ctypes
    from neuralattentionsearchlinear_amd import _capi
    L = _capi.lib()
    p = ctypes.c_void_p(256)
    args = lambda K, V, block: (1, p, p, p, p, p, p, None, p, p, 1, p, p, p, p, p, p, p, p, p, None, p, p, 1, 256, 4, 4, K, V, 256 // block, block,
                                0.1, 7, 1, None, 0, 0, None)
    assert L.natsl_linear_chunk_bwd(*args(96, 64, 64)) == -2 and b"K=96" in L.natsl_last_error()
    assert L.natsl_linear_chunk_bwd(*args(128, 48, 64)) == -2 and b"V=48" in L.natsl_last_error()
    # both forms read the forward's workspace (the Mamba form its scale vectors)
    for delta_rule in (1, 0):
        a = list(args(128, 64, 64))
        a[0], a[12] = delta_rule, None
        assert L.natsl_linear_chunk_bwd(*a) == -1 and b"null pointer" in L.natsl_last_error()


def test_invalid_block_gradient_is_refused_for_blocks_of_several_chunks():
    """The linear branch's selector gradient for blocks NOT typed linear is built for one chunk per block only: a
    larger block with the flag set raises before anything is launched."""
    import torch
    from neuralattentionsearchlinear_amd._linear_bwd import linear_chunk_backward
    q = torch.zeros(1, 128, 2, 64, dtype=torch.bfloat16)
    ty = torch.zeros(1, 1, 2, 2, dtype=torch.bfloat16)
    with pytest.raises(NotImplementedError, match="nats_block_size == 64"):
        linear_chunk_backward('gdn', q, q, q, torch.zeros(1, 128, 2), torch.zeros(1, 128, 2, dtype=torch.bfloat16), None, ty, 1.0, 128,
                              True, True, True, q, None, True)


def test_chunk_state_saving_follows_the_byte_budget():
    """_mixed_common.SAVE_CHUNK_STATES = None keeps the linear branch's chunk states for the backward only while they fit
    SAVE_CHUNK_STATES_MAX_BYTES; True / False force it."""
    import torch
    import neuralattentionsearchlinear_amd._mixed_common as MC
    small = torch.empty(1, 512, 4, 128, device='meta')
    big = torch.empty(8, 8192, 16, 128, device='meta')
    old = MC.SAVE_CHUNK_STATES
    try:
        MC.SAVE_CHUNK_STATES = None
        assert MC._keep_chunk_states(small, small, None) and not MC._keep_chunk_states(big, big, None)
        # by default a layer's training step holds no more than 64 MiB per call that the backward could compute again: 340M geometry, 8 x 4096
        assert not MC._keep_chunk_states(torch.empty(8, 4096, 6, 128, device='meta'), torch.empty(8, 4096, 6, 256, device='meta'), None)
        assert MC.SAVE_CHUNK_STATES_MAX_BYTES == 64 << 20
        MC.SAVE_CHUNK_STATES = True
        assert MC._keep_chunk_states(big, big, None)
        MC.SAVE_CHUNK_STATES = False
        assert not MC._keep_chunk_states(small, small, None)
    finally:
        MC.SAVE_CHUNK_STATES = old


def test_layer_plans_notice_every_change():
    """What the layers' fused paths remember about a layer is dropped when a weight, an option or a hook changes."""
    import torch
    from neuralattentionsearchlinear_amd._layer_step import watch
    from neuralattentionsearchlinear_amd.natsl_attn_gdn import NeuralAttentionSearchLinearAttnGDN
    layer = NeuralAttentionSearchLinearAttnGDN(hidden_size=64, expand_v=2, head_dim=64, num_heads=2, num_attn_heads=2, layer_idx=0)
    seen = watch(layer)
    assert seen is not None and watch(layer) is seen

    def new_after(change):
        nonlocal seen
        change()
        before, seen = seen, watch(layer)
        return seen is not before

    w = layer.q_conv1d.weight
    assert new_after(lambda: setattr(w, 'data', w.data.clone()))                       # another address
    assert new_after(lambda: setattr(w, 'data', w.data.view(torch.complex64)))         # the same memory as another type
    assert new_after(lambda: setattr(w, 'data', w.data.view(torch.float32)))
    q = layer.nats_out_weights_layer.weight
    assert new_after(lambda: setattr(q, 'data', q.data.t().contiguous().t()))          # another layout
    assert new_after(lambda: setattr(layer, 'decay_for_non_gdn_blocks', not layer.decay_for_non_gdn_blocks))
    assert new_after(lambda: setattr(layer.o_norm, 'eps', 1e-3))
    assert new_after(lambda: setattr(layer.b_proj, 'bias', torch.nn.Parameter(torch.zeros(2))))
    handle = layer.q_proj.register_full_backward_hook(lambda *a: None)
    assert watch(layer) is None
    handle.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert watch(layer) is None
    handle.remove()
    assert watch(layer) is seen


def test_layer_plans_keep_nothing_alive():
    """What is remembered about a layer frees a replaced weight or submodule at once."""
    import gc
    import weakref
    import torch
    from neuralattentionsearchlinear_amd._layer_step import watch
    from neuralattentionsearchlinear_amd.natsl_attn_mamba2 import NeuralAttentionSearchLinearAttnMamba
    layer = NeuralAttentionSearchLinearAttnMamba(hidden_size=64, expand_v=1, head_dim=64, num_heads=2, num_attn_heads=2, layer_idx=0)
    seen = watch(layer)
    old = [weakref.ref(t) for t in (layer.A_log, layer.q_proj.weight, layer.o_proj, layer.o_proj.weight, layer.k_conv1d.weight)]
    layer.A_log = torch.nn.Parameter(layer.A_log.detach().clone())
    layer.q_proj.weight = torch.nn.Parameter(layer.q_proj.weight.detach().clone())
    layer.k_conv1d.weight = torch.nn.Parameter(layer.k_conv1d.weight.detach().clone())
    layer.o_proj = torch.nn.Linear(128, 64, bias=False)
    gc.collect()
    assert not any(r() is not None for r in old)
    again = watch(layer)
    assert again is not seen and again is not None and watch(layer) is again


def test_which_way_a_narrow_product_goes():
    """The rules that every caller takes (natsl_narrow_*_pays, natsl_project_bwd_takes) at their edges, and that none takes what its kernel refuses."""
    from neuralattentionsearchlinear_amd._front import _ProjectSeg
    L = _lib()
    fwd, bwd, wgrad = L.natsl_narrow_fwd_pays, L.natsl_narrow_linear_bwd_pays, L.natsl_narrow_wgrad_pays
    assert fwd(1 << 20, 768, 32) and not fwd(4097, 768, 34) and fwd(4096, 768, 64) and not fwd(64, 768, 66) and not fwd(64, 760, 24) and not fwd(64, 768, 23)
    assert not fwd(0, 768, 24) and not fwd(1 << 31, 768, 24)
    assert bwd(6000, 768, 24, 0) and not bwd(2048, 768, 24, 0) and bwd(1, 768, 24, 1) and bwd(1, 128, 32, 1) and not bwd(1, 128, 52, 1) and not bwd(1, 96, 24, 1)
    assert not bwd(0, 768, 24, 1) and not bwd(6000, 768, 22, 1)
    assert wgrad(2048, 1536, 12, 1, 0) == 1 and wgrad(2049, 1536, 12, 1, 0) == 0 and wgrad(64, 1535, 12, 1, 0) == 0 and wgrad(64, 1536, 65, 1, 1) == 0
    assert wgrad(32768, 1152, 36, 0, 0) == 2 and wgrad(32768, 768, 24, 0, 0) == 0 and wgrad(32768, 768, 24, 0, 1) == 2 and wgrad(6000, 2048, 64, 0, 1) == 0
    assert wgrad(1 << 15, 1024, 24, 0, 1) == 2 and wgrad((1 << 15) + 1, 1024, 24, 0, 1) == 0 and wgrad(1 << 31, 64, 12, 0, 1) == 0
    segs = lambda *ns, y=1 << 20: (_ProjectSeg * len(ns))(*[_ProjectSeg(y, 1 << 20, n, n) for n in ns])
    takes = lambda s, dpool=1 << 20, dx=1 << 20: L.natsl_project_bwd_takes(s, len(s), dpool, dx)
    assert takes(segs(768, 32)) and takes(segs(64, 64), None) and not takes(segs(64, 32)) and not takes(segs(768, 16)) and not takes(segs(768, y=(1 << 20) + 8))
    assert not takes(segs(768), (1 << 20) + 2) and not takes(segs(768), None, 8) and not takes(segs(*[768] * 9)) and not L.natsl_project_bwd_takes(None, 0, None, None)
