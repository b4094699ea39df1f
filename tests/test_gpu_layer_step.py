"""The layers' generation step as one native call (natsl_layer_step_fwd) against the layers' general decode path (separate torch
operations and operator calls), which the other tests pin to the oracle."""
import pytest
import torch

from tests._util import rel_l2
from tests.test_gpu_layers import PUBLISHED

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _layer(kind, geometry, ops, **more):
    from neuralattentionsearchlinear_amd.natsl_attn_gdn import NeuralAttentionSearchLinearAttnGDN as G
    from neuralattentionsearchlinear_amd.natsl_attn_mamba2 import NeuralAttentionSearchLinearAttnMamba as M
    torch.manual_seed(3)
    if kind == 'gdn':
        cfg = dict(hidden_size=256, expand_v=2, head_dim=128, num_heads=2, num_attn_heads=4, ops_for_incomplete_chunks=ops, layer_idx=0)
        cfg.update(PUBLISHED[geometry] if geometry else {})
        layer = G(**dict(cfg, **more))
    else:
        layer = M(**dict(dict(hidden_size=256, expand_v=0.5, head_dim=128, num_heads=4, num_attn_heads=4, ops_for_incomplete_chunks=ops,
                              layer_idx=0), **more))
    return layer.to(DEV).to(torch.bfloat16).eval()


def _generate(layer, kind, x, T0, sizes):
    from neuralattentionsearchlinear_amd.cache import NAtSCache, NAtSMamba2Cache
    holder = NAtSCache() if kind == 'gdn' else NAtSMamba2Cache()
    kw = dict(past_key_values=holder, use_cache=True) if kind == 'gdn' else dict(cache_params=holder, use_cache=True)
    outs, t = [], 0
    with torch.no_grad():
        for n in [T0] + list(sizes):
            o = layer(x[:, t:t + n], **kw)
            outs.append(o[0] if isinstance(o, tuple) else o)
            t += n
    return outs, (holder[0] if kind == 'gdn' else holder.nats_cache[0])


@pytest.mark.parametrize("kind,geometry,ops,B,T0,sizes,more", [
    ('gdn', None, 'all', 1, 100, (1, 1, 5, 1), {}),                       # one row; several tokens at once
    ('gdn', '340M', 'all', 3, 321, (1, 20, 1), {}),                       # 20 x 3 rows: four row tiles
    ('gdn', '760M', 'all', 2, 130, (1, 2), dict(allow_neg_eigval=True, conv_bias=True)),
    ('gdn', None, 'all', 17, 70, (1, 3, 1), {}),                          # two row tiles, one of them with one row
    ('gdn', None, 'all', 64, 65, (1,), {}),                               # the most rows it takes
    ('gdn', None, 'all', 1, 128, (1, 63, 1), {}),                         # a block's first token, and a step that completes it (64 rows at most)
    ('gdn', None, 'gated_delta_net', 2, 100, (1, 3), {}),                 # the softmax operator skips the incomplete block
    ('gdn', None, 'all', 2, 200, (1, 1), dict(attn_with_short_conv=False, attn_qk_norm=False, conv_size=3, conv_activation=None)),
    ('mamba', None, 'all', 2, 257, (1, 4), {}),
    ('mamba', None, 'mamba', 5, 190, (1, 1, 1), dict(attn_qk_norm=True, conv_size=2)),
])
def test_layer_step_matches_the_general_path(kind, geometry, ops, B, T0, sizes, more, monkeypatch):
    import neuralattentionsearchlinear_amd._layer_step as LS
    from neuralattentionsearchlinear_amd import natsl_attn_gdn, natsl_attn_mamba2
    layer = _layer(kind, geometry, ops, **more)
    torch.manual_seed(T0)
    x = torch.randn(B, T0 + sum(sizes), layer.hidden_size, device=DEV).bfloat16()
    taken = []
    for mod in (natsl_attn_gdn, natsl_attn_mamba2):
        monkeypatch.setattr(mod, 'layer_step', lambda *a: taken.append(LS.layer_step(*a)) or taken[-1])
    fast, cf = _generate(layer, kind, x, T0, sizes)
    assert len(taken) == len(sizes) and all(t is not None for t in taken), "the native step declined"
    for mod in (natsl_attn_gdn, natsl_attn_mamba2):
        monkeypatch.setattr(mod, 'layer_step', lambda *a: None)
    slow, cs = _generate(layer, kind, x, T0, sizes)
    # both round to bf16 at the same places; a value that falls on a rounding edge moves by one ulp (2^-8) there, and such
    # differences pass through two more products: 5e-3 in the norm, the bound the operators are held to
    for i, (a, b) in enumerate(zip(fast, slow)):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert rel_l2(a.float(), b.float()) <= 5e-3, f"step {i}: rel-L2 {rel_l2(a.float(), b.float()):.3e}"
    assert (cf._n_tokens_in_nats_block, cf.n_attn_blocks_max, cf.n_attn_tokens_max, cf.n_observed_tokens) == \
        (cs._n_tokens_in_nats_block, cs.n_attn_blocks_max, cs.n_attn_tokens_max, cs.n_observed_tokens)
    assert torch.equal(cf.n_attn_blocks, cs.n_attn_blocks) and torch.equal(cf.valid_attn_tokens, cs.valid_attn_tokens)
    n_in, start = cf._n_tokens_in_nats_block, cf.n_attn_blocks_max * cf.nats_block_size
    pairs = [(cf.attn_k[:, start:start + n_in], cs.attn_k[:, start:start + n_in]), (cf.attn_v[:, start:start + n_in], cs.attn_v[:, start:start + n_in]),
             (cf.recurrent_state, cs.recurrent_state), (cf.g_cumsum, cs.g_cumsum), (cf.l_attn_v[:, :n_in], cs.l_attn_v[:, :n_in]),
             (cf.l_attn_k[:, :n_in], cs.l_attn_k[:, :n_in]), (cf.lattn_g[:, :n_in], cs.lattn_g[:, :n_in]),
             (cf.block_type_state[:, :n_in], cs.block_type_state[:, :n_in])] + list(zip(cf.conv_state, cs.conv_state))
    if kind == 'gdn':
        pairs.append((cf.lattn_beta[:, :n_in], cs.lattn_beta[:, :n_in]))
    if cs.recurrent_state_block_start is not None:
        pairs.append((cf.recurrent_state_block_start, cs.recurrent_state_block_start))
    for i, (a, b) in enumerate(pairs):
        assert a.shape == b.shape and rel_l2(a.float(), b.float()) <= 5e-3, f"cache tensor {i}: rel-L2 {rel_l2(a.float(), b.float()):.3e}"


@pytest.mark.parametrize("kind,B,T0,n,more", [
    ('gdn', 1, 64, 3, {}),                                                # the first rows of a chunk
    ('gdn', 2, 94, 4, dict(head_dim=64, num_heads=3, num_attn_heads=3)),  # over a chunk of keys; 192 channels of q in one chunk of 256; 3 heads
    ('gdn', 1, 126, 4, dict(head_dim=64, num_heads=5, num_attn_heads=5)), # over a block and a split; 320 channels, 5 heads on 4 waves
    ('gdn', 3, 253, 5, dict(head_dim=192, num_heads=1, num_attn_heads=3)),
    ('gdn', 1, 2110, 2, dict(num_attn_heads=2, expand_v=1)),                          # 16 splits
    ('mamba', 2, 95, 3, dict(head_dim=64, expand_v=1, num_heads=18, num_attn_heads=18)),   # more heads than a wave's four rounds of four
    ('mamba', 1, 127, 2, dict(expand_v=1)),
    ('mamba', 1, 257, 2, dict(attn_with_short_conv=False, conv_bias=True)),
    ('mamba', 16, 2100, 2, dict(num_heads=16, num_attn_heads=16)),                    # more workgroups than fit at once: three splits
    ('gdn', 16, 3000, 2, dict(num_heads=6, num_attn_heads=12)),
    ('gdn', 8, 1300, 2, dict(num_heads=6, num_attn_heads=12)),                        # all of them fit: four splits
    ('gdn', 30, 1200, 1, dict(num_heads=6, num_attn_heads=12)),                       # 128-wide values, too many: the several launches
])
def test_layer_step_of_one_token(kind, B, T0, n, more, monkeypatch):
    """The launch that does everything between the products of a one-token step, at the edges of its chunks, splits and heads."""
    test_layer_step_matches_the_general_path(kind, None, 'all', B, T0, (1,) * n, more, monkeypatch)


@pytest.mark.parametrize("kind,more", [('gdn', {}), ('gdn', dict(conv_bias=True)), ('mamba', dict(expand_v=1))])
def test_layer_step_of_one_token_with_float_parameters(kind, more, monkeypatch):
    """The small parameters in fp32, with values that bf16 does not hold: the one-token launch reads either type without a branch."""
    layer_of = _layer

    def with_floats(*a, **kw):
        layer = layer_of(*a, **kw)
        names = [n for n, q in layer.named_parameters() if n in ('A_log', 'dt_bias') or 'norm.weight' in n]
        assert len(names) >= 4, names
        for n, q in layer.named_parameters():
            if n in names:
                q.data = q.data.float() * 1.003
        return layer
    monkeypatch.setitem(globals(), '_layer', with_floats)
    test_layer_step_matches_the_general_path(kind, None, 'all', 2, 130, (1,) * 3, more, monkeypatch)


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
@pytest.mark.parametrize("float_gates", [False, True])
def test_layer_step_forms_the_general_paths_gates(kind, float_gates, monkeypatch):
    """g (kept in fp32 and summed up) and beta of a step are those of the general path and of a prefill, bit for bit: the projections
    that feed them pick single inputs, so that nothing before the gates rounds."""
    from neuralattentionsearchlinear_amd import natsl_attn_gdn, natsl_attn_mamba2
    layer = _layer(kind, None, 'all')
    torch.manual_seed(5)
    with torch.no_grad():
        for i, name in enumerate(("a_proj", "b_proj")):
            if hasattr(layer, name):
                w = getattr(layer, name).weight
                w.zero_()[torch.arange(w.shape[0]), 10 * i + torch.arange(w.shape[0])] = 4.0
        layer.dt_bias.copy_(torch.randn_like(layer.dt_bias))
        if float_gates:
            layer.A_log.data, layer.dt_bias.data = layer.A_log.data.float() * 1.003, layer.dt_bias.data.float() * 1.003
    sizes = (4,) * 15
    x = torch.randn(16, 64 + sum(sizes), layer.hidden_size, device=DEV).bfloat16()
    _, cf = _generate(layer, kind, x, 64, sizes)
    for mod in (natsl_attn_gdn, natsl_attn_mamba2):
        monkeypatch.setattr(mod, 'layer_step', lambda *a: None)
    _, cs = _generate(layer, kind, x, 64, sizes)
    n = cf._n_tokens_in_nats_block
    assert n == sum(sizes) == cs._n_tokens_in_nats_block
    assert torch.equal(cf.lattn_g[:, :n], cs.lattn_g[:, :n])
    # the same tokens as the incomplete end of one prompt
    _, cp = _generate(layer, kind, x, x.shape[1], ())
    assert torch.equal(cf.lattn_g[:, :n], cp.lattn_g[:, :n])
    if kind == 'gdn':
        assert torch.equal(cf.lattn_beta[:, :n], cs.lattn_beta[:, :n]) and torch.equal(cf.lattn_beta[:, :n], cp.lattn_beta[:, :n])


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
def test_layer_step_after_a_prefill_under_autocast(kind, monkeypatch):
    """fp32 hidden states under autocast leave a cache whose collected hidden states are fp32: bf16 steps on it fill it as the general
    path does."""
    from neuralattentionsearchlinear_amd import natsl_attn_gdn, natsl_attn_mamba2
    layer = _layer(kind, None, 'all')
    torch.manual_seed(6)
    x = torch.randn(2, 75, layer.hidden_size, device=DEV)

    def run():
        from neuralattentionsearchlinear_amd.cache import NAtSCache, NAtSMamba2Cache
        holder = NAtSCache() if kind == 'gdn' else NAtSMamba2Cache()
        kw = dict(past_key_values=holder, use_cache=True) if kind == 'gdn' else dict(cache_params=holder, use_cache=True)
        with torch.no_grad():
            with torch.autocast('cuda', dtype=torch.bfloat16):
                layer(x[:, :70], **kw)
            outs = [layer(x[:, t:t + 1].bfloat16(), **kw) for t in range(70, 75)]
        return [o[0] if isinstance(o, tuple) else o for o in outs], holder[0] if kind == 'gdn' else holder.nats_cache[0]
    fast, cf = run()
    for mod in (natsl_attn_gdn, natsl_attn_mamba2):
        monkeypatch.setattr(mod, 'layer_step', lambda *a: None)
    slow, cs = run()
    assert cf.block_type_state.dtype == cs.block_type_state.dtype
    n = cs._n_tokens_in_nats_block
    assert n == 75 % layer.nats_block_size and torch.equal(cf.block_type_state[:, :n], cs.block_type_state[:, :n])
    for a, b in zip(fast, slow):
        assert rel_l2(a.float(), b.float()) <= 5e-3


@pytest.mark.parametrize("name,change", [
    ('block_type_state', 'float'), ('l_attn_k', 'float'), ('l_attn_v', 'float'), ('attn_v', 'float'), ('attn_k', 'half'), ('lattn_g', 'bfloat16'),
    ('lattn_beta', 'float'), ('recurrent_state', 'bfloat16'), ('recurrent_state_block_start', 'bfloat16'), ('valid_attn_tokens', 'int'),
    ('l_attn_k', 'short'), ('lattn_g', 'short'), ('attn_v', 'short'), ('valid_attn_tokens', 'short'), ('recurrent_state', 'strided'), ('attn_k', 'strided'),
    ('g_cumsum', 'short'), ('conv_state', 'short')])
def test_layer_step_declines_other_cache_tensors(name, change):
    """A cache tensor of another type, shape or layout than the kernels address sends the step down the general path."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    layer = _layer('gdn', None, 'all')
    torch.manual_seed(7)
    x = torch.randn(2, 102, 256, device=DEV).bfloat16()
    with torch.no_grad():
        _, cache = _generate(layer, 'gdn', x[:, :101], 100, (1,))
        t = getattr(cache, name)
        if change == 'short':
            t = tuple(c[..., :2].contiguous() for c in t) if isinstance(t, tuple) else t[:, :-1].contiguous()
        elif change == 'strided':
            t = t.transpose(-1, -2).contiguous().transpose(-1, -2)
        else:
            t = getattr(t, change)()
        own = getattr(cache, name)
        setattr(cache, name, t)
        assert LS.layer_step(layer, 'gdn', x[:, 101:], cache) is None
        setattr(cache, name, own)
        assert LS.layer_step(layer, 'gdn', x[:, 101:], cache) is not None


def test_layer_step_follows_replaced_weights_and_declines_hooks():
    """The step reads the layer's current parameters, and a hooked submodule sends the layer down the general path."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    layer = _layer('gdn', None, 'all')
    torch.manual_seed(1)
    x = torch.randn(2, 102, 256, device=DEV).bfloat16()
    _, cache = _generate(layer, 'gdn', x[:, :100], 100, ())
    calls = []
    with torch.no_grad():
        handle = layer.v_proj.register_forward_hook(lambda *a: calls.append(1))
        assert LS.layer_step(layer, 'gdn', x[:, 100:101], cache) is None
        handle.remove()
        assert LS.layer_step(layer, 'gdn', x[:, 100:101], cache) is not None
        layer.o_proj.weight = torch.nn.Parameter(torch.zeros_like(layer.o_proj.weight))
        out = LS.layer_step(layer, 'gdn', x[:, 101:102], cache)
    assert float(out.abs().max()) == 0.0


@pytest.mark.parametrize("where,shape", [('o_proj.weight', (128, 512)), ('v_proj.weight', (256, 512)), ('A_log', (1,)), ('dt_bias', (1,)),
                                         ('o_norm.weight1', (64,)), ('k_conv1d.weight', (256, 1, 3)), ('q_norm.weight', (1,)),
                                         ('nats_out_weights_layer.weight', (256, 8))])
def test_layer_step_and_front_decline_other_weight_shapes(where, shape):
    """A weight of another shape than the layer's options say is left to the submodules: the kernels would address the options' shape."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    from neuralattentionsearchlinear_amd._front import fast_front
    layer = _layer('gdn', None, 'all')
    torch.manual_seed(8)
    x = torch.randn(2, 102, 256, device=DEV).bfloat16()
    with torch.no_grad():
        _, cache = _generate(layer, 'gdn', x[:, :100], 100, ())
        assert fast_front(layer, 'gdn', x, None, None) is not None
        assert LS.layer_step(layer, 'gdn', x[:, 100:101], cache) is not None
        p = layer.get_parameter(where)
        assert p.shape != shape
        p.data = torch.zeros(shape, dtype=p.dtype, device=DEV)
        assert LS.layer_step(layer, 'gdn', x[:, 101:], cache) is None
        assert fast_front(layer, 'gdn', x, None, None) is None
