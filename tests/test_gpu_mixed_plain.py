"""The mixed operators' forward as one native call with its host side (csrc/host/mixed_core.cpp) against the general host path, bit for bit over the forms
of input it takes; what it does not take goes the general way and ends as it did there."""
import pytest
import torch

from tests._util import make_gates, make_qkv, make_types

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _call(kind, a):
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    from neuralattentionsearchlinear_amd.mixed_attn_mamba import nats_mixed_attn_mamba
    qkv = (a['qa'], a['ka'], a['va'], a['q'], a['k'], a['v'], a['h0'], a['g'])
    kw = dict(nats_block_size=a['block'], ops_for_incomplete_chunks=a['ops'])
    if kind == 'gdn':
        return nats_mixed_attn_gdn(*qkv, a['beta'], a['types'], None, output_final_state_gated_delta=a['state'], decay_for_non_gdn_blocks=a['decay'],
                                   lattn_use_qk_l2norm_in_kernel=a['l2'], **kw)
    return nats_mixed_attn_mamba(*qkv, a['types'], None, output_final_state_mamba=a['state'], decay_for_non_mamba_blocks=a['decay'], **kw)


def _args(kind, B=2, T=130, H=2, K=64, V=64, block=64, dtype=torch.bfloat16, seed=3):
    q, k, v = make_qkv(B, T, H, K, V, seed, torch.float32)
    g, beta = make_gates(B, T, H, seed + 1, torch.float32)
    types = make_types(B, -(-T // block), H, 0.4, seed + 2)
    q, k, v, beta, types = (t.to(DEV).to(dtype) for t in (q, k, v, beta, types))
    return dict(qa=q, ka=k, va=v, q=q, k=k, v=v, h0=None, g=g.to(DEV), beta=beta if kind == 'gdn' else None, types=types, block=block, ops='all', state=True,
                decay=True, l2=True)


def _strided(t):                                           # the same numbers, every second element of a wider tensor
    wide = torch.zeros(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device=t.device)
    wide[..., ::2] = t
    return wide[..., ::2]


def _shifted(t):                                           # ... four bytes behind a 16-byte boundary
    flat = torch.empty(t.numel() + 4, dtype=t.dtype, device=t.device)
    at = 4 // t.element_size()
    flat[at:at + t.numel()] = t.flatten()
    return flat[at:at + t.numel()].view(t.shape)


def _forms():
    each = lambda f, *names: lambda a: a.update({n: f(a[n]) for n in names})
    yield 'as it is', {}, None
    yield 'fp32', dict(dtype=torch.float32), None
    yield 'fp32, copies of the same numbers', dict(dtype=torch.float32), each(torch.clone, 'qa', 'k', 'v')
    yield 'fp32 off its boundary', dict(dtype=torch.float32), each(_shifted, 'q', 'va', 'beta')
    yield 'fp32 softmax side only', {}, each(torch.Tensor.float, 'qa', 'ka', 'va')
    yield 'fp32 linear side only', {}, each(torch.Tensor.float, 'q', 'k', 'v')
    yield 'strides', {}, each(_strided, 'qa', 'k', 'v', 'beta', 'g', 'types')
    yield 'fp32 strides', dict(dtype=torch.float32), each(_strided, 'q', 'ka', 'v')
    yield 'transposed heads', {}, each(lambda t: t.transpose(1, 2).contiguous().transpose(1, 2), 'qa', 'ka', 'va', 'q', 'k', 'v')
    yield 'gates and types of the other type', {}, lambda a: a.update(g=a['g'].bfloat16(), types=a['types'].float())
    yield 'options', {}, lambda a: a.update(state=False, decay=False, l2=False)
    yield 'initial state', {}, lambda a: a.update(h0=_strided(torch.randn(2, 2, 64, 64, device=DEV)))
    yield 'grouped heads', {}, lambda a: a.update(qa=torch.cat([a['qa'], a['qa'].flip(2)], 2).contiguous())
    yield 'one token', dict(T=1, B=1), None
    yield 'longer blocks', dict(T=700, block=128, K=128), None
    yield 'wanting gradients without recording', {}, each(lambda t: t.clone().requires_grad_(True), 'q', 'va')


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
@pytest.mark.parametrize("name,sizes,change", list(_forms()), ids=[f[0] for f in _forms()])
def test_plain_call_is_the_general_one(kind, name, sizes, change, monkeypatch):
    import neuralattentionsearchlinear_amd._mixed_common as MC
    a = _args(kind, **sizes)
    if change:
        if kind == 'mamba':
            a['beta'] = torch.zeros(1, device=DEV)          # (for the change; not an argument there)
        change(a)
    with torch.no_grad():
        for ops in ('all', 'attn', 'gated_delta_net' if kind == 'gdn' else 'mamba'):
            a['ops'] = ops
            took, inner = [], MC._plain_forward
            with monkeypatch.context() as mp:
                mp.setattr(MC, '_plain_forward', lambda *x: took.append(inner(*x)) or took[-1])
                plain = _call(kind, a)
            assert took and took[0] is not None, "the native call declined"
            with monkeypatch.context() as mp:
                mp.setattr(MC, '_plain_forward', lambda *x: None)
                general = _call(kind, a)
            for x, y in zip(plain, general):
                assert (x is None) == (y is None)
                if x is not None:
                    assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride() and not x.requires_grad
                    assert torch.equal(x, y), (name, ops)


def _others():
    yield 'half', lambda a: a.update({n: a[n].half() for n in ('qa', 'q')})
    yield 'integer types', lambda a: a.update(types=a['types'].int())
    yield 'blocks of 64.9', lambda a: a.update(block=64.9)
    yield 'blocks of 64.0', lambda a: a.update(block=64.0)
    yield 'blocks of 96', lambda a: a.update(block=96)
    yield 'types of three', lambda a: a.update(types=torch.cat([a['types'], a['types'][..., :1]], -1))
    yield 'a state of another shape', lambda a: a.update(h0=torch.zeros(1, 2, 64, 64, device=DEV))
    yield 'a state in bf16', lambda a: a.update(h0=torch.randn(2, 2, 64, 64, device=DEV).bfloat16())
    yield 'on the CPU', lambda a: a.update({n: a[n].cpu() for n in ('qa', 'ka', 'va', 'q', 'k', 'v')})
    yield 'head widths that are not built', lambda a: a.update({n: a[n][..., :32].contiguous() for n in ('qa', 'ka')})


@pytest.mark.parametrize("name,change", list(_others()), ids=[f[0] for f in _others()])
def test_other_calls_end_as_they_did(name, change, monkeypatch):
    import neuralattentionsearchlinear_amd._mixed_common as MC
    a = _args('gdn')
    change(a)

    def outcome():
        try:
            with torch.no_grad():
                return [t.clone() for t in _call('gdn', a)]
        except Exception as e:                              # noqa: BLE001 (whatever it is, it is the same)
            return type(e), str(e)
    with_it = outcome()
    with monkeypatch.context() as mp:
        mp.setattr(MC, '_plain_forward', lambda *x: None)
        without = outcome()
    if isinstance(without, list):
        assert isinstance(with_it, list) and all(torch.equal(x, y) for x, y in zip(with_it, without))
    else:
        assert with_it == without


def _misfits():
    yield 'a longer key tensor', lambda a: a.update(ka=torch.cat([a['ka'], a['ka']], 1))
    yield 'a shorter gate', lambda a: a.update(g=a['g'][:, :-1])
    yield 'a shorter beta in fp32', lambda a: a.update(beta=a['beta'][:, :-1].float())
    yield 'a value tensor of one sequence', lambda a: a.update(v=a['v'][:1])
    yield 'types of one sequence', lambda a: a.update(types=a['types'][:1])
    yield 'a gate on the CPU', lambda a: a.update(g=a['g'].cpu())


@pytest.mark.parametrize("gradients", [False, True])
@pytest.mark.parametrize("name,change", list(_misfits()), ids=[f[0] for f in _misfits()])
def test_tensors_that_do_not_go_together_are_refused(name, change, gradients, monkeypatch):
    """... before anything is launched."""
    from neuralattentionsearchlinear_amd import _capi
    a = _args('gdn')
    change(a)
    if gradients:
        a['q'] = a['q'].clone().requires_grad_(True)
    for entry in ('natsl_mixed_fwd', 'natsl_route'):
        monkeypatch.setattr(_capi.lib(), entry, lambda *x: pytest.fail("launched"))
    with pytest.raises(ValueError, match=r"must have shape|is on cpu"):
        _call('gdn', a)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("force", [False, True])
def test_hard_select_of_plain_logits(dtype, force, monkeypatch):
    from neuralattentionsearchlinear_amd import _capi, nats_util
    logits = torch.randn(3, 17, 4, 2, device=DEV).to(dtype)
    core = _capi.step_core()

    class Without:
        hard_select = staticmethod(lambda *a: None)
    for t in (logits, logits.transpose(1, 2).contiguous().transpose(1, 2), logits[:, :, ::2]):
        assert core.hard_select(_capi.entries(), t, force, _capi.stream_ptr(t.device)) is not None
        plain = nats_util.hard_select(t, force)
        with monkeypatch.context() as mp:
            mp.setattr(_capi, 'step_core', lambda: Without)
            general = nats_util.hard_select(t, force)
        assert all(torch.equal(x, y) and x.dtype == y.dtype and x.stride() == y.stride() for x, y in zip(plain, general))
    assert core.hard_select(_capi.entries(), logits.half(), force, _capi.stream_ptr(logits.device)) is None
    assert core.hard_select(_capi.entries(), logits[:0], force, _capi.stream_ptr(logits.device)) is None
