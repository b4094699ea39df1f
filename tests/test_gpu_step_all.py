"""The one-token generation step as one launch, products included, against the same step as three launches, bit for bit; and what becomes of a
part of it that waits too long."""
import ctypes

import pytest
import torch

from tests.test_gpu_layer_step import _generate, _layer

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _three_launches(monkeypatch):
    from neuralattentionsearchlinear_amd import _capi
    none = ctypes.CFUNCTYPE(ctypes.c_size_t, ctypes.c_void_p)(lambda step: 0)
    monkeypatch.setattr(_capi.lib(), 'natsl_layer_step_sync_bytes', none)
    return none                                            # (held by the caller while a plan has its address)


@pytest.mark.parametrize("kind,geometry,B,T0,n,more", [
    ('gdn', '340M', 1, 777, 5, {}),
    ('gdn', '340M', 3, 100, 30, {}),                                       # over the end of a block: the cache and the splits change
    ('gdn', '760M', 1, 300, 3, dict(allow_neg_eigval=True, conv_bias=True)),
    ('gdn', None, 1, 64, 2, dict(head_dim=64, num_heads=2, num_attn_heads=2, expand_v=1)),   # rows of 128: one step of the products a wave
    ('gdn', None, 5, 127, 3, dict(hidden_size=288, head_dim=64, num_heads=5, num_attn_heads=5)),  # 9 steps, 5-row weights, products' waves of 2 and 3
    ('mamba', None, 2, 95, 3, dict(expand_v=1)),
    ('mamba', None, 16, 64, 2, dict(head_dim=64, num_heads=2, num_attn_heads=2, expand_v=1)),   # a whole row tile
    ('mamba', None, 1, 257, 2, dict(attn_with_short_conv=False, conv_bias=True)),
])
def test_one_launch_is_the_three(kind, geometry, B, T0, n, more, monkeypatch):
    layer = _layer(kind, geometry, 'all', **more)
    torch.manual_seed(T0)
    x = torch.randn(B, T0 + n, layer.hidden_size, device=DEV).bfloat16()
    one, c1 = _generate(layer, kind, x, T0, (1,) * n)
    again, _ = _generate(layer, kind, x, T0, (1,) * n)
    assert c1.step_shared is not None and int(c1.step_shared[64]) == n, "the steps were not one launch each"
    held = _three_launches(monkeypatch)
    layer2 = _layer(kind, geometry, 'all', **more)
    three, c3 = _generate(layer2, kind, x, T0, (1,) * n)
    assert c3.step_shared is None and held is not None
    for i, (a, b, c) in enumerate(zip(one, again, three)):
        assert torch.equal(a, b) and torch.equal(a, c), f"step {i}"
    for name in ('attn_k', 'attn_v', 'recurrent_state', 'g_cumsum', 'lattn_g', 'l_attn_k', 'l_attn_v'):
        a, b = getattr(c1, name), getattr(c3, name)
        n_in = c1._n_tokens_in_nats_block
        if name.startswith('l'):
            a, b = a[:, :n_in], b[:, :n_in]
        elif name.startswith('attn'):
            a, b = a[:, :c1.n_attn_tokens_max], b[:, :c1.n_attn_tokens_max]
        assert torch.equal(a, b), name


def test_a_step_that_waits_too_long_gives_no_numbers(monkeypatch):
    """With no time to wait every part of the launch gives up at once: it ends, its output is NaN, and so are those of later steps on that cache;
    another cache is not touched by it."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    torch.manual_seed(0)
    x = torch.randn(1, 103, 256, device=DEV).bfloat16()
    good, _ = _generate(_layer('gdn', None, 'all'), 'gdn', x, 100, (1,) * 3)
    monkeypatch.setattr(LS, 'MAX_WAIT_US', 0)
    layer = _layer('gdn', None, 'all')
    bad, cache = _generate(layer, 'gdn', x, 100, (1,) * 3)
    torch.cuda.synchronize()
    assert int(cache.step_shared[32]) == 1
    assert all(bool(o.isnan().all()) for o in bad[1:])
    monkeypatch.undo()
    after, _ = _generate(_layer('gdn', None, 'all'), 'gdn', x, 100, (1,) * 3)
    assert all(torch.equal(a, b) for a, b in zip(good, after))


@pytest.mark.parametrize("T,launches", [(2, 'five'), (1, 'three')])
def test_a_failed_step_is_not_gone_on_from_in_several_launches(T, launches, monkeypatch):
    """A step that failed leaves stale numbers in the cache's rows: later steps on it give none, in however many launches they are, and for another number
    of sequences, whose steps meet in other memory, too."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    from neuralattentionsearchlinear_amd.cache import NAtSCache
    torch.manual_seed(0)
    x = torch.randn(1, 110, 256, device=DEV).bfloat16()
    layer = _layer('gdn', None, 'all')
    monkeypatch.setattr(LS, 'MAX_WAIT_US', 0)
    holder = NAtSCache()
    with torch.no_grad():
        for piece in (x[:, :100], x[:, 100:101]):
            layer(piece, past_key_values=holder, use_cache=True)
        assert int(holder[0].step_shared[32]) == 1
        monkeypatch.undo()
        held = _three_launches(monkeypatch) if launches == 'three' else None
        later = _layer('gdn', None, 'all')                 # (the same weights; a plan of its own)
        out = later(x[:, 101:101 + T], past_key_values=holder, use_cache=True)[0]
        assert bool(out.isnan().all()), "numbers from a cache that a failed step has written"
        del held                                           # (the plan has its address until here)
        if launches == 'five':
            cache = holder[0]
            for name, t in list(vars(cache).items()):      # the same sequence twice
                if torch.is_tensor(t) and name != 'step_shared':
                    setattr(cache, name, t.repeat_interleave(2, 0))
            cache.conv_state = tuple(t.repeat_interleave(2, 0) for t in cache.conv_state)
            before = cache.step_shared.numel()
            out = later(x[:, 103:104].repeat_interleave(2, 0), past_key_values=holder, use_cache=True)[0]
            assert cache.step_shared.numel() != before and bool(out.isnan().all())


def test_caches_on_streams_of_their_own():
    """Steps of three caches, each on its own stream, in turn and without a wait between: those that find another's under way are three launches, and
    all give what they give alone."""
    from neuralattentionsearchlinear_amd.cache import NAtSCache
    layer, n = _layer('gdn', '340M', 'all'), 20
    torch.manual_seed(1)
    xs = [torch.randn(1, 150 + n, layer.hidden_size, device=DEV).bfloat16() for _ in range(3)]
    alone = [_generate(layer, 'gdn', x, 150, (1,) * n)[0] for x in xs]
    torch.cuda.synchronize()
    streams, holders, outs = [torch.cuda.Stream() for _ in xs], [NAtSCache() for _ in xs], [[] for _ in xs]
    with torch.no_grad():
        for t in range(n + 1):
            for x, s, h, o in zip(xs, streams, holders, outs):
                with torch.cuda.stream(s):
                    piece = x[:, :150] if t == 0 else x[:, 149 + t:150 + t]
                    o.append(layer(piece, past_key_values=h, use_cache=True)[0])
    torch.cuda.synchronize()
    for a, o in zip(alone, outs):
        assert all(torch.equal(p, q) for p, q in zip(a, o))
    assert all(int(h[0].step_shared[32]) == 0 for h in holders)


def test_a_failed_step_is_reported_where_the_host_waits(monkeypatch):
    """The host waits for a cache's steps at a block's end: there a step that gave up is an error, and no other cache's."""
    import neuralattentionsearchlinear_amd._layer_step as LS
    from neuralattentionsearchlinear_amd import _capi
    torch.manual_seed(0)
    x = torch.randn(1, 130, 256, device=DEV).bfloat16()
    good, _ = _generate(_layer('gdn', None, 'all'), 'gdn', x, 120, (1,) * 10)
    with monkeypatch.context() as mp:
        mp.setattr(LS, 'MAX_WAIT_US', 0)
        with pytest.raises(_capi.NatslError, match="gave up"):
            _generate(_layer('gdn', None, 'all'), 'gdn', x, 120, (1,) * 10)
    assert _capi.lib().natsl_layer_step_gave_up(0) > 0
    after, cache = _generate(_layer('gdn', None, 'all'), 'gdn', x, 120, (1,) * 10)
    assert all(torch.equal(a, b) for a, b in zip(good, after)) and cache._gave_up == _capi.lib().natsl_layer_step_gave_up(0)
