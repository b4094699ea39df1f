"""The layers' fused front and tail (_front.FastFront) against their general path of single submodules: outputs, gradients and caches;
and the weight-gradient kernel against an fp32 product at the edges of its tiles."""
import pytest
import torch

from tests._util import rel_l2
from tests.test_gpu_layer_step import _generate as _generate_views, _layer

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _generate(layer, kind, x, T0, sizes):
    """_generate of the steps' tests on hidden states of their own, as a model's layers hand them on (the fused front and the native calls take contiguous
    ones; a view of several sequences' first tokens is not)."""
    whole = layer.forward
    try:
        layer.forward = lambda t, **kw: whole(t.contiguous(), **kw)
        return _generate_views(layer, kind, x, T0, sizes)
    finally:
        del layer.forward


def _general(monkeypatch):
    from neuralattentionsearchlinear_amd import natsl_attn_gdn, natsl_attn_mamba2
    for mod in (natsl_attn_gdn, natsl_attn_mamba2):
        monkeypatch.setattr(mod, 'fast_front', lambda *a: None)


@pytest.mark.parametrize("kind,geometry,B,T,more", [
    ('gdn', None, 1, 64, {}), ('gdn', '340M', 2, 333, {}), ('gdn', '760M', 1, 200, dict(allow_neg_eigval=True, conv_bias=True)),
    ('gdn', None, 3, 130, dict(conv_size=3, conv_activation=None)), ('gdn', None, 2, 65, dict(conv_size=2)),
    ('mamba', None, 2, 257, {}), ('mamba', None, 1, 100, dict(attn_qk_norm=True, conv_bias=True)),
    ('gdn', '340M', 7, 1999, {}), ('gdn', None, 16, 4100, dict(conv_size=3)),             # long runs, the last one short
])
def test_front_matches_the_general_path(kind, geometry, B, T, more, monkeypatch):
    layer = _layer(kind, geometry, 'all', **more).train()
    torch.manual_seed(T)
    x0 = torch.randn(B, T, layer.hidden_size, device=DEV).bfloat16()
    do = torch.randn_like(x0)

    def run():
        x = x0.clone().requires_grad_(True)
        layer.zero_grad(set_to_none=True)
        o = layer(x)
        o = o[0] if isinstance(o, tuple) else o
        o.backward(do)
        return dict({n: p.grad for n, p in layer.named_parameters()}, x=x.grad, out=o.detach(), fraction=layer.attn_fraction)
    fast = run()
    _general(monkeypatch)
    slow = run()
    for n, b in slow.items():
        a = fast[n]
        assert a is not None and a.shape == b.shape and a.dtype == b.dtype, n
        # Both sides round to bf16 on the way (2^-9 relative each time); sums that the fused steps keep in fp32 are rounded once
        # more in the general path.  The selector's gradient is a sum of terms that largely cancel: ten times that.
        tol = 5e-2 if n == 'nats_layer.weight' else 1e-2
        assert rel_l2(a.float(), b.float()) <= tol, f"{n}: rel-L2 {rel_l2(a.float(), b.float()):.3e}"


@pytest.mark.parametrize("kind,T0,sizes", [('gdn', 128, (1, 70)), ('gdn', 100, (64,)), ('mamba', 131, (2, 100))])
def test_front_on_a_cache(kind, T0, sizes, monkeypatch):
    """Prefill and a second prompt: the same outputs and convolution states as the general path."""
    layer = _layer(kind, None, 'all')
    torch.manual_seed(T0)
    x = torch.randn(2, T0 + sum(sizes), layer.hidden_size, device=DEV).bfloat16()
    from neuralattentionsearchlinear_amd import _front
    calls, tail = [], _front.FastFront.tail
    monkeypatch.setattr(_front.FastFront, 'tail', lambda *a: (calls.append(1), tail(*a))[1])
    native = _front.FastFront.prompt
    monkeypatch.setattr(_front.FastFront, 'prompt', lambda *a: (calls.append(1), native(*a))[1])
    fast, cf = _generate(layer, kind, x, T0, sizes)
    # (pieces of fewer than 64 tokens are steps)
    assert len(calls) == 1 + sum(n >= 64 for n in sizes)
    _general(monkeypatch)
    slow, cs = _generate(layer, kind, x, T0, sizes)
    for a, b in zip(fast + list(cf.conv_state), slow + list(cs.conv_state)):
        assert rel_l2(a.float(), b.float()) <= 5e-3
    assert torch.equal(cf.n_attn_blocks, cs.n_attn_blocks)


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
@pytest.mark.parametrize("where", ['instance', 'subclass'])
@pytest.mark.parametrize("train", [False, True])
def test_an_overridden_selector_is_called(kind, where, train):
    """A layer's select_ops decides in training and prefill too, also where a subclass or an instance has its own: here every block goes
    to one operator, which the layer's own selector would not do."""
    layer = _layer(kind, None, 'all')
    own, calls = type(layer).select_ops, []

    def only_linear(self, hidden_states, cu_seqlens=None, force_last_block=True):
        calls.append(hidden_states.shape)
        types, counts, last = own(self, hidden_states, cu_seqlens, force_last_block)
        types, last = torch.zeros_like(types), torch.zeros_like(last)
        types[..., 1] = last[..., 1] = 1
        return types, counts, last
    torch.manual_seed(4)
    x = torch.randn(2, 8 * layer.nats_block_size, layer.hidden_size, device=DEV).bfloat16()
    run = lambda: layer.train()(x) if train else _generate(layer.eval(), kind, x, x.shape[1], ())
    run()
    assert float(layer.attn_fraction.float().mean()) > 0.2           # (the layer's own choice)
    if where == 'instance':
        layer.select_ops = only_linear.__get__(layer)
    else:
        layer.__class__ = type('Other', (type(layer),), dict(select_ops=only_linear))
    run()
    assert calls == [x.shape]
    assert torch.equal(layer.attn_fraction.float(), torch.full_like(layer.attn_fraction.float(), 1 / 8))     # the last block runs both


@pytest.mark.parametrize("W,bias", [(4, False), (3, True), (2, False)])
def test_conv_arithmetic_is_the_single_kernels(W, bias):
    """The fused convolution forms its activation, and the gradients behind it, with the arithmetic of natsl_short_conv_*: the same bits.
    (A reciprocal in the place of the division moves about one rounding to bf16 in 2^15; a tensor here holds 2^22 values.)"""
    from neuralattentionsearchlinear_amd import _front
    layer = _layer('gdn', None, 'all', conv_size=W, conv_bias=bias)
    torch.manual_seed(W)
    B, T = 4, 4096
    f = _front.fast_front(layer, 'gdn', torch.zeros(B, T, layer.hidden_size, device=DEV).bfloat16(), None, None)
    raw = [torch.randn(B, T, c.hidden_size, device=DEV).bfloat16() for c in (layer.q_conv1d, layer.k_conv1d, layer.v_conv1d)]
    ref = lambda i, x: (layer.q_conv1d, layer.k_conv1d, layer.v_conv1d)[i](x)[0]
    with torch.no_grad():
        for i, y in enumerate(_front._conv_norm(f, raw, None, False)[0]):
            assert torch.equal(y, ref(i, raw[i])), "qkv"[i]
    grads = []
    for fused in (True, False):
        x = [r.clone().requires_grad_(True) for r in raw]
        ys = f.conv_norm(*x, (None,) * 3, False)[:3] if fused else [ref(i, t) for i, t in enumerate(x)]
        torch.manual_seed(1)
        torch.autograd.backward(ys, [torch.randn_like(y) for y in ys])
        grads.append([t.grad for t in x])
    for a, b, n in zip(*grads, "qkv"):
        assert torch.equal(a, b), f"d{n}"


def test_mixing_softmax_is_the_separate_ones():
    """The norm-gate that takes mixing logits gives what it gives for the weights of torch's bf16 softmax, forward and backward: the same
    bits.  (An exponential an ulp off moves about one weight in 2^15 across a rounding edge; here are 2^21 of them.)"""
    from neuralattentionsearchlinear_amd import _capi
    torch.manual_seed(2)
    rows, D = 1 << 20, 32
    a, b, g, dy = (torch.randn(rows, D, device=DEV).bfloat16() for _ in range(4))
    logits = 3 * torch.randn(rows, 2, device=DEV).bfloat16()
    w = torch.rand(2, D, device=DEV)
    L, P, st = _capi.lib(), _capi.ptr, _capi.stream_ptr(a.device)
    n = L.natsl_norm_gate_bwd_workspace_bytes(rows, D)
    outs = []
    for fused, xw in ((True, logits), (False, logits.softmax(-1))):
        y, da, db, dg = (torch.empty_like(a) for _ in range(4))
        dx = torch.empty(rows, 2, dtype=torch.bfloat16 if fused else torch.float32, device=DEV)
        dw, ws = torch.empty(2, D, device=DEV), torch.empty(n, dtype=torch.uint8, device=DEV)
        fwd, bwd = (L.natsl_norm_gate_logits_fwd, L.natsl_norm_gate_logits_bwd) if fused else (L.natsl_norm_gate_fwd, L.natsl_norm_gate_bwd)
        _capi.check(fwd(P(a), P(b), P(g), P(xw), P(w[0]), P(w[1]), P(y), rows, D, _capi.BF16, 1e-5, _capi.F32, st), "forward")
        _capi.check(bwd(P(a), P(b), P(g), P(xw), P(w[0]), P(w[1]), P(dy), P(da), P(db), P(dg), P(dx), P(dw[0]), P(dw[1]), P(ws), n, rows, D,
                        _capi.BF16, 1e-5, _capi.F32, st), "backward")
        outs.append((y, da, db, dg, dw))
    for i, (p, q) in enumerate(zip(*outs)):
        assert torch.equal(p, q), f"output {i}: {int((p != q).sum())} values differ"


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
def test_replaced_weights_are_freed(kind):
    """What the fused front and the step remember of a layer keeps no tensor alive: a replaced weight, and weights that a functional call
    puts in for one forward, go with their last owner."""
    import gc
    import weakref
    layer = _layer(kind, None, 'all')
    torch.manual_seed(3)
    x = torch.randn(2, 101, layer.hidden_size, device=DEV).bfloat16()
    _generate(layer, kind, x, 100, (1,))
    old = [weakref.ref(p) for p in layer.parameters()]
    own = weakref.ref(layer.g_proj)
    for name, p in list(layer.named_parameters()):
        mod, _, leaf = name.rpartition('.')
        setattr(layer.get_submodule(mod), leaf, torch.nn.Parameter(p.detach().clone()))
    del p
    layer.g_proj = torch.nn.Linear(layer.g_proj.in_features, layer.g_proj.out_features, bias=False, device=DEV, dtype=torch.bfloat16)
    gc.collect()
    assert own() is None and not any(r() is not None for r in old)
    made = {n: p.detach().clone().requires_grad_(True) * 1.0 for n, p in layer.named_parameters()}
    old = [weakref.ref(t) for t in made.values()]
    o = torch.func.functional_call(layer.train(), made, (x[:, :100],))
    (o[0] if isinstance(o, tuple) else o).sum().backward()
    del made, o
    gc.collect()
    assert not any(r() is not None for r in old)


@pytest.mark.parametrize("T,D,widths", [(1, 8, (8,)), (31, 64, (16, 24)), (32, 256, (256,)), (33, 264, (264, 8)), (129, 72, (512,)), (5000, 128, (136,)), (9000, 768, (24,)), (9001, 128, (264, 32))])
def test_weight_grads(T, D, widths):
    """natsl_wgrad at the edges of its 32-token stages, 256-wide tiles and token slices."""
    from neuralattentionsearchlinear_amd._front import weight_grads
    torch.manual_seed(T)
    x = torch.randn(T, D, device=DEV).bfloat16()
    dys = [torch.randn(T, n, device=DEV).bfloat16() for n in widths]
    out = weight_grads(x, dys)
    again = weight_grads(x, dys)
    for dy, a, b in zip(dys, out, again):
        ref = dy.double().t() @ x.double()
        # exact products, fp32 sums (T 2^-24 of the sum of magnitudes, far below), one rounding to bf16
        assert bool(((a.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * T ** 0.5).all()), float((a.double() - ref).abs().max())
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,T,D,N,block,pool", [(1, 1, 8, 16, 64, True), (2, 100, 264, 32, 64, True), (1, 70, 1032, 0, 256, True), (3, 33, 64, 16, 64, False)])
def test_dx_init(B, T, D, N, block, pool):
    from neuralattentionsearchlinear_amd import _capi
    torch.manual_seed(D)
    nb = -(-T // block)
    dn, w = torch.randn(B * T, max(N, 16), device=DEV).bfloat16(), torch.randn(max(N, 1), D, device=DEV).bfloat16()
    dp = torch.randn(B, nb, D, device=DEV).bfloat16()
    dx = torch.full((B, T, D), float('nan'), device=DEV).bfloat16()
    P = _capi.ptr
    _capi.check(_capi.lib().natsl_dx_init(P(dn) if N else None, P(w) if N else None, P(dp) if pool else None, P(dx), B, T, D, N, max(N, 16), block,
                                          _capi.stream_ptr(dx.device)), "natsl_dx_init")
    ref = (dn[:, :N].double() @ w[:N].double()).view(B, T, D) if N else torch.zeros(B, T, D, device=DEV, dtype=torch.float64)
    if pool:
        lens = torch.full((nb,), block, device=DEV, dtype=torch.float64)
        lens[-1] = T - (nb - 1) * block
        ref = ref + (dp.double() / lens.view(1, nb, 1)).repeat_interleave(block, 1)[:, :T]
    assert bool(((dx.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all())


# around a batch of 256 / H rows, a workgroup's batches and the most workgroups; columns that fill no group of the sums' kernel
@pytest.mark.parametrize("rows,H,delta,neg", [(1, 1, True, False), (85, 6, True, True), (4099, 16, False, False), (9001, 100, True, False), (5000, 256, True, True),
                                              (140001, 32, False, False), (50000, 200, True, False)])
def test_gates_backward(rows, H, delta, neg):
    """natsl_gates_bwd against 64 bits.  bf16 outputs are rounded once; a parameter's gradient is a sum of fp32 terms that are within 4e-6 of
    exact ones (expf, log1pf, a few products) and loses a rounding where it is rounded to fp32."""
    from neuralattentionsearchlinear_amd import _capi
    torch.manual_seed(rows)
    L, P = _capi.lib(), _capi.ptr
    ld = 2 * H + 3 if delta else H + 5
    ab, a_log, bias = torch.randn(rows, ld, device=DEV).bfloat16(), torch.randn(H, device=DEV), torch.randn(H, device=DEV)
    dg, ddt = torch.randn(rows, H, device=DEV), None if delta else torch.randn(rows, H, device=DEV)
    db = torch.randn(rows, H, device=DEV).bfloat16() if delta else None
    dab, da, dd = torch.full_like(ab, 7.), torch.empty_like(a_log), torch.empty_like(bias)
    n = L.natsl_gates_bwd_workspace_bytes(rows, H)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    rc = L.natsl_gates_bwd(P(ab), P(a_log), P(bias), P(dg), P(db) if delta else None, None if delta else P(ddt), int(delta), P(dab), P(da), P(dd), P(ws), n, rows, H,
                           ld, int(neg), _capi.F32, _capi.stream_ptr(dg.device))
    _capi.check(rc, "natsl_gates_bwd")
    x, A = ab[:, :H].double() + bias.double(), a_log.double().exp()
    dt = torch.nn.functional.softplus(x, threshold=1e9)
    ta = dg.double() * -A * dt
    tb = ((0. if delta else ddt.double()) - A * dg.double()) * x.sigmoid()
    close = lambda got, ref, terms: bool(((got.double() - ref).abs() <= 2.0 ** -24 * ref.abs() + 4e-6 * terms.abs().sum(0)).all())
    assert close(da, ta.sum(0), ta) and close(dd, tb.sum(0), tb)
    assert bool(((dab[:, :H].double() - tb).abs() <= 2.0 ** -8 * tb.abs() + 1e-5).all())
    if delta:
        s = ab[:, H:2 * H].double().sigmoid().bfloat16().double()
        ref = (2. if neg else 1.) * db.double() * s * (1 - s)
        # (a sigmoid at the edge of two bf16 values may round to the other: s (1 - s) changes by less than 2^-8)
        assert bool(((dab[:, H:2 * H].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -7 * db.double().abs()).all())
    assert not bool(dab[:, (2 if delta else 1) * H:].any())


# (tokens, input width, projections): rows and columns behind the last tile, tiles of each height, more tiles than workgroups
@pytest.mark.parametrize("B,T,D,widths,block", [
    (1, 1, 128, (8,), 64), (1, 129, 160, (264, 32), 64), (3, 100, 416, (256, 64, 512, 32), 64), (2, 8200, 128, (520, 1024), 256),
    (1, 16320, 768, (96, 32), 64), (1, 16320, 160, (512, 256), 64), (2, 8191, 1024, (64, 64), 128), (1, 40000, 264, (96, 128), 64), (1, 9000, 1032, (768, 768, 1536, 1536, 32), 64)])
def test_joint_projections(B, T, D, widths, block):
    """natsl_project and natsl_project_bwd: exact products, fp32 sums and one rounding to bf16."""
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._front import _project_segs
    torch.manual_seed(T)
    L, P, rows, nb = _capi.lib(), _capi.ptr, B * T, -(-T // block)
    x, ws = torch.randn(rows, D, device=DEV).bfloat16(), [torch.randn(n, D, device=DEV).bfloat16() for n in widths]
    close = lambda a, ref: bool(((a.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * sum(widths + (D,)) ** 0.5).all())
    if D % 32 == 0:
        guard = [torch.full((rows + 1, n), 7., device=DEV).bfloat16() for n in widths]
        ys = [g[:rows] for g in guard]
        _capi.check(L.natsl_project(_project_segs(ys, ws), len(ws), P(x), rows, D, D, _capi.stream_ptr(x.device)), "natsl_project")
        for y, w, g in zip(ys, ws, guard):
            assert close(y, x.double() @ w.double().t())
            assert bool((g[rows] == 7).all())
    else:
        assert L.natsl_project(_project_segs([x], ws[:1]), 1, P(x), rows, D, D, _capi.stream_ptr(x.device)) != 0
    dys = [torch.randn(rows, n, device=DEV).bfloat16() for n in widths]
    dp = torch.randn(B, nb, D, device=DEV).bfloat16()
    lens = torch.full((nb,), block, device=DEV, dtype=torch.float64)
    lens[-1] = T - (nb - 1) * block
    spread = (dp.double() / lens.view(1, nb, 1)).repeat_interleave(block, 1)[:, :T].reshape(rows, D)
    for pool in (None, dp):
        dx = torch.full((rows + 1, D), 7., device=DEV).bfloat16()
        rc = L.natsl_project_bwd(_project_segs(dys, ws), len(ws), P(pool) if pool is not None else None, P(dx), B, T, D, block, _capi.stream_ptr(x.device))
        if sum(widths) < 128 or any(n % 32 for n in widths):
            assert rc != 0                                                  # (refused: the caller's other path)
            continue
        _capi.check(rc, "natsl_project_bwd")
        ref = sum(dy.double() @ w.double() for dy, w in zip(dys, ws))
        assert close(dx[:rows], ref if pool is None else ref + spread)
        assert bool((dx[rows] == 7).all())


@pytest.mark.parametrize("rows,D,N", [(1, 128, 4), (33, 768, 24), (63, 1152, 36), (64, 2048, 32), (65, 1280, 48), (257, 384, 44), (4099, 256, 16), (16387, 1152, 40)])
def test_narrow_product_backward(rows, D, N):
    """natsl_narrow_linear_bwd at the edges of its tiles of tokens, columns and weight rows; what it is chosen for, and the library's else."""
    from neuralattentionsearchlinear_amd import _capi, _front
    torch.manual_seed(rows)
    L, P = _capi.lib(), _capi.ptr
    w, dy = torch.randn(N, D, device=DEV).bfloat16(), torch.randn(rows, N, device=DEV).bfloat16()
    dx = torch.full((rows + 1, D), 7., device=DEV).bfloat16()
    _capi.check(L.natsl_narrow_linear_bwd(P(dy), P(w), P(dx), rows, D, N, _capi.stream_ptr(w.device)), "natsl_narrow_linear_bwd")
    ref = dy.double() @ w.double()
    # exact products, fp32 sums, one rounding to bf16
    bound = 2.0 ** -8 * ref.abs() + 1e-5 * D ** 0.5
    assert bool(((dx[:rows].double() - ref).abs() <= bound).all()) and bool((dx[rows] == 7).all())
    for refused in (N + 2, 52):
        assert L.natsl_narrow_linear_bwd(P(dy), P(w), P(dx), rows, D, refused, _capi.stream_ptr(w.device)) != 0
    got = _front._narrow_bwd(dy, w)
    assert torch.equal(got, dx[:rows]) if _front._narrow_pays(rows, N, D) else bool(((got.double() - ref).abs() <= bound).all())


def test_joint_projections_only_where_they_pay():
    """The line between natsl_project and the library: fewer rounds of tiles, and for wide inputs many fewer."""
    from neuralattentionsearchlinear_amd._front import _joint_pays
    pays = lambda rows, D, *widths: _joint_pays(rows, D, widths, 256)
    assert pays(32768, 1024, 768, 768, 1536, 1536) and pays(16384, 1536, 1152, 1152, 2304, 2304) and pays(1, 1024, 768, 768, 1536, 1536)
    assert not pays(32768, 1024, 2048, 2048, 1024, 1024) and not pays(0, 1024, 768, 768, 1536, 1536) and not pays(777, 1032, 768, 768, 1536, 1536)
    wide = 2048, 1536, 1536, 3072, 3072
    assert pays(3000, *wide) and pays(12000, *wide) and not any(pays(rows, *wide) for rows in (0, 4096, 16384, 24000, 49152))


def test_narrow_product_only_where_it_pays():
    """The line between natsl_narrow_linear_bwd and the library: rows of the weight, and elements of what is written."""
    from neuralattentionsearchlinear_amd._front import _narrow_pays
    assert _narrow_pays(6000, 24, 768) and _narrow_pays(6000, 36, 1152) and _narrow_pays(65536, 48, 768) and _narrow_pays(32768, 8, 512)
    assert not any(_narrow_pays(rows, N, D) for rows in (1, 777, 65536) for N in (32, 52, 60, 64) for D in (128, 1280, 2048))
    assert not _narrow_pays(2048, 24, 768) and not _narrow_pays(2048, 36, 1152) and not _narrow_pays(0, 24, 768)


@pytest.mark.parametrize("n_a,n_b", [(16, 0), (6, 6), (16, 16), (8, 40), (24, 24), (32, 0)])
def test_narrow_projections_of_any_count_join_the_backward(n_a, n_b):
    """The narrow projections' joint weight is made of whole stages where a gradient is asked for, whatever their rows are: one natsl_project_bwd
    and no natsl_dx_init.  Operands are bf16, sums fp32, one rounding each: 2^-8 in the norm at most."""
    from neuralattentionsearchlinear_amd import _front
    torch.manual_seed(n_a + n_b)
    B, T, D = 2, 130, 256
    x = torch.randn(B, T, D, device=DEV).bfloat16().requires_grad_(True)
    ws = [(torch.randn(n, D, device=DEV) / 16).bfloat16().requires_grad_(True) if n else None for n in (128, 128, 256, 256, n_a, n_b)]
    q, k, v, g, ab, pooled = _front._Project.apply(x, *ws, 64)
    used = n_a + n_b
    assert ab.shape[-1] % 32 == 0 and ab.shape[-1] - used < 32
    dys = [torch.randn_like(t) for t in (q, k, v, g, ab, pooled)]
    dys[4][..., used:] = 0
    got = torch.autograd.grad((q, k, v, g, ab, pooled), [x] + [w for w in ws if w is not None], dys)
    x32, w32 = x.detach().float().requires_grad_(True), [w.detach().float().requires_grad_(True) for w in ws if w is not None]
    outs = [x32 @ w.t() for w in w32]
    means = torch.stack([x32[:, t:t + 64].mean(1) for t in range(0, T, 64)], 1)
    ups = [d.float() for d in dys[:4]] + [d.contiguous() for d in dys[4][..., :used].float().split([n for n in (n_a, n_b) if n], -1)] + [dys[5].float()]
    want = torch.autograd.grad(outs + [means], [x32] + w32, ups)
    for a, b in zip(got, want):
        assert a.shape == b.shape and rel_l2(a.float(), b) <= 2 ** -8


@pytest.mark.parametrize("B,T,D,n_a,n_b,n_l,params", [
    (1, 1, 32, 1, 0, 0, torch.float32), (2, 63, 96, 6, 6, 12, torch.bfloat16), (1, 64, 512, 16, 0, 32, torch.float32), (3, 65, 544, 8, 8, 2, torch.bfloat16),
    (2, 129, 1536, 6, 6, 12, torch.float32), (1, 257, 1024, 16, 16, 64, torch.bfloat16), (1, 200, 160, 36, 0, 0, torch.float32), (1, 70, 1184, 31, 31, 0, torch.float32)])
def test_narrow_front(B, T, D, n_a, n_b, n_l, params):
    """natsl_layer_front at the edges of its 64-token tiles, of its 64-column steps and of 16 weight rows, with and without logits; what it refuses."""
    import ctypes
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._front import _FrontArgs
    torch.manual_seed(T + D)
    L, nb, ld, N = _capi.lib(), -(-T // 64), -(-(n_a + n_b) // 32) * 32, n_a + n_b
    bf = lambda *s: (torch.randn(*s, device=DEV) / D ** 0.25).bfloat16()
    x, wa, wb, wn = bf(B, T, D), bf(n_a, D), bf(n_b, D), bf(n_l, D)
    a_log, bias = torch.randn(n_a, device=DEV).to(params), torch.randn(n_a, device=DEV).to(params)
    delta = n_b == n_a
    full = lambda *s, dt=torch.bfloat16: torch.full(s, 7., device=DEV, dtype=dt)
    ab, pooled, logits, wab = full(B * T + 1, ld), full(B * nb + 1, D), full(B * nb + 1, max(n_l, 1)), full(ld + 1, D)
    g, beta, dt = full(B * T + 1, n_a, dt=torch.float32), full(B * T + 1, n_a), full(B * T + 1, n_a, dt=torch.float32)
    a = _FrontArgs()
    for n, t in dict(x=x, wa=wa, wb=wb if n_b else None, wn=wn if n_l else None, a_log=a_log, dt_bias=bias, ab=ab, pooled=pooled if n_l else None,
                     logits=logits if n_l else None, beta=beta if delta else None, wab=wab, g=g, dt=dt).items():
        setattr(a, n, None if t is None else t.data_ptr())
    a.B, a.T, a.D, a.NA, a.NB, a.NL, a.ld, a.neg_eigval, a.param_dtype, a.wab_rows = B, T, D, n_a, n_b, n_l, ld, int(T % 2), _capi.dtype_code(params), ld
    run = lambda: L.natsl_layer_front(ctypes.byref(a), _capi.stream_ptr(x.device))
    _capi.check(run(), "natsl_layer_front")
    # exact products, fp32 sums, one rounding to bf16
    close = lambda got, ref, k: bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * k ** 0.5).all())
    x2 = x.view(B * T, D).double()
    assert close(ab[:B * T, :N], x2 @ torch.cat([wa, wb]).double().t(), D) and not bool(ab[:B * T, N:].any())
    assert torch.equal(wab[:N], torch.cat([wa, wb])) and not bool(wab[N:ld].any())
    if n_l:
        means = torch.stack([x[:, t:t + 64].double().mean(1) for t in range(0, T, 64)], 1).view(B * nb, D)
        assert close(pooled[:B * nb], means, 64) and close(logits[:B * nb], pooled[:B * nb].double() @ wn.double().t(), D)
    step = torch.nn.functional.softplus(ab[:B * T, :n_a].double() + bias.double())
    assert torch.allclose(dt[:B * T].double(), step, rtol=1e-5, atol=1e-30) and torch.allclose(g[:B * T].double(), -a_log.double().exp() * step, rtol=1e-5, atol=1e-30)
    if delta:
        ref = torch.sigmoid(ab[:B * T, n_a:N].double()) * (2 if T % 2 else 1)
        assert close(beta[:B * T], ref, 1)
    for t in (ab, pooled, logits, wab, g, beta, dt):                        # nothing behind the ends
        assert bool((t[-1] == 7).all())
    a.D = D + 8
    assert run() != 0
    a.D, a.NL = D, 65 if n_l else 0
    a.NA = n_a if n_l else 65
    assert run() != 0


@pytest.mark.parametrize("rows,D,N", [(1, 32, 2), (31, 96, 12), (33, 1024, 16), (256, 130, 17), (513, 1152, 36), (1024, 64, 64)])
def test_narrow_weight_gradient(rows, D, N):
    """natsl_narrow_wgrad at the edges of its 32-token steps, 32 columns and 16 weight rows; and the library where it is not chosen."""
    from neuralattentionsearchlinear_amd import _capi, _front
    torch.manual_seed(rows)
    L, P = _capi.lib(), _capi.ptr
    x, dy = torch.randn(rows, D, device=DEV).bfloat16(), torch.randn(rows, N, device=DEV).bfloat16()
    dw = torch.full((N + 1, D), 7., device=DEV).bfloat16()
    _capi.check(L.natsl_narrow_wgrad(P(dy), P(x), P(dw), rows, D, N, _capi.stream_ptr(x.device)), "natsl_narrow_wgrad")
    ref = dy.double().t() @ x.double()
    close = lambda got: bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * rows ** 0.5).all())
    assert close(dw[:N]) and bool((dw[N] == 7).all()) and close(_front._narrow_wgrad(dy, x))
    assert L.natsl_narrow_wgrad(P(dy), P(x), P(dw), rows, D, 65, _capi.stream_ptr(x.device)) != 0
    many = torch.randn(2049, N, device=DEV).bfloat16(), torch.randn(2049, D, device=DEV).bfloat16()
    assert torch.equal(_front._narrow_wgrad(*many), torch.mm(many[0].t(), many[1]))


@pytest.mark.parametrize("rows,D,N", [(1, 32, 2), (31, 96, 12), (257, 130, 17), (2049, 1024, 16), (6000, 1152, 36), (6001, 66, 63), (16385, 64, 44), (20000, 96, 24)])
def test_narrow_weight_gradient_over_many_rows(rows, D, N):
    """natsl_narrow_wgrad_split with fewer steps of 256 tokens than parts, with cut ones, with 8 and 32 parts; and weight_grads, which takes it."""
    from neuralattentionsearchlinear_amd import _capi, _front
    torch.manual_seed(rows)
    L, P = _capi.lib(), _capi.ptr
    x, dy = torch.randn(rows, D, device=DEV).bfloat16(), torch.randn(rows, N, device=DEV).bfloat16()
    dw = torch.full((N + 1, D), 7., device=DEV).bfloat16()
    n = L.natsl_narrow_wgrad_workspace_bytes(rows, D, N)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    call = lambda size, cols: L.natsl_narrow_wgrad_split(P(dy), P(x), P(dw), rows, D, cols, P(ws), size, _capi.stream_ptr(x.device))
    _capi.check(call(n, N), "natsl_narrow_wgrad_split")
    ref = dy.double().t() @ x.double()
    # (one rounding to bf16; fp32 sums of `rows` products of two normal values in any order)
    close = lambda got: bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * rows ** 0.5).all())
    assert close(dw[:N]) and bool((dw[N] == 7).all()) and close(_front.weight_grads(x, [None, dy])[1])
    assert call(n - 1, N) != 0 and call(n, 65) != 0


@pytest.mark.parametrize("width", [8, 16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("what,silu,T", [('rms', 1, 37), ('l2', 0, 9), ('number', 1, 130)])
def test_convolution_with_heads_of_any_width(width, what, silu, T):
    """natsl_conv_norm_* for every head width (lanes of a head within a row of 16 lanes, across rows, a whole wave; four and eight channels a
    thread) and for each of what follows the convolution, against float64 autograd."""
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._front import _ConvSeg
    torch.manual_seed(width + T)
    L, B, D, W = _capi.lib(), 2, 2 * max(width, 48) // width * width, 3
    bf = lambda *s: torch.randn(*s, device=DEV).bfloat16()
    x, w, bias, nw, dy, dn, add = bf(B, T, D), bf(D, 1, W), bf(D), bf(width), bf(B, T, D), bf(B, T, D), bf(B, T, D)
    num = torch.rand(B, T, D // width, device=DEV)
    y, yn, dx = (torch.empty_like(x) for _ in range(3))
    dw, db, dnw, dnum = torch.empty_like(w), torch.empty_like(bias), torch.empty_like(nw), torch.empty_like(num)
    seg = (_ConvSeg * 1)()
    s = seg[0]
    for n, t in dict(x=x, weight=w, bias=bias, y=y, y_norm=yn, dy_a=dy, dy_norm=dn, dx_add=add, dx=dx, dweight=dw, dbias=db).items():
        setattr(s, n, t.data_ptr())
    s.D, s.norm_lanes, s.norm_l2, s.norm_eps = D, width // 8, int(what == 'l2'), 1e-5
    if what == 'rms':
        s.norm_weight, s.dnorm_weight = nw.data_ptr(), dnw.data_ptr()
    if what == 'number':
        s.scale, s.dscale = num.data_ptr(), dnum.data_ptr()
    st = _capi.stream_ptr(x.device)
    _capi.check(L.natsl_conv_norm_fwd(seg, 1, B, T, W, silu, _capi.BF16, st), "natsl_conv_norm_fwd")
    n = L.natsl_conv_norm_bwd_workspace_bytes(seg, 1, B, T, W)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    _capi.check(L.natsl_conv_norm_bwd(seg, 1, B, T, W, silu, _capi.BF16, ws.data_ptr(), n, st), "natsl_conv_norm_bwd")
    x6, w6, b6, nw6, num6 = (t.detach().double().requires_grad_(True) for t in (x, w, bias, nw, num))
    c = torch.nn.functional.conv1d(torch.nn.functional.pad(x6.transpose(1, 2), (W - 1, 0)), w6, b6, groups=D).transpose(1, 2)
    c = torch.nn.functional.silu(c) if silu else c
    r = c + (c.detach().bfloat16().double() - c.detach())                  # (what follows reads the rounded activation)
    h = r.view(B, T, -1, width)
    if what == 'rms':
        o = h * torch.rsqrt((h * h).mean(-1, keepdim=True) + 1e-5) * nw6
    elif what == 'l2':
        o = h * torch.rsqrt((h * h).sum(-1, keepdim=True) + 1e-5)
    else:
        o = h * num6.unsqueeze(-1)
    torch.autograd.backward([c, o.reshape(B, T, D)], [dy.double(), dn.double()])
    # one rounding to bf16 of each result: 2^-9 relative, 2^-8 in the norm with the few activations that fp32 rounds the other way
    for name, got, ref in [('y', y, c), ('follows', yn, o.reshape(B, T, D)), ('dx', dx, x6.grad + add.double()), ('dw', dw, w6.grad), ('db', db, b6.grad)] + \
            ([('dnw', dnw, nw6.grad)] if what == 'rms' else [('dnum', dnum, num6.grad)] if what == 'number' else []):
        assert rel_l2(got.double(), ref.detach()) <= 2 ** -8, (name, rel_l2(got.double(), ref.detach()))


def test_convolution_with_numbers_that_nothing_follows():
    """natsl_conv_norm_bwd with a head's numbers and no gradient of the product: the numbers' is zero, the others are those without numbers."""
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._front import _ConvSeg
    torch.manual_seed(3)
    L, B, T, D, W, width = _capi.lib(), 2, 33, 128, 4, 64
    x, w, dy = torch.randn(B, T, D, device=DEV).bfloat16(), torch.randn(D, 1, W, device=DEV).bfloat16(), torch.randn(B, T, D, device=DEV).bfloat16()
    num, dnum = torch.rand(B, T, D // width, device=DEV), torch.full((B, T, D // width), 7., device=DEV)
    got = []
    for scale in (None, num):
        dx, dw = torch.empty_like(x), torch.empty_like(w)
        seg = (_ConvSeg * 1)()
        s = seg[0]
        for n, t in dict(x=x, weight=w, dy_a=dy, dx=dx, dweight=dw).items():
            setattr(s, n, t.data_ptr())
        s.D = D
        if scale is not None:
            s.norm_lanes, s.scale, s.dscale = width // 8, num.data_ptr(), dnum.data_ptr()
        n = L.natsl_conv_norm_bwd_workspace_bytes(seg, 1, B, T, W)
        ws = torch.empty(n, dtype=torch.uint8, device=DEV)
        _capi.check(L.natsl_conv_norm_bwd(seg, 1, B, T, W, 1, _capi.BF16, ws.data_ptr(), n, _capi.stream_ptr(x.device)), "natsl_conv_norm_bwd")
        got.append((dx, dw))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and not dnum.any()


def _stepwise(monkeypatch):
    """The fused steps one by one instead of the native call."""
    from neuralattentionsearchlinear_amd import _front
    monkeypatch.setattr(_front, '_native_plan', lambda *a: None)


def _train(layer, x0, do):
    x = x0.clone().requires_grad_(True)
    layer.zero_grad(set_to_none=True)
    o = layer(x)
    o = o[0] if isinstance(o, tuple) else o
    o.backward(do)
    return dict({n: p.grad for n, p in layer.named_parameters()}, x=x.grad, out=o.detach(), fraction=layer.attn_fraction)


@pytest.mark.parametrize("kind,geometry,B,T,more", [
    ('gdn', None, 1, 64, {}), ('gdn', '340M', 2, 2113, {}), ('gdn', '760M', 1, 200, dict(allow_neg_eigval=True, conv_bias=True)),
    ('gdn', None, 3, 130, dict(conv_size=3, conv_activation=None, compute_dnats_for_invalid_blocks_attn=True, compute_dnats_for_invalid_blocks_linear_att=True)),
    ('mamba', None, 2, 257, {}), ('mamba', None, 2, 4100, dict(conv_bias=True, conv_size=2)),
    ('gdn', None, 2, 200, dict(ops_for_incomplete_chunks='gated_delta_net')), ('mamba', None, 2, 300, dict(ops_for_incomplete_chunks='mamba'))])
@pytest.mark.parametrize("side,keep", [(False, False), (True, True), (True, False), (None, None)])
def test_native_layer_is_its_steps(kind, geometry, B, T, more, side, keep, monkeypatch):
    """A training step through the native call against the same launches one by one: the streams' and the kept states' switches, sequences that cut a block,
    incomplete blocks for both operators and for the linear one alone."""
    from neuralattentionsearchlinear_amd import _front, _mixed_common
    more = dict(more)
    ops = more.pop('ops_for_incomplete_chunks', 'all')
    layer = _layer(kind, geometry, ops, **more).train()
    torch.manual_seed(T)
    x, do = (torch.randn(B, T, layer.hidden_size, device=DEV).bfloat16() for _ in range(2))
    calls, inner = [], _front._Layer.forward
    monkeypatch.setattr(_front._Layer, 'forward', staticmethod(lambda *a: (calls.append(1), inner(*a))[1]))
    monkeypatch.setattr(_mixed_common, 'CONCURRENT_BRANCHES', side)
    monkeypatch.setattr(_mixed_common, 'SAVE_CHUNK_STATES', keep)
    got = [_train(layer, x, do) for _ in range(2)]
    assert calls == [1, 1]
    other = _layer(kind, geometry, ops, **more).train()
    other.load_state_dict(layer.state_dict())
    _stepwise(monkeypatch)
    want = _train(other, x, do)
    assert calls == [1, 1]
    for g in got:
        for n, b in want.items():
            # the same kernels; the mixing logits' products may be others (a rounding of a bf16 value now and then), and the block types' gradient is
            # summed by atomic additions
            assert g[n].shape == b.shape and g[n].dtype == b.dtype and rel_l2(g[n].float(), b.float()) <= (2e-2 if n == 'nats_layer.weight' else 5e-3), n


@pytest.mark.parametrize("kind,geometry,B,T", [('gdn', '340M', 2, 1999), ('gdn', '760M', 1, 1100), ('gdn', '760M', 4, 1100), ('mamba', None, 3, 700)])
def test_native_layer_takes_the_steps_products(kind, geometry, B, T, monkeypatch):
    """One rule chooses each product, whichever way the layer runs: the same bits in training, as native call and as steps, and in evaluation with
    gradients (always the steps) and without."""
    from neuralattentionsearchlinear_amd import _front
    torch.manual_seed(T)
    layer, other = _layer(kind, geometry, 'all'), _layer(kind, geometry, 'all')
    other.load_state_dict(layer.state_dict())
    x, do = (torch.randn(B, T, layer.hidden_size, device=DEV).bfloat16() for _ in range(2))
    calls, inner = [], _front._Layer.forward
    monkeypatch.setattr(_front._Layer, 'forward', staticmethod(lambda *a: (calls.append(1), inner(*a))[1]))
    native = _train(layer.train(), x, do)
    first = lambda o: o[0] if isinstance(o, tuple) else o
    evaluated = [first(layer.eval()(x))]
    with torch.no_grad():
        evaluated.append(first(layer(x)))
    _stepwise(monkeypatch)
    library, linear = [], _front.F.linear
    monkeypatch.setattr(_front.F, 'linear', lambda a, w, *more: (library.append(w.data_ptr()), linear(a, w, *more))[1])
    steps = _train(other.train(), x, do)
    w = other.nats_out_weights_layer.weight
    assert (w.data_ptr() in library) != bool(_front._capi.lib().natsl_narrow_fwd_pays(B * T, w.shape[1], w.shape[0]))
    assert calls == [1] and evaluated[0].requires_grad and all(torch.equal(native['out'], o) for o in evaluated)
    for n, want in steps.items():
        assert torch.equal(native[n], want), n


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
def test_native_layer_under_autograd(kind, monkeypatch):
    """What autograd asks of the one node: gradients for what wants them only, saved tensors through hooks, a second backward, changed weights
    refused, no graph where nothing wants a gradient."""
    from neuralattentionsearchlinear_amd import _front
    calls, inner = [], _front._Layer.forward
    monkeypatch.setattr(_front._Layer, 'forward', staticmethod(lambda *a: (calls.append(1), inner(*a))[1]))
    layer = _layer(kind, None, 'all').train()
    torch.manual_seed(5)
    x, do = (torch.randn(2, 150, layer.hidden_size, device=DEV).bfloat16() for _ in range(2))
    out = lambda t: (lambda o: o[0] if isinstance(o, tuple) else o)(layer(t))
    want = _train(layer, x, do)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):
        got = _train(layer, x, do)
    for n, b in want.items():
        assert rel_l2(got[n].float(), b.float()) <= (2e-2 if n == 'nats_layer.weight' else 1e-6), n
    assert len(calls) == 2
    layer.zero_grad(set_to_none=True)
    some = {'wo': layer.o_proj.weight, 'wa': layer.a_proj.weight, 'mix': layer.nats_out_weights_layer.weight}
    for p in layer.parameters():
        p.requires_grad_(any(p is s for s in some.values()))
    o = out(x)
    o.backward(do, retain_graph=True)
    first = {n: p.grad.clone() for n, p in some.items()}
    o.backward(do)
    for n, p in layer.named_parameters():
        assert (p.grad is not None) == p.requires_grad
    for n, p in some.items():
        assert rel_l2(p.grad.float(), 2 * first[n].float()) <= 1e-2
    o = out(x)
    with torch.no_grad():
        layer.a_proj.weight.mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(do)
    assert len(calls) == 4
    for p in layer.parameters():
        p.requires_grad_(False)
    assert not out(x).requires_grad
    with torch.no_grad():
        assert torch.equal(out(x), out(x))


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
@pytest.mark.parametrize("train", [('o_proj',), ('o_proj', 'o_norm'), ('nats_out_weights_layer',), ('nats_layer',), ('q_conv1d', 'v_conv1d'), ('A_log', 'dt_bias'),
                                   ('a_proj',), ('g_proj',), ('k_proj', 'o_norm')])
def test_native_layer_of_which_a_part_trains(kind, train, monkeypatch):
    """The gradients of a part of the weights are those of all of them; what is held for them is no more than the steps' nodes hold, and what no
    gradient reads may change before the backward."""
    from neuralattentionsearchlinear_amd import _front
    layer = _layer(kind, None, 'all').train()
    torch.manual_seed(11)
    x, do = (torch.randn(2, 2049, layer.hidden_size, device=DEV).bfloat16() for _ in range(2))
    want = _train(layer, x, do)
    trains = lambda n: n.startswith(train)
    calls, inner = [], _front._Layer.forward
    monkeypatch.setattr(_front._Layer, 'forward', staticmethod(lambda *a: (calls.append(1), inner(*a))[1]))

    def forward(m):
        for n, p in m.named_parameters():
            p.requires_grad_(trains(n))
            p.grad = None
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        o = m(x)
        o = o[0] if isinstance(o, tuple) else o
        return o, torch.cuda.memory_allocated() - before
    o, held = forward(layer)
    assert calls == [1]
    if not any('_proj' in n and n != 'o_proj' for n in train):
        x.add_(1.0)
    if train == ('o_proj',):
        with torch.no_grad():
            layer.q_proj.weight.add_(0.0)
            layer.o_norm.weight1.add_(0.0)
    o.backward(do)
    for n, p in layer.named_parameters():
        assert (p.grad is not None) == trains(n), n
        # (the weight gradients' products share their launch with other ones: fp32 sums of 4098 terms in another order, off by 2^-24 4098^(1/2), so one
        # result in a thousand rounds to the bf16 value next to it, 2^-8 away: 2^-8 1000^(-1/2))
        assert p.grad is None or rel_l2(p.grad.float(), want[n].float()) <= (1.3e-4 if '_proj' in n else 1e-6), n
    del o
    other = _layer(kind, None, 'all').train()
    other.load_state_dict(layer.state_dict())
    _stepwise(monkeypatch)
    _, most = forward(other)
    # (the allocator gives a tensor a block with up to 1 MiB more than it asks for; up to 27 tensors are kept, of 2 MB and more)
    assert calls == [1] and held <= most + most // 2, (held, most)


@pytest.mark.parametrize("kind", ['gdn', 'mamba'])
@pytest.mark.parametrize("train,follow", [
    (('nats_layer',), {'logits'}), (('A_log',), {'g'}), (('dt_bias',), {'g', 'dt', 'v'}), (('g_proj',), {'gate'}), (('k_proj',), {'k', 'ky', 'kn', 'kr'}),
    (('a_proj',), {'g', 'dt', 'v'}), (('q_conv1d',), {'qy', 'qn', 'mix'}), (('nats_out_weights_layer',), {'mix'}), (('v_conv1d',), {'v', 'vr'})])
def test_steps_of_which_a_part_trains(kind, train, follow):
    """Of the fused steps' outputs only those follow a gradient that are made from what trains (qy: the convolution, qn: its norm, qr: attention's view
    where that is the projection, or for v in the delta rule's layer the convolution; v: with dt)."""
    from neuralattentionsearchlinear_amd import _front
    layer = _layer(kind, None, 'all').train()
    for n, p in layer.named_parameters():
        p.requires_grad_(n.startswith(train))
    delta = kind == 'gdn'
    x = torch.randn(2, 130, layer.hidden_size, device=DEV).bfloat16()
    f = _front.fast_front(layer, kind, x, None, None)
    q, k, v, gate, (g, beta, dt), logits = f.project(x, 64, layer.nats_layer)
    qy, ky, vy, qn, kn, mix, qr, kr, vr, _ = f.conv_norm(q, k, v, None, False, None if delta else dt)
    got = dict(gate=gate, g=g, beta=beta, dt=dt, logits=logits, k=k, qy=qy, ky=ky, v=vy, qn=qn, kn=kn, mix=mix, qr=qr, kr=kr, vr=vr)
    if delta:
        follow = follow - {'kr'} - ({'dt', 'v'} if 'dt' in follow else set())
    else:
        follow = follow - {'ky'} - ({'vr'} if train == ('v_conv1d',) else set())
    assert {n for n, t in got.items() if t is not None and t.requires_grad} == follow
    with torch.no_grad():
        if not any(n.endswith('_proj') for n in train):
            x.add_(1.0)                                    # (nothing of the input is read by these gradients)
    outs = [t for n, t in got.items() if n in follow]
    torch.autograd.backward(outs, [torch.randn_like(t) for t in outs])
    for n, p in layer.named_parameters():
        assert (p.grad is not None and bool(p.grad.any())) == n.startswith(train), n


@pytest.mark.parametrize("kind,geometry,heads", [('gdn', '340M', {}), ('mamba', None, dict(hidden_size=512, head_dim=128, expand_v=0.5, num_heads=16, num_attn_heads=16))])
@pytest.mark.parametrize("what", ['train', 'retain', 'eval', 'prompt'])
def test_native_layer_needs_no_more_memory_than_its_steps(kind, geometry, heads, what, monkeypatch):
    """The most that is allocated during a call: the native one drops a tensor behind its last use, as a graph of a node for each step does.  Sizes of
    6 to 12 MB, so that what the allocator rounds up stays below two per cent."""
    torch.manual_seed(1)
    layer = _layer(kind, geometry, 'all', **heads)
    layer.train(what in ('train', 'retain'))
    x = torch.randn(4, 2048, layer.hidden_size, device=DEV).bfloat16().requires_grad_(layer.training)
    do = torch.randn(x.shape, device=DEV).bfloat16()

    def most():
        out = []
        for _ in range(2):                                 # (the first one allocates what is kept for good)
            layer.zero_grad(set_to_none=True)
            x.grad = None
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            if what == 'prompt':
                with torch.no_grad():
                    o = _generate(layer, kind, x, x.shape[1], ())
            else:
                with torch.set_grad_enabled(layer.training):
                    o = layer(x)
                o = o[0] if isinstance(o, tuple) else o
                if layer.training:
                    o.backward(do, retain_graph=what == 'retain')
            torch.cuda.synchronize()
            out.append(torch.cuda.max_memory_allocated() - before)
            del o
        return out[1]
    native = most()
    _stepwise(monkeypatch)
    torch.cuda.empty_cache()
    from neuralattentionsearchlinear_amd import _layer_step
    _layer_step._watches.pop(layer)                        # (its plan has the native form)
    steps = most()
    print(kind, what, native >> 20, steps >> 20)
    assert native <= 1.02 * steps


@pytest.mark.parametrize("kind,T0", [('gdn', 128), ('gdn', 777), ('mamba', 64), ('mamba', 2113)])
@pytest.mark.parametrize("ops", ['all', 'attn', 'linear'])
def test_native_prompt_is_its_steps(kind, T0, ops, monkeypatch):
    """A first prompt through the native calls against the same launches one by one: outputs, what the cache holds, and the tokens behind it."""
    from neuralattentionsearchlinear_amd import _front
    if ops == 'linear':
        ops = 'gated_delta_net' if kind == 'gdn' else 'mamba'
    calls, inner = [], _front.FastFront.prompt
    monkeypatch.setattr(_front.FastFront, 'prompt', lambda *a: (calls.append(1), inner(*a))[1])
    layer = _layer(kind, None, ops)
    torch.manual_seed(T0)
    x = torch.randn(2, T0 + 3, layer.hidden_size, device=DEV).bfloat16()
    fast, cf = _generate(layer, kind, x, T0, (1, 2))
    other = _layer(kind, None, ops)
    other.load_state_dict(layer.state_dict())
    _stepwise(monkeypatch)
    assert calls == [1]
    slow, cs = _generate(other, kind, x, T0, (1, 2))
    assert calls == [1]
    names = ['attn_k', 'attn_v', 'l_attn_k', 'l_attn_v', 'lattn_g', 'lattn_beta', 'recurrent_state', 'recurrent_state_block_start', 'g_cumsum', 'block_type_state']
    for a, b in zip(fast + list(cf.conv_state) + [getattr(cf, n) for n in names], slow + list(cs.conv_state) + [getattr(cs, n) for n in names]):
        assert (a is None) == (b is None) and (a is None or a.shape == b.shape and rel_l2(a.float(), b.float()) <= 2e-3)
    for n in ('n_attn_blocks', 'valid_attn_tokens'):
        assert torch.equal(getattr(cf, n), getattr(cs, n))
    assert rel_l2(layer.last_recurrent_state, other.last_recurrent_state) <= 2e-3
