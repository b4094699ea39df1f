"""What surrounds the mixed operator inside the two layers, as a few fused steps with their backward: the projections of one input,
the short convolutions with the row norms behind them, the gates, the selector, the mixing logits and the output norm-gate.

`fast_front` says whether a forward may take this path: bf16 tensors on the GPU and the layers' own, unhooked submodules.  What it
declines runs through the submodules one by one (the layers' general path).  Per step the saving is passes over [B,T,D] tensors
(gradients that meet at a tensor are added where they are used, norms and mixing softmax ride on their neighbours' passes),
weight-gradient products that split the tokens (natsl_wgrad), and launches.
"""
from __future__ import annotations

import ctypes
import functools

import torch
import torch.nn.functional as F

from . import _capi, _mixed_common
from ._layer_step import _PARAMS, _PLAIN_TENSORS, watch, weight_shapes
from .modules import _NORM_GATE_WIDTHS

_NAMES = [p[0] for p in _PARAMS]
_EITHER = {"norm_q", "norm_k", "a_log", "dt_bias", "out_norm1", "out_norm2"}
_ab_rows = lambda n: -(-n // 32) * 32


class _WgradSeg(ctypes.Structure):
    _fields_ = [("dy", ctypes.c_void_p), ("out", ctypes.c_void_p), ("n", ctypes.c_int32), ("ld", ctypes.c_int32)]


class _ProjectSeg(ctypes.Structure):
    _fields_ = [("y", ctypes.c_void_p), ("w", ctypes.c_void_p), ("n", ctypes.c_int32), ("ld", ctypes.c_int32)]


class _FrontArgs(ctypes.Structure):
    """natsl_front of include/natsl.h."""
    _fields_ = ([(n, ctypes.c_void_p) for n in ("x", "wa", "wb", "wn", "a_log", "dt_bias", "ab", "pooled", "logits", "beta", "wab", "g", "dt")] +
                [(n, ctypes.c_int32) for n in ("B", "T", "D", "NA", "NB", "NL", "ld", "neg_eigval", "param_dtype", "wab_rows")])


class _ConvSeg(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in ("x", "weight", "bias", "state", "norm_weight", "y", "y_norm", "state_out", "dy_a", "dy_b", "dy_norm",
                                                "dx_add", "dx", "dweight", "dbias", "dnorm_weight")] +
                [("D", ctypes.c_int32), ("norm_lanes", ctypes.c_int32), ("norm_l2", ctypes.c_int32), ("norm_eps", ctypes.c_float),
                 ("scale", ctypes.c_void_p), ("dscale", ctypes.c_void_p)])


def _p(t):
    return None if t is None else t.data_ptr()


def weight_grads(x2, dys):
    """[dy_i^T x2 for dy_i [rows, n_i] in dys] (bf16; entries may be None): natsl_wgrad for widths that are multiples of 8, natsl_narrow_wgrad_split
    for narrow ones that are not, or that are alone, else torch."""
    rows, D = x2.shape
    out = [None] * len(dys)
    todo, L = [], _capi.lib()
    alone = sum(dy is not None for dy in dys) == 1
    for i, dy in enumerate(dys):
        if dy is None:
            continue
        if L.natsl_narrow_wgrad_pays(rows, D, dy.shape[1], 0, alone) and x2.data_ptr() % 4 == 0 and dy.dtype == x2.dtype == torch.bfloat16:
            out[i] = torch.empty(dy.shape[1], D, dtype=torch.bfloat16, device=x2.device)
            n = L.natsl_narrow_wgrad_workspace_bytes(rows, D, dy.shape[1])
            ws = torch.empty(n, dtype=torch.uint8, device=x2.device)
            _capi.check(L.natsl_narrow_wgrad_split(dy.data_ptr(), x2.data_ptr(), out[i].data_ptr(), rows, D, dy.shape[1], ws.data_ptr(), n,
                                                   _capi.stream_ptr(x2.device)), "natsl_narrow_wgrad_split")
        elif dy.shape[1] % 8 or D % 8 or x2.data_ptr() % 16 or dy.data_ptr() % 16 or dy.dtype != torch.bfloat16:
            out[i] = torch.mm(dy.t(), x2)
        else:
            out[i] = torch.empty(dy.shape[1], D, dtype=torch.bfloat16, device=x2.device)
            todo.append(i)
    if todo:
        segs = (_WgradSeg * len(todo))()
        for s, i in zip(segs, todo):
            s.dy, s.out, s.n, s.ld = dys[i].data_ptr(), out[i].data_ptr(), dys[i].shape[1], dys[i].shape[1]
        n = L.natsl_wgrad_workspace_bytes(segs, len(todo), rows, D)
        ws = torch.empty(n, dtype=torch.uint8, device=x2.device)
        _capi.check(L.natsl_wgrad(segs, len(todo), x2.data_ptr(), rows, D, D, ws.data_ptr(), n, _capi.stream_ptr(x2.device)), "natsl_wgrad")
    return out


class _Linear(torch.autograd.Function):
    """F.linear with the weight gradient of natsl_wgrad."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return F.linear(x, w)

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.shape[-1]).contiguous()
        dx = torch.mm(dy2, w).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = weight_grads(x.reshape(-1, x.shape[-1]), [dy2])[0] if ctx.needs_input_grad[1] else None
        return dx, dw


def linear(x, w):
    if torch.is_grad_enabled() and (x.requires_grad or w.requires_grad):
        return _Linear.apply(x, w)
    return F.linear(x, w)


# ---- the projections of one input -----------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=512)
def _joint_pays(rows, D, widths, cus):
    """Whether one launch for all projections (natsl_project) beats the library's products one by one: where it takes fewer rounds of
    256 x 256 tiles over the CUs.  Measured (one by one / joint, us): 340M geometry 8 x 4096 tokens, 10 / 9 rounds: 267 / 260, 1 x 777,
    4 / 1: 39 / 17; 760M 8 x 2048, 10 / 7: 337 / 288, 1 x 4096, 4 / 2: 99 / 79; but Mamba 4 x 8192, 12 / 12: 341 / 350, 760M 8 x 8192, 28 / 28:
    1065 / 1187.  From inputs wider than 1536 on a round of the library's is the shorter one (2048 columns in, 9216 out, 16384 tokens, 10 / 9:
    461 / 502, 4096 tokens, 4 / 3: 138 / 141, 12000, 10 / 7: 407 / 390): there at most seven tenths of its rounds."""
    tiles = [-(-rows // 256) * -(-n // 256) for n in widths]
    joint, alone = -(-sum(tiles) // cus), sum(-(-t // cus) for t in tiles)
    return D % 32 == 0 and D >= 128 and all(n % 8 == 0 for n in widths) and (joint < alone if D <= 1536 else 0 < 10 * joint <= 7 * alone)


def _project_segs(ys, ws):
    segs = (_ProjectSeg * len(ys))()
    for s, y, w in zip(segs, ys, ws):
        s.y, s.w, s.n, s.ld = y.data_ptr(), w.data_ptr(), w.shape[0], y.shape[-1]
    return segs


def _on_16(*tensors):
    return not any(t.data_ptr() & 15 for t in tensors)


def _wide(x, ws):
    """[F.linear(x, w) for w in ws]"""
    D = x.shape[-1]
    rows = x.numel() // D
    cus = torch.cuda.get_device_properties(x.device).multi_processor_count
    if not _joint_pays(rows, D, tuple([w.shape[0] for w in ws]), cus) or not _on_16(x, *ws):
        return [F.linear(x, w) for w in ws]
    ys = [torch.empty(*x.shape[:-1], w.shape[0], dtype=x.dtype, device=x.device) for w in ws]
    _capi.check(_capi.lib().natsl_project(_project_segs(ys, ws), len(ws), x.data_ptr(), rows, D, D, _capi.stream_ptr(x.device)), "natsl_project")
    return ys


def _narrow(f, x, want_selector, keep):
    """The narrow products of one input, the gates behind them and the selector's logits over the means of 64 tokens, one pass over x:
    -> (g fp32, beta bf16 or None, dt fp32 or None [B,T,H], logits [B,TN,NL] or None, what the backward needs, each where `keep` says so: (a and b of
    every token, their joint weight in whole stages of 32 rows, the block means)).  As separate products and passes it is four launches, two of them the
    library's (340M geometry, 8 x 4096 tokens: 36 -> 24 us; 1 x 777 25 -> 9)."""
    B, T, D = x.shape
    w, H, dev = f.w, f.H, x.device
    wb = w["wb"] if f.delta else None
    a = _FrontArgs()
    a.B, a.T, a.D, a.NA, a.NB, a.neg_eigval, a.param_dtype = B, T, D, H, H if f.delta else 0, f.neg, f.gate_dtype
    g = torch.empty(B, T, H, dtype=torch.float32, device=dev)
    beta = torch.empty(B, T, H, dtype=torch.bfloat16, device=dev) if f.delta else None
    dt = None if f.delta else torch.empty_like(g)
    logits = pooled = ab = wab = None
    if want_selector:
        nb = -(-T // 64)
        logits = torch.empty(B, nb, f.wn.shape[0], dtype=torch.bfloat16, device=dev)
        a.wn, a.logits, a.NL = f.wn.data_ptr(), logits.data_ptr(), f.wn.shape[0]
        if keep[2]:
            pooled = torch.empty(B, nb, D, dtype=torch.bfloat16, device=dev)
            a.pooled = pooled.data_ptr()
    if keep[0]:
        a.ld = _ab_rows(a.NA + a.NB)
        ab = torch.empty(B, T, a.ld, dtype=torch.bfloat16, device=dev)
        a.ab = ab.data_ptr()
    if keep[1]:
        a.wab_rows = _ab_rows(a.NA + a.NB)
        wab = torch.empty(a.wab_rows, D, dtype=torch.bfloat16, device=dev)
        a.wab = wab.data_ptr()
    a.x, a.wa, a.wb, a.a_log, a.dt_bias = x.data_ptr(), w["wa"].data_ptr(), _p(wb), w["a_log"].data_ptr(), w["dt_bias"].data_ptr()
    a.g, a.beta, a.dt = g.data_ptr(), _p(beta), _p(dt)
    _capi.check(_capi.lib().natsl_layer_front(ctypes.byref(a), _capi.stream_ptr(dev)), "natsl_layer_front")
    return g, beta, dt, logits, (ab, wab, pooled)


def _only_for(ctx, *outputs):
    """Marks the outputs (tensor or None, whether an input that it is made from wants a gradient) for which nothing behind them has to run backwards."""
    ctx.mark_non_differentiable(*[t for t, wanted in outputs if t is not None and not wanted])


def _project(x, wq, wk, wv, wg, wa, wb, pool_block, whole=16):
    """-> ((q, k, v, gate, ab, block means or None), the joint weight of a and b).  The narrow projections share one product: their
    rows and, where these are no multiple of `whole`, enough others to make whole stages of 32 (the columns behind a and b are never read)."""
    narrow = (wa,) if wb is None else (wa, wb)
    used = sum(w.shape[0] for w in narrow)
    wab = torch.cat(narrow + (wq[:_ab_rows(used) - used],)) if used % whole else torch.cat(narrow) if len(narrow) > 1 else wa
    pooled = None
    if pool_block:
        from .nats_util import _mean_pooling_fwd
        pooled = _mean_pooling_fwd(x.unsqueeze(-2), pool_block, None).squeeze(-2)
    return (*_wide(x, (wq, wk, wv, wg)), F.linear(x, wab), pooled), wab


def _project_bwd(x, wide, wab, n_a, n_b, dys, dpool, block, needs):
    """dx and the weights' gradients (wq, wk, wv, wg, wa, wb) of the projections of one input: dx is one launch (natsl_project_bwd), or starts as what
    is no wide product (natsl_dx_init) and the wide ones accumulate onto it; all weight gradients are one launch.  dys: gradients of the four wide
    outputs and of the joint narrow one, dpool: of the block means; each may be None.  needs: x, then the six weights."""
    B, T, D = x.shape
    rows = B * T
    wq, wk, wv, wg = wide
    dys = [None if t is None else t.reshape(rows, t.shape[-1]).contiguous() for t in dys]
    dx = None
    if needs[0]:
        dx = torch.empty_like(x)
        dp = None if dpool is None else dpool.contiguous()
        some = [(dy, w) for dy, w in zip(dys, (wq, wk, wv, wg, wab)) if dy is not None]
        segs = _project_segs(*zip(*some)) if some else None
        joint = _capi.lib().natsl_project_bwd_takes(segs, len(some), _p(dp), dx.data_ptr())
    if needs[0] and joint:
        # one pass over dx where four accumulating products and dx_init made five (340M geometry, 8 x 4096 tokens: 342 -> 237 us, 1 x 777
        # 56 -> 49).  Below some 500 tokens the one launch takes longer than the five (760M, 128 tokens: 54 / 68), but a step is the host's
        # there, which issues one for five: the layer at 760M, 300 tokens 1.45 -> 1.2 ms
        rc = _capi.lib().natsl_project_bwd(segs, len(some), _p(dp), dx.data_ptr(), B, T, D, block or T,
                                           _capi.stream_ptr(x.device))
        _capi.check(rc, "natsl_project_bwd")
    elif needs[0]:
        n = 0 if dys[4] is None else wab.shape[0]
        rc = _capi.lib().natsl_dx_init(_p(dys[4]), wab.data_ptr(), _p(dp), dx.data_ptr(), B, T, D, n, max(n, 16), block or T,
                                       _capi.stream_ptr(x.device))
        _capi.check(rc, "natsl_dx_init")
        dx2 = dx.view(rows, D)
        for dy, w in zip(dys, wide):
            if dy is not None:
                dx2.addmm_(dy, w)
    wants = [needs[1], needs[2], needs[3], needs[4], needs[5] or needs[6]]
    dws = weight_grads(x.view(rows, D), [dy if want else None for dy, want in zip(dys, wants)])
    da = db = None
    if dws[4] is not None:
        da = dws[4][:n_a]
        db = dws[4][n_a:n_a + n_b] if n_b else None
    return dx, dws[0], dws[1], dws[2], dws[3], da, db


class _Project(torch.autograd.Function):
    """The projections with the block means (selector blocks of other than 64 tokens, and widths that natsl_layer_front does not take)."""

    @staticmethod
    def forward(ctx, x, wq, wk, wv, wg, wa, wb, pool_block):
        # natsl_project_bwd takes whole stages: sixteen heads' one narrow projection is filled up for it, one more launch here (training step of
        # the Mamba layer, 8 x 4096 tokens 4342 -> 4218 us, 3 x 3001 1690 -> 1605)
        out, wab = _project(x, wq, wk, wv, wg, wa, wb, pool_block, 32 if ctx.needs_input_grad[0] else 16)
        ctx.save_for_backward(x, wq, wk, wv, wg, wab)
        ctx.block, ctx.n_a, ctx.n_b = pool_block, wa.shape[0], 0 if wb is None else wb.shape[0]
        ctx.set_materialize_grads(False)
        return out

    @staticmethod
    def backward(ctx, dq, dk, dv, dg, dab, dpool):
        x, wq, wk, wv, wg, wab = ctx.saved_tensors
        return (*_project_bwd(x, (wq, wk, wv, wg), wab, ctx.n_a, ctx.n_b, (dq, dk, dv, dg, dab), dpool, ctx.block, ctx.needs_input_grad), None)


class _ProjectAll(torch.autograd.Function):
    """The projections, the gates behind the narrow ones and the selector's logits (f.wn: the selector's weight, or None without them)."""

    @staticmethod
    def forward(ctx, f, x, wq, wk, wv, wg, wa, wb, wn, a_log, dt_bias):
        _, nx, nq, nk, nv, ng, na, nb, nn, nal, ndt = ctx.needs_input_grad
        gates = nx or na or nb or nal or ndt
        g, beta, dt, logits, (ab, wab, pooled) = _narrow(f, x, wn is not None, (gates, nx, nn))
        q, k, v, gate = _wide(x, (wq, wk, wv, wg))
        ctx.f = f
        only = lambda on, *ts: ts if on else (None,) * len(ts)
        ctx.save_for_backward(*only(any(ctx.needs_input_grad[1:8]), x), *only(nx, wq, wk, wv, wg, wab), ab, pooled, *only(nx, wn), *only(gates, a_log, dt_bias))
        ctx.set_materialize_grads(False)
        _only_for(ctx, (q, nx or nq), (k, nx or nk), (v, nx or nv), (gate, nx or ng), (g, nx or na or nal or ndt), (beta, nx or nb), (dt, nx or na or ndt),
                  (logits, nx or nn))
        return q, k, v, gate, g, beta, dt, logits

    @staticmethod
    def backward(ctx, dq, dk, dv, dgate, dg, dbeta, ddt, dlogits):
        f, need = ctx.f, ctx.needs_input_grad
        x, wq, wk, wv, wg, wab, ab, pooled, wn, a_log, dt_bias = ctx.saved_tensors
        dab = da_log = ddt_bias = dpool = dwn = None
        if dg is not None or dbeta is not None or ddt is not None:
            dab, da_log, ddt_bias = _gates_bwd(f, ab, dg, dbeta, ddt)
        if dlogits is not None:
            dl = dlogits.reshape(-1, dlogits.shape[-1]).contiguous()
            if need[1]:
                dpool = _narrow_bwd(dl, wn, few=True).view(*dlogits.shape[:2], -1)
            if need[8]:
                dwn = _narrow_wgrad(dl, pooled.view(-1, pooled.shape[-1]))
        dx, dws = None, (None,) * 6
        if x is not None:
            dx, *dws = _project_bwd(x, (wq, wk, wv, wg), wab, f.H, f.H if f.delta else 0, (dq, dk, dv, dgate, dab), dpool, 64, need[1:8])
        return (None, dx, *dws, dwn, da_log, ddt_bias)


# ---- a narrow weight: the mixing logits' layer ------------------------------------------------------------------------------------
def _narrow_pays(rows, N, D):
    """Whether natsl_narrow_linear_bwd forms dy [rows, N] w [N, D]."""
    return bool(_capi.lib().natsl_narrow_linear_bwd_pays(rows, D, N, 0))


def _narrow_bwd(dy, w, few=False):
    """dy [rows, N] w.  few: the selector's, over the block means."""
    N, D = w.shape
    if not _capi.lib().natsl_narrow_linear_bwd_pays(dy.shape[0], D, N, few) or not _on_16(dy, w):
        return torch.mm(dy, w)
    dx = torch.empty(dy.shape[0], D, dtype=dy.dtype, device=dy.device)
    _capi.check(_capi.lib().natsl_narrow_linear_bwd(dy.data_ptr(), w.data_ptr(), dx.data_ptr(), dy.shape[0], D, N, _capi.stream_ptr(dy.device)),
                "natsl_narrow_linear_bwd")
    return dx


def _narrow_wgrad(dy, x):
    """dy [rows, N]^T x [rows, D] over the block means"""
    rows, N = dy.shape
    D = x.shape[1]
    if not _capi.lib().natsl_narrow_wgrad_pays(rows, D, N, 1, 0) or x.data_ptr() % 4:
        return torch.mm(dy.t(), x)
    dw = torch.empty(N, D, dtype=dy.dtype, device=dy.device)
    _capi.check(_capi.lib().natsl_narrow_wgrad(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), rows, D, N, _capi.stream_ptr(dy.device)), "natsl_narrow_wgrad")
    return dw


def _mix_logits(yq, w):
    """yq [B, T, D] w^T [B, T, N]"""
    B, T, D = yq.shape
    if not _capi.lib().natsl_narrow_fwd_pays(B * T, D, w.shape[0]) or not _on_16(yq, w):
        return F.linear(yq, w)
    y = torch.empty(B, T, w.shape[0], dtype=torch.bfloat16, device=yq.device)
    a = _FrontArgs()
    a.x, a.wa, a.ab = yq.data_ptr(), w.data_ptr(), y.data_ptr()
    a.B, a.T, a.D, a.NA, a.ld, a.param_dtype = 1, B * T, D, w.shape[0], w.shape[0], _capi.BF16
    _capi.check(_capi.lib().natsl_layer_front(ctypes.byref(a), _capi.stream_ptr(yq.device)), "natsl_layer_front")
    return y


# ---- convolutions, norms, mixing logits --------------------------------------------------------------------------------------------
def _conv_segs(f, raw, dt=None):
    """The segments of natsl_conv_norm_*: q, k, v with their weights; f: the layer's FastFront; dt: what conv(v)'s heads are multiplied by, or None."""
    segs = (_ConvSeg * 3)()
    for s, x, n in zip(segs, raw, "qkv"):
        s.x, s.D, s.weight, s.bias = x.data_ptr(), x.shape[-1], _p(f.w["conv_w" + n]), _p(f.w["conv_b" + n])
        if n == "v" and dt is not None:
            s.norm_lanes, s.scale = x.shape[-1] // f.H // 8, dt.data_ptr()
        if n != "v":
            s.norm_lanes, s.norm_l2, s.norm_eps = f.norm_width // 8, int(f.l2), f.front_eps
            s.norm_weight = None if f.l2 else f.w["norm_" + n].data_ptr()
    return segs


def _conv_norm(f, raw, states, want_states, dt=None):
    """-> (conv(q) or None, conv(k) or None, conv(v) (times dt), normed q, normed k, new states)."""
    B, T, _ = raw[0].shape
    segs = _conv_segs(f, raw, dt)
    ys = [torch.empty_like(raw[0]), None if f.l2 else torch.empty_like(raw[1]), torch.empty_like(raw[2])]
    ns = [torch.empty_like(raw[0]), torch.empty_like(raw[1])]
    new = None
    if want_states:
        new = tuple([torch.empty(B, x.shape[-1], f.W, dtype=torch.bfloat16, device=x.device) for x in raw])
    for i, s in enumerate(segs):
        if i < 2 or dt is None:
            s.y = _p(ys[i])
        else:
            s.y_norm = ys[i].data_ptr()
        if i < 2:
            s.y_norm = ns[i].data_ptr()
        if states is not None and states[i] is not None:
            s.state = states[i].data_ptr()
        if new is not None:
            s.state_out = new[i].data_ptr()
    _capi.check(_capi.lib().natsl_conv_norm_fwd(segs, 3, B, T, f.W, f.act, f.norm_dtype, _capi.stream_ptr(raw[0].device)), "natsl_conv_norm_fwd")
    return ys, ns, new


class _ConvNorm(torch.autograd.Function):
    """(q, k, v projections) -> (conv(q), conv(k), conv(v) (times dt where that is given), normed q, normed k, mixing logits, and what attention takes:
    the projections themselves, or only conv(v) once more); the last three only carry attention's gradient to where it is added (dx_add, dy_b)."""

    @staticmethod
    def forward(ctx, f, q, k, v, wq, bq, wk, bk, wv, bv, nq, nk, w_mix, dt):
        ys, ns, _ = _conv_norm(f, (q, k, v), None, False, dt)
        ctx.f = f
        # (the parameters are saved for the check that nobody changes them before the backward reads them through f)
        ctx.save_for_backward(q, k, v, ys[0], w_mix, dt, wq, bq, wk, bk, wv, bv, nq, nk)
        ctx.set_materialize_grads(False)
        raw = tuple(t.view(t.shape) for t in (q, k, v)) if f.raw_attention else (None, None, ys[2].detach())
        _, nq_, nk_, nv_, *nw, nnq, nnk, nmix, ndt = ctx.needs_input_grad
        cq, ck, cv = nq_ or nw[0] or nw[1], nk_ or nw[2] or nw[3], nv_ or nw[4] or nw[5]
        mix = _mix_logits(ys[0], w_mix)
        _only_for(ctx, (ys[0], cq), (ys[1], ck), (ys[2], cv or ndt), (ns[0], cq or nnq), (ns[1], ck or nnk), (mix, cq or nmix),
                  *zip(raw, (nq_, nk_, nv_ if f.raw_attention else cv)))
        return (ys[0], ys[1], ys[2], ns[0], ns[1], mix) + raw

    @staticmethod
    def backward(ctx, dq, dk, dv, dqn, dkn, dlogits, dq_raw, dk_raw, dv_raw):
        f = ctx.f
        q, k, v, yq, w_mix, dt = ctx.saved_tensors[:6]
        B, T, _ = q.shape
        dev = q.device
        dw_mix = dq_mix = None
        if dlogits is not None:
            d2 = dlogits.reshape(B * T, -1).contiguous()
            dq_mix = _narrow_bwd(d2, w_mix)
            dw_mix = weight_grads(yq.view(B * T, -1), [d2])[0]
        hold = []

        def at(t):
            if t is None:
                return None
            t = t.contiguous()
            hold.append(t)
            return t.data_ptr()
        segs = _conv_segs(f, (q, k, v), dt)
        dv_conv = dv_scaled = ddt = None
        if not f.raw_attention:
            dv_conv, dv_raw = dv_raw, None
        if dt is not None:
            dv, dv_scaled = None, dv
            if dv_scaled is not None and ctx.needs_input_grad[13]:
                ddt = torch.empty_like(dt)
                segs[2].dscale = ddt.data_ptr()
        grads = []
        for s, x, n, da, db, dn, add in zip(segs, (q, k, v), "qkv", (dq, dk, dv), (dq_mix, None, dv_conv), (dqn, dkn, dv_scaled), (dq_raw, dk_raw, dv_raw)):
            w, b = f.w["conv_w" + n], f.w["conv_b" + n]
            dx, dw = torch.empty_like(x), torch.empty_like(w)
            dbias = None if b is None else torch.empty_like(b)
            dnorm = torch.empty_like(f.w["norm_" + n]) if n != "v" and not f.l2 else None
            s.dy_a, s.dy_b, s.dy_norm, s.dx_add = at(da), at(db), at(dn), at(add)
            s.dx, s.dweight, s.dbias, s.dnorm_weight = dx.data_ptr(), dw.data_ptr(), _p(dbias), _p(dnorm)
            if dn is None and dnorm is not None:
                dnorm.zero_()
            grads.append((dx, dw, dbias, dnorm))
        L = _capi.lib()
        n = L.natsl_conv_norm_bwd_workspace_bytes(segs, 3, B, T, f.W)
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        _capi.check(L.natsl_conv_norm_bwd(segs, 3, B, T, f.W, f.act, f.norm_dtype, ws.data_ptr(), n, _capi.stream_ptr(dev)), "natsl_conv_norm_bwd")
        (dxq, dwq, dbq, dnq), (dxk, dwk, dbk, dnk), (dxv, dwv, dbv, _) = grads
        return None, dxq, dxk, dxv, dwq, dbq, dwk, dbk, dwv, dbv, dnq, dnk, dw_mix, ddt


# ---- gates ---------------------------------------------------------------------------------------------------------------------------
def _gates(f, ab):
    """-> (g fp32, beta bf16 or None, dt fp32 or None), each [B,T,H]."""
    B, T, ld = ab.shape
    g = torch.empty(B, T, f.H, dtype=torch.float32, device=ab.device)
    beta = torch.empty(B, T, f.H, dtype=torch.bfloat16, device=ab.device) if f.delta else None
    dt = None if f.delta else torch.empty_like(g)
    rc = _capi.lib().natsl_gates_fwd(ab.data_ptr(), f.w["a_log"].data_ptr(), f.w["dt_bias"].data_ptr(), g.data_ptr(), _p(beta), _p(dt), B * T, f.H, ld,
                                     f.neg, f.gate_dtype, _capi.stream_ptr(ab.device))
    _capi.check(rc, "natsl_gates_fwd")
    return g, beta, dt


def _gates_bwd(f, ab, dg, dbeta, ddt):
    """-> gradients of ab, A_log, dt_bias; each of the three may be None."""
    B, T, ld = ab.shape
    c = lambda t, dt: None if t is None else t.to(dt).contiguous()
    dg, dbeta, ddt = c(dg, torch.float32), c(dbeta, torch.bfloat16), c(ddt, torch.float32)
    dab = torch.empty_like(ab)
    da_log, ddt_bias = torch.empty_like(f.w["a_log"]), torch.empty_like(f.w["dt_bias"])
    L = _capi.lib()
    n = L.natsl_gates_bwd_workspace_bytes(B * T, f.H)
    ws = torch.empty(n, dtype=torch.uint8, device=ab.device)
    rc = L.natsl_gates_bwd(ab.data_ptr(), f.w["a_log"].data_ptr(), f.w["dt_bias"].data_ptr(), _p(dg), _p(dbeta), _p(ddt), int(f.delta), dab.data_ptr(),
                           da_log.data_ptr(), ddt_bias.data_ptr(), ws.data_ptr(), n, B * T, f.H, ld, f.neg, f.gate_dtype,
                           _capi.stream_ptr(ab.device))
    _capi.check(rc, "natsl_gates_bwd")
    return dab, da_log, ddt_bias


class _Gates(torch.autograd.Function):
    @staticmethod
    def forward(ctx, f, ab, a_log, dt_bias):
        ctx.f = f
        ctx.save_for_backward(ab, a_log, dt_bias)
        ctx.set_materialize_grads(False)
        return _gates(f, ab)

    @staticmethod
    def backward(ctx, dg, dbeta, ddt):
        return (None, *_gates_bwd(ctx.f, ctx.saved_tensors[0], dg, dbeta, ddt))


# ---- output norm-gate with the mixing logits -------------------------------------------------------------------------------------------
def _tail(f, o_lin, o_attn, gate, logits):
    y = torch.empty_like(o_attn)
    D = o_attn.shape[-1]
    rc = _capi.lib().natsl_norm_gate_logits_fwd(o_lin.data_ptr(), o_attn.data_ptr(), gate.data_ptr(), logits.data_ptr(), f.w["out_norm1"].data_ptr(),
                                                f.w["out_norm2"].data_ptr(), y.data_ptr(), o_attn.numel() // D, D, _capi.BF16, f.out_eps, f.out_dtype,
                                                _capi.stream_ptr(y.device))
    _capi.check(rc, "natsl_norm_gate_logits_fwd")
    return y


class _Tail(torch.autograd.Function):
    @staticmethod
    def forward(ctx, f, o_lin, o_attn, gate, logits, w1, w2):
        ctx.f = f
        ctx.save_for_backward(o_lin, o_attn, gate, logits, w1, w2)
        return _tail(f, o_lin, o_attn, gate, logits)

    @staticmethod
    def backward(ctx, dy):
        f = ctx.f
        a, b, g, lg = ctx.saved_tensors[:4]
        D = b.shape[-1]
        rows = b.numel() // D
        dy = dy.contiguous()
        w1, w2 = f.w["out_norm1"], f.w["out_norm2"]
        da, db, dg, dl = torch.empty_like(a), torch.empty_like(b), torch.empty_like(g), torch.empty_like(lg)
        dw = torch.empty(2, D, dtype=torch.float32, device=a.device)
        L = _capi.lib()
        n = L.natsl_norm_gate_bwd_workspace_bytes(rows, D)
        ws = torch.empty(n, dtype=torch.uint8, device=a.device)
        rc = L.natsl_norm_gate_logits_bwd(a.data_ptr(), b.data_ptr(), g.data_ptr(), lg.data_ptr(), w1.data_ptr(), w2.data_ptr(), dy.data_ptr(),
                                          da.data_ptr(), db.data_ptr(), dg.data_ptr(), dl.data_ptr(), dw.data_ptr(), dw.data_ptr() + 4 * D,
                                          ws.data_ptr(), n, rows, D, _capi.BF16, f.out_eps, f.out_dtype, _capi.stream_ptr(a.device))
        _capi.check(rc, "natsl_norm_gate_logits_bwd")
        dw = dw.to(w1.dtype)
        return None, da, db, dg, dl, dw[0], dw[1]


# ---- selector ------------------------------------------------------------------------------------------------------------------------
def _select(logits, want_raw):
    """-> (types with the last block forced, counts, attention's share per head, types before that or None)."""
    logits = logits.contiguous()
    B, TN, HN, _ = logits.shape
    types, raw = torch.empty_like(logits), torch.empty_like(logits) if want_raw else None
    counts = torch.empty(B, HN, 2, dtype=torch.int32, device=logits.device)
    fraction = torch.empty(HN, dtype=torch.float32, device=logits.device)
    rc = _capi.lib().natsl_layer_select(logits.data_ptr(), types.data_ptr(), _p(raw), counts.data_ptr(), fraction.data_ptr(), B, TN, HN,
                                        _capi.dtype_code(logits.dtype), _capi.stream_ptr(logits.device))
    _capi.check(rc, "natsl_layer_select")
    return types, counts, fraction, raw


class _Select(torch.autograd.Function):
    """Hard selection with the straight-through gradient; the last block, forced to both ops, has none."""

    @staticmethod
    def forward(ctx, logits, want_raw):
        types, counts, fraction, raw = _select(logits.detach(), want_raw)
        ctx.save_for_backward(logits)
        ctx.mark_non_differentiable(counts, fraction, *((raw,) if want_raw else ()))
        ctx.set_materialize_grads(False)               # (zeros for the counts and shares would be two launches)
        return types, counts, fraction, raw

    @staticmethod
    def backward(ctx, dtypes, *_):
        if dtypes is None:
            return None, None
        (logits,) = ctx.saved_tensors
        lg, d = logits.contiguous(), dtypes.to(logits.dtype).contiguous()
        out = torch.empty_like(lg)
        B, TN, HN, _ = lg.shape
        rc = _capi.lib().natsl_hard_select_bwd(lg.data_ptr(), d.data_ptr(), out.data_ptr(), B, TN, HN, _capi.dtype_code(lg.dtype), 1,
                                               _capi.stream_ptr(lg.device))
        _capi.check(rc, "natsl_hard_select_bwd")
        return out, None


# ---- a layer as one call each way -------------------------------------------------------------------------------------------------------
class _Layer(torch.autograd.Function):
    """A layer's training forward and its backward, one native call each (csrc/host/layer_core.cpp): what FastFront's steps and the mixed operator's
    autograd function launch, in that order, without an autograd node, a Python call and an allocation for each."""

    @staticmethod
    def forward(ctx, f, flags, x, *weights):
        side, joint, states = flags
        out, fraction, kept = _capi.step_core().layer_train(f.native, x, weights, _capi.stream_ptr(x.device), side, joint, ctx.needs_input_grad[2:], states)
        ctx.native, ctx.how = f.native, f.how
        ctx.save_for_backward(*kept)
        ctx.mark_non_differentiable(fraction)
        ctx.set_materialize_grads(False)
        return out, fraction

    @staticmethod
    def backward(ctx, dout, _):
        if dout is None:
            return (None,) * len(ctx.needs_input_grad)
        stream = _capi.stream_ptr(dout.device)
        kept = list(ctx.saved_tensors)
        ctx.maybe_clear_saved_tensors()                    # (not where the graph is retained; nodes of their own are freed one by one, too)
        grads = _capi.step_core().layer_backward(
            ctx.native, dout.to(torch.bfloat16), kept, ctx.needs_input_grad[2:], stream, _beside(dout, ctx.how, stream, True), ctx.how["invalid_attn"],
            ctx.how["invalid_linear"])
        return (None, None, *grads)


def _beside(x, how, stream, gradients):
    """The stream of the softmax branch: the side stream, or the caller's."""
    if _mixed_common._layer_runs_side_by_side(x.device, x.shape[0], x.shape[1], how, gradients):
        return _mixed_common._get_attn_stream(x.device).cuda_stream
    return stream


def _native_plan(layer, kind, constants, w, wn):
    """(what csrc/host/layer_core.cpp keeps of a layer, the sizes used here), or None where it is not built for the layer."""
    delta, dev = constants["delta"], w["wq"].device
    H, K, V, HQ = layer.num_heads, layer.head_k_dim, layer.head_v_dim, layer.num_attn_heads
    KA, VA, HN, D = layer.head_attn_k_dim, layer.head_attn_v_dim, layer.num_nats_head, layer.hidden_size
    if layer.nats_block_size != 64 or D % 32 or (1 + delta) * H > 32 or K not in (64, 128, 192) or V % 64 or KA not in (64, 128) or VA not in (64, 128) or \
            HQ * KA != H * K or HQ * VA != H * V or HQ % HN or H % HN or not (delta or constants["takes_dt"] and not layer.attn_qk_norm):
        return None
    if not _on_16(*[t for t in w.values() if t is not None]):
        return None
    ops = layer.ops_for_incomplete_chunks
    decay = layer.decay_for_non_gdn_blocks if delta else layer.decay_for_non_mamba_blocks
    if ops not in ('all', 'attn', 'gated_delta_net' if delta else 'mamba'):
        return None
    L, c = _capi.lib(), constants
    core = _capi.step_core().make_layer(
        L._handle, _capi.check,
        (dev.index, int(delta), D, H, K, V, HQ, KA, VA, HN, wn.shape[0], c["W"], c["act"], c["norm_width"], c["norm_dtype"], c["gate_dtype"], c["out_dtype"],
         c["neg"], int(decay), int(ops in ('all', 'attn')), int(ops != 'attn')),
        (c["front_eps"], c["out_eps"], KA ** -0.5, K ** -0.5 if delta else 1.0))
    return core, dict(H=H, K=K, V=V, widths=(w["wq"].shape[0], w["wk"].shape[0], w["wv"].shape[0], w["wg"].shape[0]), D=D,
                      cus=torch.cuda.get_device_properties(dev).multi_processor_count)


class FastFront:
    """A layer's parameters at one forward, with the constants of its plan.  (The plan, which outlives the forward, holds no tensor.)"""

    def __init__(self, constants, w, wn):
        self.__dict__.update(constants)
        self.w, self.wn, self.native = w, wn, None

    def _call(self, x, gradients=False):
        """-> (stream, the softmax branch's stream, whether the wide projections are one launch)."""
        how, rows = self.how, x.shape[0] * x.shape[1]
        stream = _capi.stream_ptr(x.device)
        return stream, _beside(x, how, stream, gradients), _joint_pays(rows, how["D"], how["widths"], how["cus"])

    def train(self, x):
        """The layer's training forward on whole sequences (`native` only) -> (output, attention's share per head)."""
        weights = (*self.w.values(), self.wn)
        gradients = self.grad(x, *weights)
        stream, side, joint = self._call(x, gradients)
        if gradients:
            how = self.how
            states = _mixed_common._keep_states_of(x.shape[0], x.shape[0], x.shape[1], how["H"], how["K"], how["V"])
            return _Layer.apply(self, (side, joint, states), x, *weights)
        return _capi.step_core().layer_train(self.native, x, weights, stream, side, joint, None, False)[:2]

    def prompt(self, x, seen):
        """The layer's forward outside of training (`native` only, no gradients).  seen: None, or a call that gets the blocks' types as soon as they are
        enqueued -> (output, attention's share per head, None or what a cache keeps: types before the last block was forced, (k, v) of attention,
        (k, v, beta, g) of the linear branch, convolution states, final state, the state that entered the last block, sum of g over it)."""
        weights, core = (*self.w.values(), self.wn), _capi.step_core()
        stream, side, joint = self._call(x)
        front = core.layer_front(self.native, x, weights, stream)
        if seen is not None:
            seen(front[5])
        out, ka, va, kl, vl, cq, ck, cv, ht, hs, gs = core.layer_rest(self.native, x, weights, front, stream, side, joint, seen is not None)
        return out, front[7], None if seen is None else (front[5], (ka, va), (kl, vl, front[1], front[0]), (cq, ck, cv), ht, hs, gs)

    def grad(self, *tensors):
        return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)

    def project(self, x, pool_block, selector):
        """-> (q, k, v, gate, (g, beta, dt), selector logits or None without pool_block); selector: the layer's own product behind the means."""
        w = self.w
        wb = w["wb"] if self.delta else None
        narrow = (1 + self.delta) * self.H
        if x.shape[-1] % 32 == 0 and narrow <= (32 if pool_block else 64) and (not pool_block or pool_block == 64 and self.wn is not None) and \
                _on_16(x, w["wa"], *([] if wb is None else [wb]), *([self.wn] if pool_block else [])):
            wide, wn = (w["wq"], w["wk"], w["wv"], w["wg"]), self.wn if pool_block else None
            if self.grad(x, *wide, w["wa"], wb, wn, w["a_log"], w["dt_bias"]):
                q, k, v, gate, g, beta, dt, logits = _ProjectAll.apply(self, x, *wide, w["wa"], wb, wn, w["a_log"], w["dt_bias"])
            else:
                g, beta, dt, logits, _ = _narrow(self, x, wn is not None, (False, False, False))
                q, k, v, gate = _wide(x, wide)
            return q, k, v, gate, (g, beta, dt), logits
        args = (x, w["wq"], w["wk"], w["wv"], w["wg"], w["wa"], wb, pool_block)
        q, k, v, gate, ab, pooled = _Project.apply(*args) if self.grad(*args[:7]) else _project(*args)[0]
        return q, k, v, gate, self.gates(ab), selector(pooled) if pool_block else None

    def conv_norm(self, q, k, v, states, want_states, dt=None):
        """-> (conv(q), conv(k) or None, conv(v) (times dt), normed q, normed k, mixing logits, raw q, k, v
        (or None, None, conv(v) again: attention's), new states).  dt (`takes_dt` only): fp32 [B,T,H], a number for every head of conv(v); as
        separate passes (a training step of the Mamba layer, 8 x 4096) it is seven launches and 0.4 ms."""
        w = self.w
        args = (q, k, v, w["conv_wq"], w["conv_bq"], w["conv_wk"], w["conv_bk"], w["conv_wv"], w["conv_bv"],
                w["norm_q"] if self.delta else None, w["norm_k"] if self.delta else None, w["w_mix"], dt)
        if self.grad(*args):
            return _ConvNorm.apply(self, *args) + (None,)
        ys, ns, new = _conv_norm(self, (q, k, v), states, want_states, dt)
        return ys[0], ys[1], ys[2], ns[0], ns[1], _mix_logits(ys[0], w["w_mix"]), *((q, k, v) if self.raw_attention else (None, None, ys[2])), new

    def gates(self, ab):
        if self.grad(ab, self.w["a_log"], self.w["dt_bias"]):
            return _Gates.apply(self, ab, self.w["a_log"], self.w["dt_bias"])
        return _gates(self, ab)

    def select(self, logits, want_raw):
        """-> (types with the last block forced, counts, attention's share per head, types before that: the forced ones unless wanted)."""
        types, counts, fraction, raw = _Select.apply(logits, want_raw) if self.grad(logits) else _select(logits, want_raw)
        return types, counts, fraction, raw if want_raw else types

    def tail(self, o_lin, o_attn, gate, logits):
        args = (o_lin.contiguous(), o_attn.contiguous(), gate.contiguous(), logits.contiguous())
        w1, w2 = self.w["out_norm1"], self.w["out_norm2"]
        y = _Tail.apply(self, *args, w1, w2) if self.grad(*args, w1, w2) else _tail(self, *args)
        return linear(y.flatten(-2), self.w["wo"])


def _front_plan(layer, kind, w):
    """A FastFront's constants, or None where the layer's weights (by field) or options are not what the fused steps are built for."""
    shapes = weight_shapes(layer)
    delta = kind == 'gdn'
    if not layer.use_short_conv or layer.num_v_heads != layer.num_heads or layer.attn_with_short_conv != delta or (delta and not layer.attn_qk_norm):
        return None
    for n, t in w.items():
        if t is None:
            if n.startswith("conv_b") or (not delta and n in ("wb", "norm_q", "norm_k")):
                continue
            return None
        if not t.is_cuda or t.device != w["wq"].device or not t.is_contiguous() or t.shape != shapes[n] or \
                (t.dtype != torch.bfloat16 and (n not in _EITHER or t.dtype != torch.float32)):
            return None
    if w["a_log"].dtype != w["dt_bias"].dtype or w["out_norm1"].dtype != w["out_norm2"].dtype or (delta and w["norm_q"].dtype != w["norm_k"].dtype):
        return None
    convs = (layer.q_conv1d, layer.k_conv1d, layer.v_conv1d)
    if any(c.kernel_size[0] != layer.conv_size or (c.activation is None) != (convs[0].activation is None) for c in convs) or layer.conv_size not in (2, 3, 4):
        return None
    if any(layer._modules[m].bias is not None for m in ("q_proj", "k_proj", "v_proj", "g_proj", "a_proj", "nats_out_weights_layer", "o_proj")) or \
            (delta and layer.b_proj.bias is not None):
        return None
    norms = (layer.q_norm, layer.k_norm) if delta else (layer.q_norm2, layer.k_norm2)
    width = layer.head_attn_k_dim if delta else layer.head_k_dim
    if norms[0].eps != norms[1].eps or width not in (32, 64, 128, 256, 512) or layer.head_attn_v_dim not in _NORM_GATE_WIDTHS or \
            layer.hidden_size % 8 or layer.num_heads > 256 or layer.value_dim % 8:
        return None
    code = lambda n: _capi.dtype_code(w[n].dtype)
    return dict(delta=delta, H=layer.num_heads, W=layer.conv_size, act=0 if layer.q_conv1d.activation is None else 1, l2=not delta,
                raw_attention=not delta, norm_width=width, front_eps=norms[0].eps, norm_dtype=code("norm_q") if delta else _capi.BF16,
                takes_dt=layer.head_v_dim in (8, 16, 32, 64, 128, 256, 512), gate_dtype=code("a_log"), out_dtype=code("out_norm1"), neg=int(delta and layer.allow_neg_eigval), out_eps=layer.o_norm.eps)


def _selector_weight(layer, like):
    """The weight of the selector's product where it is a plain one over few rows, else None (the layer's own product runs)."""
    m = layer._modules.get("nats_layer")
    if type(m) is not torch.nn.Linear or m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or "forward" in m.__dict__:
        return None
    w = m._parameters.get("weight")
    if m._parameters.get("bias") is not None or w is None or type(w) not in _PLAIN_TENSORS or w.dtype != torch.bfloat16 or not w.is_contiguous() or \
            w.device != like.device or w.dim() != 2 or w.shape[1] != like.shape[1] or w.shape[0] != layer.num_nats_head * layer.n_ops or w.shape[0] > 64:
        return None
    return w


def fast_front(layer, kind, x, cache, cu_seqlens):
    """The layer's FastFront for this forward, or None where the general path has to run."""
    if not x.is_cuda or x.dtype != torch.bfloat16 or cu_seqlens is not None or not x.is_contiguous() or x.numel() == 0 or \
            torch.is_autocast_enabled():
        return None
    seen = watch(layer)
    if seen is None:
        return None
    w = dict(zip(_NAMES, seen.weights(layer)))
    if seen.front_plan is None:
        seen.front_plan = (_front_plan(layer, kind, w),)
    constants = seen.front_plan[0]
    if constants is None or w["wq"].device != x.device:
        return None
    f = FastFront(constants, w, _selector_weight(layer, w["wa"]))
    if f.wn is not None and seen.native_plan is None:
        seen.native_plan = (_native_plan(layer, kind, constants, w, f.wn),)
    if f.wn is not None and seen.native_plan[0] is not None and layer.incomplete_block_start_with_ht and _mixed_common.TIMING_HOOK is None and \
            x.device.index == torch.cuda.current_device() and x.dim() == 3 and x.shape[2] == layer.hidden_size and _on_16(x, f.wn):
        f.native, how = seen.native_plan[0]
        # (the Mamba layer calls its operator with that operator's defaults)
        f.how = dict(how, invalid_attn=kind == 'gdn' and bool(layer.compute_dnats_for_invalid_blocks_attn),
                     invalid_linear=kind != 'gdn' or bool(layer.compute_dnats_for_invalid_blocks_linear_att))
    if cache is not None:
        if torch.is_grad_enabled() and (x.requires_grad or any(t is not None and t.requires_grad for t in w.values())):
            return None
        st = cache.conv_state
        if st is not None and any(s is not None and (s.dtype != torch.bfloat16 or not s.is_contiguous() or s.device != x.device or
                                                     s.shape != (x.shape[0], f.w["conv_w" + n].shape[0], f.W)) for s, n in zip(st, "qkv")):
            return None
    return f
