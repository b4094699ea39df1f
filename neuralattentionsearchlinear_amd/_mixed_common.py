"""Shared host logic of the two mixed operators."""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _capi
from .nats_util import CHUNK_SIZE, PackedSeqs, _seq_args, pack_sequences_here

_attn_streams: dict = {}
_cu_counts: dict = {}


class _Cast(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("n", ctypes.c_int64)]


_MAX_CASTS = 8
_INTS = ("is_delta", "B", "T", "H", "HN", "K", "V", "TN", "block", "flags", "T_attn", "TN_attn", "HQ", "HKV", "KA", "VA", "same_block_visible",
         "types_dtype", "n_seqs", "total_chunks", "total_qtiles", "n_cast_in", "n_cast_out", "private_tables")
_POINTERS = ("q_attn", "k_attn", "v_attn", "types_attn", "o_attn", "lse", "block_indices", "n_blocks", "q", "k", "v", "g", "beta", "h0", "o", "ht",
             "h_block_start", "g_block_sum", "chunk_states", "chunk_v_new", "types", "workspace")


class _Mixed(ctypes.Structure):
    """natsl_mixed of include/natsl.h."""
    _fields_ = ([(n, ctypes.c_int32) for n in _INTS] + [("scale_attn", ctypes.c_float), ("scale_linear", ctypes.c_float)] +
                [(n, ctypes.c_void_p) for n in _POINTERS] +
                [("workspace_bytes", ctypes.c_size_t), ("seqs", ctypes.c_void_p), ("cast_in", _Cast * _MAX_CASTS), ("cast_out", _Cast * _MAX_CASTS)])


_CONVERT, _ROUTE, _SOFTMAX, _LINEAR, _JOIN = 1, 2, 4, 8, 16
_ITEM_BYTES = {torch.bfloat16: 2, torch.float32: 4, torch.int32: 4, torch.uint8: 1}

# Optional timing hook: when set to a callable(name, stream) it is invoked right before and right
# after each branch is enqueued ("softmax:start", "softmax:end", "linear:start", "linear:end") so a
# caller can record events on the stream the kernels were launched on.
TIMING_HOOK = None

# Where the softmax branch is launched.  True: on a side stream next to the linear branch (as the
# reference's Mamba operator does); False: on the caller's stream, one branch after the other (as the
# reference's GDN operator does); None: decide per call - side by side where the linear branch's chain is long enough and its scan leaves CUs.  The scan
# walks the chunks one by one with a few large workgroups, so the softmax kernel fills the CUs it leaves; both take most of a CU's
# LDS (127 KiB / 159 KiB) and never share one, so a scan that fills the chip by itself gains nothing (B8 T8192 H16: 1042
# and 1045 us); B4 T8192 H8 400 -> 326, Mamba B4 T8192 H32 764 -> 699, four packed documents of 65536 tokens 2274 -> 2162 us.  Ordering two
# streams costs a call about 50 us (22 us one after the other, where the softmax tiles share a launch with the prep kernel, 72 us side by side at T 256),
# which the overlap repays from a chain of 2048 tokens at K = 128 on (4096 at K = 64): at B1 H4 T2000 84 -> 74 us with half attention and 66 -> 72 with
# a tenth, 154 -> 111 us at H6 T 4096, but 48 -> 72 us at T 1024.
CONCURRENT_BRANCHES = None
_SIDE_BY_SIDE_TOKENS_X_K = 2048 * 128
_SCAN_COLUMNS_PER_WG = 64           # state columns of the scans' widest workgroup (csrc/natsl_linear.hip, natsl_linear_bwd.hip)

# What the differentiable operator keeps from its forward for the linear branch's backward.  Keeping means: the state entering
# every chunk (bf16, K*V per chunk and head), v_new (64*V bf16) and the prep kernel's workspace (17 KiB) stay in device memory
# until the backward, which then starts at its reverse scan - about 66 KiB per chunk and head at K = V = 128, 1.1 GB per call
# at B8 T8192 H16, for every layer of a model.  Not keeping means: only the inputs are saved and the backward runs the forward's two
# kernels once more, as the reference's backward does (src/nats/ops/gated_delta_rule/chunk.py:170-332 recomputes h); a model that
# fits in memory under the reference then fits here.  The gradients are the same bit for bit either way.  The default keeps what no
# model misses (at most 1.5 GiB over 24 layers); more is the caller's trade and set by the caller.
#   SAVE_CHUNK_STATES = None  (default) keep only when what would be kept is at most SAVE_CHUNK_STATES_MAX_BYTES per call
#                     = True  always keep        = False  never keep
SAVE_CHUNK_STATES = None
SAVE_CHUNK_STATES_MAX_BYTES = 64 << 20
_PREP_WORKSPACE_BYTES = 17 * 1024   # per chunk and head (csrc/natsl_linear.hip)


def _run_side_by_side(dev, packed: bool, n_seqs: int, B: int, T: int, H: int, K: int, V: int) -> bool:
    """Whether the softmax branch (forward or backward) goes to the side stream (see CONCURRENT_BRANCHES)."""
    if CONCURRENT_BRANCHES is not None:
        return bool(CONCURRENT_BRANCHES)
    if T * B // n_seqs * K < _SIDE_BY_SIDE_TOKENS_X_K:
        return False
    if packed:
        return True                                # chains of different lengths
    return _scan_leaves_cus(dev, n_seqs, H, V)


def _scan_leaves_cus(dev, n_seqs: int, H: int, V: int) -> bool:
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    cus = _cu_counts.get(index)
    if cus is None:
        cus = _cu_counts[index] = torch.cuda.get_device_properties(index).multi_processor_count
    workgroups = n_seqs * H * max(1, V // _SCAN_COLUMNS_PER_WG)
    return -workgroups % cus >= cus // 16          # CUs that the scan's last round leaves


def _layer_runs_side_by_side(dev, B: int, T: int, how, gradients: bool) -> bool:
    """_run_side_by_side for a layer's native calls.  Ordering the streams costs the host 90 us of a forward and 100 to 150 us of a training step: two streams
    pay where one would take longer than the host then does.  What one takes follows the products' work (tokens times weights) and the length of the chains.
    The host's share of a training step is one of two figures, which a process keeps: 400 and 590 us with one stream (340M 1 x 832), 505 to 600 and 700 to
    720 with two; two processes of three have the smaller one.  One stream's time over two streams', us, mean of six processes: 340M 1 x 1500 561 / 590,
    1 x 2048 576 / 552, 4 x 1024 637 / 633, 1 x 3000 755 / 626; 760M 1 x 1200 588 / 626, 1 x 1536 645 / 618; 16 heads of 128/64 1 x 1536 535 / 586,
    2 x 1536 649 / 616.  A forward from chains of 2048 tokens at K = 128 on, as the operators, and with more work: 340M 1 x 2048 242 / 346, 3 x 2048 303 / 356,
    4 x 2048 363 / 360, 1 x 3000 258 / 318, 2 x 3000 336 / 322; 760M 1 x 2048 282 / 342, 1 x 3000 379 / 350; shorter ones are 0.95 to 1.06 either way."""
    if CONCURRENT_BRANCHES is not None:
        return bool(CONCURRENT_BRANCHES)
    work = B * T * how["D"] * (sum(how["widths"]) + how["widths"][-1])       # (the output projection is as wide as the gate's)
    if work + 15_000_000 * T < 42_000_000_000 if gradients else work + 12_000_000 * T < 72_000_000_000 or T * how["K"] < _SIDE_BY_SIDE_TOKENS_X_K:
        return False
    return _scan_leaves_cus(dev, B, how["H"], how["V"])


def _keep_chunk_states(q, v, cu_seqlens) -> bool:
    """Whether the differentiable forward keeps the linear branch's chunk states (see SAVE_CHUNK_STATES)."""
    B, T, H, K = q.shape
    return _keep_states_of(B if cu_seqlens is None else len(cu_seqlens) - 1, B, T, H, K, v.shape[-1])                     # (a host list here)


def _keep_states_of(n_seq, B, T, H, K, V) -> bool:
    if SAVE_CHUNK_STATES is not None:
        return bool(SAVE_CHUNK_STATES)
    chunks = -(-B * T // CHUNK_SIZE) + n_seq                       # upper bound on the chunks of all sequences
    return chunks * H * (2 * K * V + 2 * CHUNK_SIZE * V + _PREP_WORKSPACE_BYTES) <= SAVE_CHUNK_STATES_MAX_BYTES


def _get_attn_stream(device: torch.device) -> torch.cuda.Stream:
    """One cached side stream per device for the softmax branch (default priority), as the
    reference does at src/nats/ops/mixed_ops/mixed_attn_mamba.py:26-30,114-124."""
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if idx not in _attn_streams:
        _attn_streams[idx] = torch.cuda.Stream(device=idx)
    return _attn_streams[idx]


def _wants_grad(*tensors) -> bool:
    return torch.is_grad_enabled() and any(t is not None and torch.is_tensor(t) and t.requires_grad for t in tensors)


def linear_chunk_fwd(kind: str, q, k, v, g, beta, h0, types, scale: float, block: int, flags: int,
                     output_final_state: bool, seqs: Optional[PackedSeqs], block_start_state: bool = False,
                     chunk_states: bool = False, outputs: bool = True, beside: Optional[int] = None):
    """Launch the chunked linear branch ('gdn' or 'mamba'); returns (o, final_state or None), or with
    block_start_state (o, final_state, state entering the last block, sum of g over the last block), or with chunk_states
    (o, final_state, the state entering every chunk as bf16 [total_chunks, H, V, K], v_new [B, T, H, V] (for 'mamba': v),
    the workspace); with outputs=False (chunk_states only) o is None and costs nothing, and beside names a stream that is made to wait for
    this one up to the scan."""
    B, T, H, K = q.shape
    V = v.shape[-1]
    TN, HN = types.shape[1], types.shape[2]
    dev = q.device
    n = seqs.n_seqs if seqs is not None else B
    total_chunks = seqs.total_chunks if seqs is not None else B * (-(-T // CHUNK_SIZE))
    L = _capi.lib()
    ws = torch.empty(L.natsl_linear_workspace_bytes(total_chunks, H), dtype=torch.uint8, device=dev)
    o = torch.empty(B, T, H, V, dtype=q.dtype, device=dev) if outputs else None
    ht = torch.empty(n, H, K, V, dtype=torch.float32, device=dev) if output_final_state else None
    hs = torch.empty(n, H, K, V, dtype=torch.float32, device=dev) if block_start_state else None
    gs = torch.empty(n, H, dtype=torch.float32, device=dev) if block_start_state else None
    sc = torch.empty(total_chunks, H, V, K, dtype=torch.bfloat16, device=dev) if chunk_states else None
    if h0 is not None:
        if tuple(h0.shape) != (n, H, K, V):
            raise ValueError(f"initial state must have shape {(n, H, K, V)}, got {tuple(h0.shape)}")
        h0 = h0.to(torch.float32).contiguous()
    sp, ns, tot = _seq_args(seqs, total_chunks)
    vn = torch.empty_like(v) if chunk_states and kind == 'gdn' else None
    if not outputs:
        rc = L.natsl_linear_chunk_states(
            int(kind == 'gdn'), _capi.ptr(q), _capi.ptr(k), _capi.ptr(v), _capi.ptr(g), _capi.ptr(beta), _capi.ptr(h0), _capi.ptr(ht), _capi.ptr(sc), _capi.ptr(vn),
            _capi.ptr(types), _capi.dtype_code(types.dtype), B, T, H, HN, K, V, TN, block, float(scale), flags, _capi.ptr(ws), ws.numel(),
            _capi.dtype_code(q.dtype), sp, ns, tot, _capi.stream_ptr(dev), beside)
        _capi.check(rc, "natsl_linear_chunk_states")
        return None, ht, sc, (vn if kind == 'gdn' else v), ws
    common = (_capi.ptr(h0), _capi.ptr(o), _capi.ptr(ht), _capi.ptr(hs), _capi.ptr(gs), _capi.ptr(sc),
              *((_capi.ptr(vn),) if kind == 'gdn' else ()), _capi.ptr(types), _capi.dtype_code(types.dtype), B, T, H, HN, K, V, TN,
              block, float(scale), flags, _capi.ptr(ws), ws.numel(), _capi.dtype_code(q.dtype), sp, ns, tot,
              _capi.stream_ptr(dev))
    if kind == 'gdn':
        rc = L.natsl_gdn_chunk_fwd(_capi.ptr(q), _capi.ptr(k), _capi.ptr(v), _capi.ptr(g), _capi.ptr(beta), *common)
        _capi.check(rc, "natsl_gdn_chunk_fwd")
    else:
        rc = L.natsl_mamba_chunk_fwd(_capi.ptr(q), _capi.ptr(k), _capi.ptr(v), _capi.ptr(g), *common)
        _capi.check(rc, "natsl_mamba_chunk_fwd")
    if block_start_state:
        return o, ht, hs, gs
    if chunk_states:
        return o, ht, sc, (vn if kind == 'gdn' else v), ws
    return o, ht


def state_behind(ht, hs, gs, last):
    """The state the next block starts from where the input ends on a block's end: the final state ht [N,H,K,V] where the last block's type (last [N,HN,2])
    is linear, else the one that entered it, hs, decayed by gs [N,H], the sum of g over it (None: not decayed)."""
    n, H, K, V = ht.shape
    dev = ht.device
    # (a launch goes to the current device, torch's operations to their tensors')
    if last.is_cuda and last.device == dev and dev.index in (None, torch.cuda.current_device()) and \
            last.dtype in (torch.bfloat16, torch.float32) and last.dim() == 3 and last.shape[0] == n and \
            last.stride(2) == 1 and H % last.shape[1] == 0 and last.shape[2] > 1 and n * H <= 65535:
        h_start = torch.empty_like(ht)
        rc = _capi.lib().natsl_roll_state(ht.data_ptr(), hs.data_ptr(), _capi.ptr(gs), last.data_ptr(), _capi.dtype_code(last.dtype), last.stride(0),
                                          last.stride(1), h_start.data_ptr(), n, H, last.shape[1], K * V, _capi.stream_ptr(dev))
        _capi.check(rc, "natsl_roll_state")
        return h_start
    lin = (last[..., 1] > 0)
    lin = lin.repeat_interleave(H // lin.shape[1], dim=1).view(n, H, 1, 1)
    return torch.where(lin, ht, hs if gs is None else hs * torch.exp(gs).view(n, H, 1, 1))


def _same_rows(t, shape) -> bool:
    """Whether t holds the rows of `shape` in its order (sizes of one more or less do not move a number)."""
    return t.shape == shape or [n for n in t.shape if n != 1] == [n for n in shape if n != 1]


def _check_operands(q_attn, k_attn, v_attn, q, k, v, g, beta, types, n_prefix: int = 0):
    """ValueError unless the tensors go together: the kernels take every size from q_attn, q and the widths of the others, so a tensor of another size would be
    read past its end or at strides that are not its own.  (The branches may have other numbers of tokens than each other while these make as many blocks,
    which the native entry compares.)"""
    B, T, H, K = q.shape
    _, T_attn, HQ, KA = q_attn.shape
    keys = (B, T_attn + n_prefix, *k_attn.shape[2:3])
    for name, t, shape in (("q_attn", q_attn, (B, T_attn, HQ, KA)), ("k_attn", k_attn, (*keys, KA)), ("v_attn", v_attn, (*keys, *v_attn.shape[3:4])),
                           ("k_lattn", k, (B, T, H, K)), ("v_lattn", v, (B, T, H, *v.shape[3:4])), ("nats_block_types", types, (B, *types.shape[1:3], 2))):
        if len(shape) != 4 or t.shape != shape:
            raise ValueError(f"{name} must have shape {list(shape)} beside q_lattn {list(q.shape)} and q_attn {list(q_attn.shape)}, got {list(t.shape)}")
    for name, t in (("g", g), ("beta", beta)):
        if t is not None and not _same_rows(t, (B, T, H)):
            raise ValueError(f"{name} must have shape {[B, T, H]} beside q_lattn {list(q.shape)}, got {list(t.shape)}")
    for name, t in (("q_attn", q_attn), ("k_attn", k_attn), ("v_attn", v_attn), ("k_lattn", k), ("v_lattn", v), ("g", g), ("beta", beta),
                    ("nats_block_types", types)):
        if t is not None and t.device != q.device:
            raise ValueError(f"{name} is on {t.device}, q_lattn on {q.device}")


def _check_packed(seqs, T: int, T_attn: int, TN: int):
    """ValueError unless the packed sequences lie in rows of T (and T_attn) tokens and TN selector blocks."""
    if seqs is not None and seqs.n_seqs and (seqs.cu_seqlens[0] < 0 or seqs.cu_seqlens[-1] > min(T, T_attn) or seqs.cu_seqlens_nats[0] < 0 or seqs.cu_seqlens_nats[-1] > TN):
        raise ValueError(f"cu_seqlens runs from {seqs.cu_seqlens[0]} to {seqs.cu_seqlens[-1]} in {min(T, T_attn)} tokens, cu_seqlens_nats from "
                         f"{seqs.cu_seqlens_nats[0]} to {seqs.cu_seqlens_nats[-1]} in {TN} selector blocks")


def _mixed_forward_impl(kind, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types,
                  scale_attn, scale_lattn, cu_seqlens, cu_seqlens_nats, nats_block_size, attn_sw_size,
                  attn_same_block: bool, lin_intra: bool, output_final_state: bool, decay_non_linear: bool,
                  incomplete_block_start_with_ht: bool, use_g_for_attn: bool, qk_l2norm: bool,
                  inference: bool = False, op_type_last_chunk=None, n_tokens_in_current_block: int = 0, return_aux: bool = False,
                  keep_chunk_states: bool = False, attn_prefix_valid: Optional[torch.Tensor] = None):
    """Shared forward of the mixed operators.  With inference=True it also returns the state at the
    start of the current selector block (4-tuple), as the reference's *_chunk_inference operators do.  With return_aux
    and keep_chunk_states the auxiliary dict also holds what the linear backward would otherwise recompute
    (`linear_saved`: chunk states, v_new, workspace).

    attn_prefix_valid (bool [B, NP, HN], inference only): k_attn and v_attn start with NP more whole blocks than the other
    tensors -- cached keys; block j of that prefix is visible to selector head h's queries where the flag is set.  The softmax
    branch then runs over prefix + tokens with no queries in the prefix (a chunked forward that continues a cache: the
    reference's attention operator sizes its output by the keys, src/nats/ops/attns/attns.py:1439,1491, and cannot)."""
    if nats_block_size < CHUNK_SIZE:
        raise AssertionError("nats_block_size must be at least the compute chunk (64)")   # mixed_attn_gdn.py:90
    if nats_block_size % CHUNK_SIZE:
        raise NotImplementedError("nats_block_size must be a multiple of 64")
    if attn_sw_size is not None:
        raise NotImplementedError("attn_sw_size is not used by the reference layers and is not built")
    if use_g_for_attn:
        raise NotImplementedError("use_g_for_attn is disabled in every reference layer and is not built")
    if lin_intra and not incomplete_block_start_with_ht:
        raise NotImplementedError("incomplete_block_start_with_ht=False is not built")
    if n_tokens_in_current_block != 0:
        raise NotImplementedError("n_tokens_in_current_block != 0 is never passed by the reference layers and is not built")
    if inference and (cu_seqlens is not None):
        raise NotImplementedError("packed sequences are not supported by the prefill hand-off")
    if not q_lattn.is_cuda:
        raise _capi.NatslError("the NAtS-L mixed operator runs on the GPU only (no CPU fallback)")
    if nats_block_types.shape[-1] != 2:
        raise NotImplementedError("routing is built for n_ops == 2")
    _check_operands(q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, g, beta, nats_block_types,
                    0 if attn_prefix_valid is None else attn_prefix_valid.shape[1] * nats_block_size)
    io_dtype = q_lattn.dtype
    if io_dtype not in (torch.bfloat16, torch.float32):
        raise NotImplementedError(f"dtype {io_dtype} is not supported (bf16, or fp32 which is computed in bf16)")

    m = _Mixed()
    dev = q_lattn.device
    # What only this call uses (conversions, routing tables, workspaces) lives in one allocation; what the backward keeps
    # (return_aux) is made of tensors of its own.
    scratch, total = [], 0

    def own(shape, dtype, set_pointer, hidden=True):
        """A tensor of this call: a place in the scratch when nobody sees it afterwards (-> None), else a torch tensor."""
        nonlocal total
        if hidden and not return_aux:
            scratch.append((set_pointer, total))
            n = _ITEM_BYTES[dtype]
            for d in shape:
                n *= d
            total += (n + 255) & ~255
            return None
        t = torch.empty(shape, dtype=dtype, device=dev)
        set_pointer(t.data_ptr())
        return t

    copies = {}

    def as_bf16(t, name):
        """Names t (bf16, contiguous) in the call's arguments; an fp32 tensor's copy is filled by the call (one launch for all of
        them).  -> the bf16 tensor, or t itself where its copy is in the scratch."""
        if t is None:
            return None
        t = t.detach()
        if t.dtype == torch.float32 and t.numel() > 0:
            t = t.contiguous()
            if t.data_ptr() % 16 == 0:
                got = copies.get((t.data_ptr(), t.shape))
                if got is None:
                    c = m.cast_in[len(copies)]
                    c.src, c.n = t.data_ptr(), t.numel()
                    fields = [name]

                    def point(at):
                        c.dst = at
                        for f in fields:
                            setattr(m, f, at)
                    got = copies[(t.data_ptr(), t.shape)] = (own(t.shape, torch.bfloat16, point, attn_prefix_valid is None), fields, t)
                elif got[0] is None:
                    got[1].append(name)
                if got[0] is None:
                    return t
                setattr(m, name, got[0].data_ptr())
                return got[0]
        t = t if t.dtype == torch.bfloat16 else t.to(torch.bfloat16)
        t = t.contiguous()
        setattr(m, name, t.data_ptr())
        return t

    q_attn, k_attn, v_attn = as_bf16(q_attn, "q_attn"), as_bf16(k_attn, "k_attn"), as_bf16(v_attn, "v_attn")
    q_lattn, k_lattn, v_lattn, beta = as_bf16(q_lattn, "q"), as_bf16(k_lattn, "k"), as_bf16(v_lattn, "v"), as_bf16(beta, "beta")
    m.n_cast_in = len(copies)
    g = g.detach().to(torch.float32).contiguous()
    types = nats_block_types.detach()
    if types.dtype not in (torch.bfloat16, torch.float32):
        types = types.float()
    types = types.contiguous()
    B, T, H, K = q_lattn.shape
    V = v_lattn.shape[-1]
    TN, HN = types.shape[1], types.shape[2]
    # Boundaries that lie on the GPU are read behind everything that can be made without them: the host waits there for the work before this
    # call, and what it does afterwards the GPU waits for.
    late = torch.is_tensor(cu_seqlens) and cu_seqlens.dim() == 1 and cu_seqlens.numel() > 1 and not keep_chunk_states
    seqs = None if late else pack_sequences_here(cu_seqlens, cu_seqlens_nats, nats_block_size, dev)
    cur, L = _capi.stream_ptr(dev), _capi.lib()

    n_prefix, types_attn = 0, types
    if attn_prefix_valid is not None:
        if not inference or cu_seqlens is not None:
            raise NotImplementedError("a key prefix is built for the prefill operators on unpacked input")
        NP = attn_prefix_valid.shape[1]
        n_prefix = NP * nats_block_size
        if k_attn.shape[1] != q_attn.shape[1] + n_prefix or v_attn.shape[1] != k_attn.shape[1]:
            raise ValueError(f"with a prefix of {NP} blocks the keys must hold {q_attn.shape[1] + n_prefix} tokens, got {k_attn.shape[1]}")
        if m.n_cast_in:                                   # the queries are put together below: their conversion comes first
            _capi.check(L.natsl_mixed_fwd(ctypes.byref(m), _CONVERT, cur, cur), "natsl_mixed_fwd")
            m.n_cast_in = 0
        pv = attn_prefix_valid.to(types.dtype)
        types_attn = torch.cat([torch.stack([pv, 1 - pv], -1), types], 1).contiguous()
        q_attn = torch.cat([q_attn.new_zeros(q_attn.shape[0], n_prefix, *q_attn.shape[2:]), q_attn], 1)
        m.q_attn = q_attn.data_ptr()
    T_attn, HQ, KA = q_attn.shape[1:]
    HKV, VA = k_attn.shape[2], v_attn.shape[3]

    if late:
        n_seqs = cu_seqlens.numel() - 1
        total_chunks = B * T // CHUNK_SIZE + n_seqs            # (no sequences of T tokens have more)
    else:
        n_seqs = seqs.n_seqs if seqs is not None else B
        total_chunks = seqs.total_chunks if seqs is not None else B * (-(-T // CHUNK_SIZE))
    # every tensor below belongs to the caller's stream; the softmax branch's stream starts after what that stream holds and is
    # waited for before the call returns, so memory that is freed later is only ever used again behind both
    side = _get_attn_stream(dev) if _run_side_by_side(dev, cu_seqlens is not None, n_seqs, B, T, H, K, V) else None
    attn_stream = cur if side is None else side.cuda_stream
    want_start = inference and output_final_state
    chunk_states = keep_chunk_states and not want_start
    bf16, f32 = torch.bfloat16, torch.float32
    point = lambda name: lambda at: setattr(m, name, at)
    ws_bytes = L.natsl_mixed_workspace_bytes(total_chunks, H)
    idx = own((B, types_attn.shape[1], HN, 2), torch.int32, point("block_indices"))
    nblk = own((n_seqs, HN, 2), torch.int32, point("n_blocks"))
    lse = own((B, T_attn, HQ), f32, point("lse"))
    ws = own((ws_bytes,), torch.uint8, point("workspace"))
    o_attn = torch.empty(B, T_attn, HQ, VA, dtype=io_dtype, device=dev)
    o_lin = torch.empty(B, T, H, V, dtype=io_dtype, device=dev)
    o_attn16, o_lin16 = o_attn, o_lin
    if io_dtype == bf16:
        m.o_attn, m.o = o_attn.data_ptr(), o_lin.data_ptr()
    else:
        def out(c, name, dst):
            c.dst, c.n = dst.data_ptr(), dst.numel()

            def set_both(at):
                c.src = at
                setattr(m, name, at)
            return own(dst.shape, bf16, set_both)
        o_attn16, o_lin16 = out(m.cast_out[0], "o_attn", o_attn), out(m.cast_out[1], "o", o_lin)
        m.n_cast_out = 2
    ht = torch.empty(n_seqs, H, K, V, dtype=f32, device=dev) if output_final_state else None
    hs = torch.empty(n_seqs, H, K, V, dtype=f32, device=dev) if want_start else None
    gs = torch.empty(n_seqs, H, dtype=f32, device=dev) if want_start else None
    sc = torch.empty(total_chunks, H, V, K, dtype=bf16, device=dev) if chunk_states else None
    vn = torch.empty_like(v_lattn) if chunk_states and kind == 'gdn' else None
    if scratch:
        block = torch.empty(total, dtype=torch.uint8, device=dev)
        base = block.data_ptr()
        for set_pointer, at in scratch:
            set_pointer(base + at)
    h0 = None
    if initial_state is not None:
        if tuple(initial_state.shape) != (n_seqs, H, K, V) or initial_state.device != dev:
            raise ValueError(f"initial state must have shape {(n_seqs, H, K, V)} on {dev}, got {tuple(initial_state.shape)} on {initial_state.device}")
        h0 = initial_state.detach().to(f32).contiguous()
    m.is_delta, m.B, m.T, m.H, m.HN, m.K, m.V, m.TN, m.block = int(kind == 'gdn'), B, T, H, HN, K, V, TN, nats_block_size
    m.flags = (_capi.DECAY_NON_LINEAR if decay_non_linear else 0) | (_capi.QK_L2NORM if qk_l2norm else 0) | (_capi.INTRA_CHUNK if lin_intra else 0)
    m.T_attn, m.TN_attn, m.HQ, m.HKV, m.KA, m.VA = T_attn, types_attn.shape[1], HQ, HKV, KA, VA
    m.same_block_visible, m.types_dtype, m.private_tables = int(attn_same_block), _capi.dtype_code(types.dtype), int(not return_aux)
    m.scale_attn, m.scale_linear = scale_attn, scale_lattn
    m.g, m.types, m.types_attn, m.workspace_bytes = g.data_ptr(), types.data_ptr(), types_attn.data_ptr(), ws_bytes
    for name, t in (("h0", h0), ("ht", ht), ("h_block_start", hs), ("g_block_sum", gs), ("chunk_states", sc), ("chunk_v_new", vn)):
        if t is not None:
            setattr(m, name, t.data_ptr())
    if late:
        seqs = pack_sequences_here(cu_seqlens, cu_seqlens_nats, nats_block_size, dev)
    _check_packed(seqs, T, T_attn, TN)
    if seqs is not None:
        m.seqs, m.n_seqs, m.total_chunks, m.total_qtiles = seqs.table.data_ptr(), seqs.n_seqs, seqs.total_chunks, seqs.total_qtiles
    ref = ctypes.byref(m)
    if TIMING_HOOK is None:
        _capi.check(L.natsl_mixed_fwd(ref, _CONVERT | _ROUTE | _SOFTMAX | _LINEAR | _JOIN, cur, attn_stream), "natsl_mixed_fwd")
    else:
        here = torch.cuda.current_stream(dev)
        step = lambda phases: _capi.check(L.natsl_mixed_fwd(ref, phases, cur, attn_stream), "natsl_mixed_fwd")
        step(_CONVERT | _ROUTE)
        if side is None:
            TIMING_HOOK("softmax:start", here)
            step(_SOFTMAX)
            TIMING_HOOK("softmax:end", here)
            TIMING_HOOK("linear:start", here)
            step(_LINEAR)
            TIMING_HOOK("linear:end", here)
        else:                                              # (side by side the order is the call's own; softmax includes its wait)
            TIMING_HOOK("softmax:start", side)
            TIMING_HOOK("linear:start", here)
            step(_SOFTMAX | _LINEAR)
            TIMING_HOOK("softmax:end", side)
            TIMING_HOOK("linear:end", here)
        step(_JOIN)
    if n_prefix:
        o_attn = o_attn[:, n_prefix:]
    if return_aux:
        aux = dict(q_attn=q_attn, k_attn=k_attn, v_attn=v_attn, q_lattn=q_lattn, k_lattn=k_lattn, v_lattn=v_lattn, beta=beta, g=g,
                   types=types, lse=lse, nats_block_indices=idx, n_nats_blocks=nblk, o_attn=o_attn16,
                   linear_saved=(sc, vn if kind == 'gdn' else v_lattn, ws) if chunk_states else None)
        return o_lin, o_attn, ht, aux
    if not inference:
        return o_lin, o_attn, ht
    h_start = None
    if want_start:
        # State at the start of the current block (src/nats/ops/gated_delta_rule/chunk_fwd.py:178-206):
        # with an incomplete last block it is the state that entered that block; when the input ends on
        # a block boundary it is the state after the last block under its TRUE type -- the final state
        # if that type is linear, otherwise the entering state rolled forward by the block's decay.
        if T % nats_block_size != 0:
            h_start = hs
        else:
            if op_type_last_chunk is None:
                raise AssertionError("op_type_last_chunk is required when the input ends on a block boundary")
            h_start = state_behind(ht, hs, gs if decay_non_linear else None, op_type_last_chunk)
    return o_lin, o_attn, ht, h_start


class _MixedFunction(torch.autograd.Function):
    """The mixed operator with its backward (src/nats/ops/mixed_ops/mixed_attn_gdn.py:193-283,
    src/nats/ops/mixed_ops/mixed_attn_mamba.py:194-292): the softmax branch's gradients come from the HIP backward
    (natsl_softmax_sparse_bwd), the linear branch's from natsl_linear_chunk_bwd behind _linear_bwd.linear_chunk_backward; the
    selector's straight-through gradient is returned for nats_block_types, column 0 = softmax op, column 1 = linear op."""

    @staticmethod
    def forward(ctx, cfg, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types):
        from ._linear_bwd import hip_backward_is_built
        keep = _keep_chunk_states(q_lattn, v_lattn, cfg['cu_seqlens']) and hip_backward_is_built(q_lattn.shape[-1], v_lattn.shape[-1])
        with torch.no_grad():
            o_lin, o_attn, ht, aux = _mixed_forward_impl(
                cfg['kind'], q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types,
                cfg['scale_attn'], cfg['scale_lattn'], cfg['cu_seqlens'], cfg['cu_seqlens_nats'], cfg['block'], None,
                cfg['attn_same_block'], cfg['lin_intra'],
                cfg['output_final_state'], cfg['decay_non_linear'], True, False, cfg['qk_l2norm'], return_aux=True,
                keep_chunk_states=keep)
        ctx.cfg = cfg
        ctx.in_dtypes = tuple(None if t is None else t.dtype for t in (q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn,
                                                                       initial_state, g, beta, nats_block_types))
        ctx.has_h0 = initial_state is not None
        # a tensor given to both branches gets one gradient, added up by the linear branch's last kernel (bf16: the same sum, rounded the
        # same way, as autograd's)
        ctx.shared = tuple(a is l and a.dtype == torch.bfloat16 for a, l in ((q_attn, q_lattn), (k_attn, k_lattn), (v_attn, v_lattn)))
        saved = [aux[n] for n in ('q_attn', 'k_attn', 'v_attn', 'q_lattn', 'k_lattn', 'v_lattn', 'g', 'types', 'lse',
                                  'nats_block_indices', 'n_nats_blocks')]
        saved += [aux['o_attn'], aux['beta'] if aux['beta'] is not None else g.new_zeros(0),
                  initial_state if initial_state is not None else g.new_zeros(0)]
        ctx.n_linear_saved = 0
        if aux['linear_saved'] is not None:
            # (for 'mamba' the second entry is v_lattn itself, saved above already: the same tensor, no second copy)
            saved += list(aux['linear_saved'])
            ctx.n_linear_saved = len(aux['linear_saved'])
        ctx.save_for_backward(*saved)
        ctx.set_materialize_grads(False)        # (a final state that nothing follows is neither filled with zeros nor read)
        if ht is None:
            return o_lin, o_attn, None
        return o_lin, o_attn, ht

    @staticmethod
    def backward(ctx, do_lin, do_attn, dht):
        from ._linear_bwd import hip_backward_is_built, linear_chunk_backward
        from .attns import prepare_attn_nats_bwd
        cfg = ctx.cfg
        (q_a, k_a, v_a, q_l, k_l, v_l, g, types, lse, idx, nblk, o_attn, beta, h0) = ctx.saved_tensors[:14]
        linear_saved = tuple(ctx.saved_tensors[14:]) if ctx.n_linear_saved else None
        beta = beta if beta.numel() else None
        h0 = h0 if ctx.has_h0 else None
        B, NB, HN, _ = types.shape
        seqs = pack_sequences_here(cfg['cu_seqlens'], cfg['cu_seqlens_nats'], cfg['block'], types.device)
        if do_lin is None:
            do_lin = torch.zeros(*q_l.shape[:3], v_l.shape[-1], dtype=torch.float32, device=q_l.device)
        if do_attn is not None:
            do_attn = do_attn.to(torch.bfloat16).contiguous()
        # The softmax branch's tensors are made first, on this stream, and live until this stream has its kernels behind it (nothing
        # that is allocated in between can share their memory).  Side by side, both scans are enqueued first (see natsl_mixed_fwd), with the
        # softmax branch behind the kernel in front of the first, and the per-chunk kernel, which adds the branches' gradients of a
        # tensor they share, behind both.
        attn = side = release = None
        if do_attn is not None:
            attn = prepare_attn_nats_bwd(q_a, k_a, v_a, o_attn, types, idx, nblk, None, lse, do_attn, cfg['scale_attn'], cfg['block'], 0,
                                         cfg['attn_same_block'], cfg['dnats_invalid_attn'], None, None, None, True, seqs)
            here = torch.cuda.current_stream(q_l.device)
            if _run_side_by_side(q_l.device, seqs is not None, B if seqs is None else seqs.n_seqs, *q_l.shape, v_l.shape[-1]):
                side = _get_attn_stream(q_l.device)
                if linear_saved is None and hip_backward_is_built(q_l.shape[-1], v_l.shape[-1]):
                    release = side.cuda_stream
                else:
                    side.wait_stream(here)
            else:
                attn[0](here.cuda_stream)

        def softmax_beside():
            nonlocal side
            if side is not None:
                beside, side = side, None
                try:
                    attn[0](beside.cuda_stream)
                finally:
                    here.wait_stream(beside)
        onto = (None, None, None)
        if attn is not None and hip_backward_is_built(q_l.shape[-1], v_l.shape[-1]):
            onto = tuple(t if both else None for t, both in zip(attn[1], ctx.shared))
        lin_args = (cfg['scale_lattn'], cfg['block'], cfg['decay_non_linear'], cfg['qk_l2norm'], cfg['lin_intra'])
        later = []
        dq_l, dk_l, dv_l, dg, dbeta, dh0, dn_lin = linear_chunk_backward(
            cfg['kind'], q_l, k_l, v_l, g, beta, h0, types, *lin_args, do_lin, dht, cfg['dnats_invalid_linear'], seqs,
            saved=linear_saved, later=later, release=release, meanwhile=softmax_beside, beside=0 if side is None else 4, onto=onto)
        softmax_beside()                                   # (where the linear branch did not call it)
        lin = [dq_l, dk_l, dv_l]
        if attn is not None:
            dq_a, dk_a, dv_a, dn_attn = attn[1]
            lin = [None if have is not None else t for t, have in zip(lin, onto)]
            if not later:
                dn_attn = dn_attn.view(B, NB, HN, -1).sum(-1)
        else:
            dq_a, dk_a, dv_a = torch.zeros_like(q_a), torch.zeros_like(k_a), torch.zeros_like(v_a)
            dn_attn = torch.zeros(B, NB, q_a.shape[2] if later else HN, dtype=torch.float32, device=types.device)
        d_types = later[0](dn_attn) if later else torch.stack([dn_attn.float(), dn_lin.float()], -1)
        grads = [dq_a, dk_a, dv_a, *lin, dh0, dg, dbeta, d_types]
        grads = [None if (t is None or dt is None) else t.to(dt) for t, dt in zip(grads, ctx.in_dtypes)]
        return (None, *grads)


def _plain_forward(kind, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, types, scale_attn, scale_lattn, block,
                   attn_same_block, lin_intra, output_final_state, decay_non_linear, qk_l2norm):
    """The forward of an ordinary call as one native call (csrc/host/mixed_core.cpp), None where it is not one."""
    B, T, H, K = q_lattn.shape
    dev = q_lattn.device
    cur = _capi.stream_ptr(dev)
    side = _get_attn_stream(dev).cuda_stream if B > 0 and _run_side_by_side(dev, False, B, B, T, H, K, v_lattn.shape[-1]) else cur
    options = (kind == 'gdn') | bool(decay_non_linear) << 1 | bool(qk_l2norm) << 2 | bool(lin_intra) << 3 | bool(attn_same_block) << 4 | \
        bool(output_final_state) << 5
    done = _capi.step_core().mixed_plain(_capi.entries(), options, block, scale_attn, scale_lattn, cur, side, q_attn, k_attn, v_attn, q_lattn, k_lattn,
                                         v_lattn, initial_state, g, beta, types)
    if done is not None and type(done) is not tuple:
        _capi.check(done, "natsl_mixed_fwd")
    return done


def _host_list(x):
    return None if x is None else [int(t) for t in (x.tolist() if torch.is_tensor(x) else x)]


def mixed_forward(kind, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types,
                  scale_attn, scale_lattn, cu_seqlens, cu_seqlens_nats, nats_block_size, attn_sw_size,
                  attn_same_block: bool, lin_intra: bool, output_final_state: bool, decay_non_linear: bool,
                  incomplete_block_start_with_ht: bool, use_g_for_attn: bool, qk_l2norm: bool,
                  inference: bool = False, op_type_last_chunk=None, n_tokens_in_current_block: int = 0,
                  dnats_invalid_attn: bool = False, dnats_invalid_linear: bool = False, attn_prefix_valid=None):
    """Entry of the mixed operators: the plain forward, or, when a tensor requires grad, the differentiable operator."""
    tensors = (q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types)
    # (the prefill operators are plain functions in the reference too: their outputs carry no gradient)
    if inference or not _wants_grad(*tensors):
        if not inference and cu_seqlens is None and attn_prefix_valid is None and attn_sw_size is None and n_tokens_in_current_block == 0 and \
                not use_g_for_attn and incomplete_block_start_with_ht and TIMING_HOOK is None and q_lattn.is_cuda and q_lattn.dim() == 4 and \
                type(nats_block_size) is int:
            done = _plain_forward(kind, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta, nats_block_types, scale_attn,
                                  scale_lattn, nats_block_size, attn_same_block, lin_intra, output_final_state, decay_non_linear, qk_l2norm)
            if done is not None:
                return done
        return _mixed_forward_impl(kind, q_attn, k_attn, v_attn, q_lattn, k_lattn, v_lattn, initial_state, g, beta,
                                   nats_block_types, scale_attn, scale_lattn, cu_seqlens, cu_seqlens_nats, nats_block_size,
                                   attn_sw_size, attn_same_block, lin_intra, output_final_state, decay_non_linear,
                                   incomplete_block_start_with_ht, use_g_for_attn, qk_l2norm, inference, op_type_last_chunk,
                                   n_tokens_in_current_block, attn_prefix_valid=attn_prefix_valid)
    if attn_prefix_valid is not None:
        raise NotImplementedError("a key prefix is built for the prefill operators (no gradient)")
    if attn_sw_size is not None or use_g_for_attn or not incomplete_block_start_with_ht:
        raise NotImplementedError("attn_sw_size / use_g_for_attn / incomplete_block_start_with_ht=False are not built")
    cfg = dict(kind=kind, scale_attn=float(scale_attn), scale_lattn=float(scale_lattn), block=int(nats_block_size),
               attn_same_block=bool(attn_same_block), lin_intra=bool(lin_intra), output_final_state=bool(output_final_state),
               decay_non_linear=bool(decay_non_linear), qk_l2norm=bool(qk_l2norm), dnats_invalid_attn=bool(dnats_invalid_attn),
               dnats_invalid_linear=bool(dnats_invalid_linear), cu_seqlens=_host_list(cu_seqlens),
               cu_seqlens_nats=_host_list(cu_seqlens_nats))
    return _MixedFunction.apply(cfg, *tensors)
