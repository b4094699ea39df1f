"""GPU parity of the persistent softmax kernel (whole 256-query tiles, cut lengths and packed sequences, enough tiles for every CU):
against the oracle, bit for bit against the per-tile kernel (same chunk order, same arithmetic; but for the tile of a cut chunk), its
row sums there against 64-bit arithmetic, and its work queues across launches."""
import pytest
import torch

from oracle import softmax_branch as sb
from tests._util import assert_close, make_qkv, make_types

pytestmark = pytest.mark.gpu


def _inputs(B, T, HQ, H, HN, K, V, block, p_attn, seed, dev):
    q, k, v = make_qkv(B, T, H, K, V, seed, HQ=HQ)
    ty = make_types(B, -(-T // block), HN, p_attn, seed + 1, torch.bfloat16)
    return q, k, v, ty, q.to(dev), k.to(dev), v.to(dev), ty.to(dev)


def _call(qd, kd, vd, tyd, K, block, same_block, persistent=True, seqs=None):
    """The softmax branch through the C ABI: natsl_softmax_sparse_fwd (picks the persistent kernel for these shapes), or
    natsl_softmax_sparse_fwd_per_tile (one workgroup per query tile, the same results)."""
    from neuralattentionsearchlinear_amd import _capi, nats_util
    r = nats_util.route(tyd, qd.shape[1], block, seqs)
    B, T, HQ, _ = qd.shape
    H, V = kd.shape[2], vd.shape[-1]
    TN, HN = tyd.shape[1], tyd.shape[2]
    o = torch.empty(B, T, HQ, V, dtype=vd.dtype, device=qd.device)
    lse = torch.empty(B, T, HQ, dtype=torch.float32, device=qd.device)
    L = _capi.lib()
    fn = L.natsl_softmax_sparse_fwd if persistent else L.natsl_softmax_sparse_fwd_per_tile
    if persistent:
        assert L.natsl_softmax_fwd_variant(B, T, HQ, H, block, seqs.n_seqs if seqs else 0) == 2, "shape does not reach the persistent kernel on this GPU"
    rc = fn(_capi.ptr(qd), _capi.ptr(kd), _capi.ptr(vd), _capi.ptr(o), _capi.ptr(lse), _capi.ptr(tyd), _capi.dtype_code(tyd.dtype),
            _capi.ptr(r['nats_block_indices']), _capi.ptr(r['n_nats_blocks']), B, T, HQ, H, HN, K, V, TN, block, float(K ** -0.5),
            int(bool(same_block)), _capi.dtype_code(qd.dtype), *((_capi.ptr(seqs.table), seqs.n_seqs, seqs.total_qtiles) if seqs else (None, 0, 0)),
            _capi.stream_ptr(qd.device))
    _capi.check(rc, "natsl_softmax_sparse_fwd")
    return o, lse


def _enough_tiles(B, HQ, T):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return T % 256 == 0 and B * HQ * (T // 256) >= 2 * cus


@pytest.mark.parametrize("same_block", [True, False])
@pytest.mark.parametrize("K,V", [(128, 128), (64, 64), (64, 128), (128, 64)])
def test_persistent_kernel_against_the_oracle(K, V, same_block):
    B, T, HQ, H, HN, block = 4, 2048, 16, 4, 8, 64
    dev = torch.device('cuda:0')
    assert _enough_tiles(B, HQ, T), "shape does not reach the persistent kernel on this GPU"
    q, k, v, ty, qd, kd, vd, tyd = _inputs(B, T, HQ, H, HN, K, V, block, 0.3, 11, dev)
    o_ref, lse_ref = sb.softmax_branch(q, k, v, ty, K ** -0.5, block, same_block)
    o, lse = _call(qd, kd, vd, tyd, K, block, same_block)
    torch.cuda.synchronize()
    assert_close(o.float(), o_ref, "o_attn")
    assert_close(lse, lse_ref, "lse")


@pytest.mark.parametrize("B,T,HQ,H,HN,K,V,block,p_attn,same_block", [
    (8, 8192, 16, 16, 16, 128, 128, 64, 0.25, True),     # the benchmark shape
    (2, 8192, 16, 4, 8, 128, 128, 128, 0.3, True),       # grouped kv heads and selector heads
    (4, 4096, 32, 32, 32, 64, 64, 256, 0.5, False),      # only earlier attention blocks visible
    (3, 2048, 24, 8, 24, 64, 128, 512, 0.4, True),       # blocks larger than a tile, head count not a multiple of 8
    (2, 4096, 16, 16, 16, 128, 64, 2048, 0.5, True),     # 32 chunks from the block start
    (8, 4096, 16, 16, 16, 128, 128, 64, 1.0, True),      # dense causal
    (8, 4096, 16, 16, 16, 128, 128, 64, 0.0, True),      # nothing but the own block
    (8, 4096, 16, 16, 16, 128, 128, 64, 0.0, False),     # nothing visible at all
    (1, 65536, 8, 8, 8, 128, 128, 64, 0.1, True),        # longest admitted sequence: 1024 blocks in the list
])
def test_persistent_kernel_equals_the_per_tile_kernel(B, T, HQ, H, HN, K, V, block, p_attn, same_block):
    dev = torch.device('cuda:0')
    assert _enough_tiles(B, HQ, T), "shape does not reach the persistent kernel on this GPU"
    _, _, _, _, qd, kd, vd, tyd = _inputs(B, T, HQ, H, HN, K, V, block, p_attn, 23, dev)
    o1, l1 = _call(qd, kd, vd, tyd, K, block, same_block, persistent=False)
    o2, l2 = _call(qd, kd, vd, tyd, K, block, same_block, persistent=True)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2)
    assert torch.equal(l1, l2)


@pytest.mark.parametrize("T", [769, 801, 831, 832, 833, 895, 897, 960, 1023, 3 * 256 + 224])
@pytest.mark.parametrize("K,V,H,block,same_block", [(128, 128, 32, 64, True), (64, 64, 8, 128, True), (64, 128, 32, 512, True), (128, 64, 16, 64, False)])
def test_persistent_kernel_with_a_cut_last_tile(T, K, V, H, block, same_block):
    """Sequences that end inside a tile, a wave's queries or a chunk: bit for bit what the per-tile kernel gives for whole chunks (same
    order, same arithmetic), also where the rows behind a sequence's end, the next one's first, hold NaNs.  The tile of a cut chunk
    goes another way in that kernel (other reference maxima): there both are held to the bound that each is held to against the
    oracle."""
    from neuralattentionsearchlinear_amd import _capi
    B, HQ, HN, dev = 22, 32, 8, torch.device('cuda:0')
    g = torch.Generator(device=dev).manual_seed(31)
    qd, kd, vd = (torch.randn(B, T, h, d, device=dev, generator=g).bfloat16() for h, d in ((HQ, K), (H, K), (H, V)))
    tyd = make_types(B, -(-T // block), HN, 0.4, 32, torch.bfloat16).to(dev)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus == 256:                                        # (three tiles per CU on long cut lengths, eight on others)
        assert [_capi.lib().natsl_softmax_fwd_variant(1, n, HQ, H, block, 0) for n in (6143, 6145, 6208, 2048)] == [1, 2, 1, 1]
    assert _capi.lib().natsl_softmax_fwd_variant(20, T, HQ, H, block, 0) == (1 if 20 * HQ * T < 8 * cus * 256 else 2)
    kd[2, :5] = float('nan')
    vd[2, :5] = float('inf')
    o1, l1 = _call(qd, kd, vd, tyd, K, block, same_block, persistent=False)
    o2, l2 = _call(qd, kd, vd, tyd, K, block, same_block, persistent=True)
    torch.cuda.synchronize()
    rest = [i for i in range(B) if i != 2]
    for x, y in ((o1, o2), (l1, l2)):
        assert bool(torch.isfinite(y[rest]).all())
        whole = T if T % 64 == 0 else T // 256 * 256
        assert torch.equal(x[rest, :whole], y[rest, :whole])
        assert torch.equal(x[2].isnan(), y[2].isnan())
        if whole < T:
            assert_close(y[rest, whole:].float(), x[rest, whole:].float(), "last tile")


@pytest.mark.parametrize("K,V,H,block,same_block", [(128, 128, 32, 64, True), (64, 128, 8, 256, True), (128, 64, 16, 64, False)])
@pytest.mark.parametrize("lens", [[300, 64, 1, 1000, 257, 511, 2048, 63, 12200], [16384, 65], [257] * 64, [257] * 65, [255] * 8 + [256] * 56])
def test_persistent_kernel_on_packed_sequences(lens, K, V, H, block, same_block):
    """Packed sequences, up to as many as the kernel's table holds and one more or shorter ones than a tile (which go to the per-tile
    kernel), against that kernel as above; one sequence holds NaNs."""
    from neuralattentionsearchlinear_amd import _capi, nats_util
    HQ, HN, dev = 32, 8, torch.device('cuda:0')
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    T, bad = cu[-1], 1
    seqs = nats_util.pack_sequences(cu, None, block, dev)
    q, k, v = make_qkv(1, T, H, K, V, 41, HQ=HQ)
    ty = make_types(1, seqs.total_blocks, HN, 0.4, 42, torch.bfloat16)
    k[0, cu[bad]], v[0, cu[bad]] = float('nan'), float('inf')
    qd, kd, vd, tyd = q.to(dev), k.to(dev), v.to(dev), ty.to(dev)
    r = nats_util.route(tyd, T, block, seqs)
    L, out = _capi.lib(), []
    assert L.natsl_softmax_fwd_variant(1, T, HQ, H, block, len(lens)) == (2 if len(lens) <= 64 and T >= 256 * len(lens) else 1)
    for fn in (L.natsl_softmax_sparse_fwd_per_tile, L.natsl_softmax_sparse_fwd):
        o, lse = torch.empty(1, T, HQ, V, dtype=torch.bfloat16, device=dev), torch.empty(1, T, HQ, device=dev)
        rc = fn(_capi.ptr(qd), _capi.ptr(kd), _capi.ptr(vd), _capi.ptr(o), _capi.ptr(lse), _capi.ptr(tyd), _capi.dtype_code(tyd.dtype),
                _capi.ptr(r['nats_block_indices']), _capi.ptr(r['n_nats_blocks']), 1, T, HQ, H, HN, K, V, ty.shape[1], block, float(K ** -0.5),
                int(same_block), _capi.dtype_code(qd.dtype), _capi.ptr(seqs.table), seqs.n_seqs, seqs.total_qtiles, _capi.stream_ptr(dev))
        _capi.check(rc, "softmax")
        out.append((o[0], lse[0]))
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(cu[:-1], cu[1:])):
        whole = b if (b - a) % 64 == 0 else a + (b - a) // 256 * 256
        for x, y in zip(*out):
            assert torch.equal(x[a:b].isnan(), y[a:b].isnan())
            if i == bad:
                continue
            assert bool(torch.isfinite(y[a:b]).all()) and torch.equal(x[a:whole], y[a:whole])
            if whole < b:
                assert_close(y[whole:b].float(), x[whole:b].float(), f"sequence {i}")


@pytest.mark.parametrize("K,V", [(128, 128), (64, 64), (64, 128), (128, 64)])
@pytest.mark.parametrize("T,packed", [(769, False), (831, False), (897, False), (1023, False), (831, True)])
def test_row_sums_of_a_cut_last_tile_are_fp32(K, V, T, packed):
    """The log-sum-exp of the tile that a sequence's end cuts inside a chunk, against 64-bit arithmetic on the scaled bf16 queries that
    the kernel multiplies.  With fp32 probabilities in the sums it is off by the rounding of K products of a few units (K 2^-24 x 8 at
    most, 6e-5 for 128 aligned signs, 1.5e-6 seen) and of at most T additions whose partial sums are below 2^3 of the result; 1e-5 lies
    between that and probabilities rounded to bf16 (2^-9 each: 1.6e-4 on average, 5e-4 to 1.4e-3 at most)."""
    import math
    from neuralattentionsearchlinear_amd import nats_util
    B, H, block, dev = 22, 32, 64, torch.device('cuda:0')
    g = torch.Generator(device=dev).manual_seed(T)
    q, k, v = (torch.randn(B, T, H, d, device=dev, generator=g).bfloat16() for d in (K, K, V))
    ty = make_types(B, -(-T // block), H, 0.4, 33, torch.bfloat16).to(dev)
    one_row = lambda t: t.reshape(1, -1, *t.shape[2:])
    for persistent in (False, True):
        if packed:
            seqs = nats_util.pack_sequences([T * i for i in range(B + 1)], None, block, dev)
            _, lse = _call(one_row(q), one_row(k), one_row(v), one_row(ty), K, block, True, persistent, seqs)
            lse = lse.view(B, T, H)
        else:
            _, lse = _call(q, k, v, ty, K, block, True, persistent)
        b, whole = 3, T // 256 * 256
        scale = torch.tensor(K ** -0.5, dtype=torch.float32, device=dev) * 1.4426950408889634
        qs = (q[b].float() * scale).bfloat16().double()
        s = torch.matmul(qs[whole:].transpose(0, 1).contiguous(), k[b].double().permute(1, 2, 0).contiguous())      # [H, queries, keys], log2 units
        i, j = torch.arange(whole, T, device=dev)[:, None], torch.arange(T, device=dev)[None]
        typed = (ty[b, :, :, 0] > 0.5).T[:, torch.arange(T, device=dev) // block][:, None, :]
        seen = (j <= i) & ((j // block == i // block) | typed)
        ref = torch.logsumexp(torch.where(seen, s * math.log(2), torch.full_like(s, -1e300)), -1) / math.log(2)
        worst = float((lse[b, whole:].T.double() - ref).abs().max())
        assert worst <= 1e-5, f"persistent {persistent}: {worst:.2e}"


def test_operator_and_entry_agree_on_a_cut_length():
    """The same tiles from work queues (the operators) and dealt out (the entry): the same bits."""
    import torch.nn.functional as F
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    B, T, H, D, block, dev = 22, 1023, 32, 64, 64, torch.device('cuda:0')
    _, _, _, _, q, k, v, ty = _inputs(B, T, H, H, H, D, D, block, 0.4, 8, dev)
    beta, g = torch.sigmoid(torch.randn(B, T, H, device=dev)).bfloat16(), -F.softplus(torch.randn(B, T, H, device=dev))
    with torch.no_grad():
        out = nats_mixed_attn_gdn(q, k, v, q, k, v, None, g, beta, ty, None, ops_for_incomplete_chunks='all')
    assert torch.equal(out[1], _call(q, k, v, ty, D, block, True)[0])


def test_persistent_kernel_queues_across_launches_and_streams():
    """The ticket counters are shared device state: one slot per launch in rotation, zeroed on the launch's stream right
    before it."""
    B, T, HQ, H, HN, K, V, block = 4, 4096, 16, 16, 16, 128, 128, 64
    dev = torch.device('cuda:0')
    assert _enough_tiles(B, HQ, T)
    _, _, _, _, qd, kd, vd, tyd = _inputs(B, T, HQ, H, HN, K, V, block, 0.25, 5, dev)
    _, _, _, _, qe, ke, ve, tye = _inputs(B, T, HQ, H, HN, K, V, block, 0.5, 6, dev)
    o_ref, l_ref = _call(qd, kd, vd, tyd, K, block, True, persistent=False)
    o_ref2, l_ref2 = _call(qe, ke, ve, tye, K, block, True, persistent=False)
    torch.cuda.synchronize()
    for _ in range(70):   # more launches than there are slots
        o, l = _call(qd, kd, vd, tyd, K, block, True)
    torch.cuda.synchronize()
    assert torch.equal(o, o_ref) and torch.equal(l, l_ref)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()   # default priority
    s1.wait_stream(torch.cuda.current_stream())
    s2.wait_stream(torch.cuda.current_stream())
    outs = []
    for _ in range(4):
        with torch.cuda.stream(s1):
            outs.append((_call(qd, kd, vd, tyd, K, block, True), (o_ref, l_ref)))
        with torch.cuda.stream(s2):
            outs.append((_call(qe, ke, ve, tye, K, block, True), (o_ref2, l_ref2)))
    s1.synchronize()
    s2.synchronize()
    for (o, l), (orf, lrf) in outs:
        assert torch.equal(o, orf) and torch.equal(l, lrf)


def test_persistent_kernel_in_a_captured_graph():
    """The launch (queue fill kernel + persistent kernel) replays from a HIP graph: every replay, with eager work and
    synchronisations between the replays, gives the eager result."""
    B, T, HQ, H, HN, K, V, block = 4, 4096, 16, 16, 16, 128, 128, 64
    dev = torch.device('cuda:0')
    assert _enough_tiles(B, HQ, T)
    _, _, _, _, qd, kd, vd, tyd = _inputs(B, T, HQ, H, HN, K, V, block, 0.25, 7, dev)
    from neuralattentionsearchlinear_amd import _capi, nats_util
    r = nats_util.route(tyd, T, block)
    o_ref, l_ref = _call(qd, kd, vd, tyd, K, block, True, persistent=False)
    o = torch.empty_like(o_ref)
    lse = torch.empty_like(l_ref)
    L = _capi.lib()

    def launch():
        rc = L.natsl_softmax_sparse_fwd(_capi.ptr(qd), _capi.ptr(kd), _capi.ptr(vd), _capi.ptr(o), _capi.ptr(lse), _capi.ptr(tyd),
                                        _capi.dtype_code(tyd.dtype), _capi.ptr(r['nats_block_indices']), _capi.ptr(r['n_nats_blocks']),
                                        B, T, HQ, H, HN, K, V, tyd.shape[1], block, float(K ** -0.5), 1, _capi.dtype_code(qd.dtype),
                                        None, 0, 0, _capi.stream_ptr(dev))
        _capi.check(rc, "natsl_softmax_sparse_fwd")

    launch()   # first use on the device outside the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        launch()
    for i in range(4):
        o.fill_(float('nan'))
        lse.fill_(float('nan'))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, o_ref) and torch.equal(lse, l_ref), f"replay {i}"
        if i & 1:
            _call(qd, kd, vd, tyd, K, block, True)   # an eager launch between replays, on the same stream
            torch.cuda.synchronize()
