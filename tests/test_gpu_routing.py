"""GPU parity (bit-exact): selector, pooling and routing tables through the C ABI vs the oracle."""
import pytest
import torch

from oracle import routing as R
from tests._util import make_types
from tests.test_oracle_routing import _bf16_neighbours

pytestmark = pytest.mark.gpu


def _dev():
    return torch.device('cuda:0')


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_hard_select_random(dtype):
    from neuralattentionsearchlinear_amd import nats_util
    g = torch.Generator().manual_seed(0)
    logits = torch.randn(8, 128, 16, 2, generator=g).to(dtype)
    ref = R.hard_select(logits)
    ty, nb = nats_util.hard_select(logits.to(_dev()))
    assert torch.equal(ty.cpu(), ref)
    assert torch.equal(nb.cpu(), R.n_blocks(ref))
    ty2, nb2 = nats_util.hard_select(logits.to(_dev()), force_last_block=True)
    ref2 = R.force_last_block(ref)
    assert torch.equal(ty2.cpu(), ref2)
    assert torch.equal(nb2.cpu(), R.n_blocks(ref2))


def test_hard_select_bf16_near_ties_exhaustive():
    """every positive/negative normal bf16 paired with its 0..6-ulp neighbours, both orders"""
    from neuralattentionsearchlinear_amd import nats_util
    lg = _bf16_neighbours(6)
    lg = torch.cat([lg, lg.flip(-1)], 0)
    n = lg.shape[0]
    ref = R.hard_select(lg)
    ty, _ = nats_util.hard_select(lg.view(1, n, 1, 2).to(_dev()))
    assert torch.equal(ty.cpu().view(n, 2), ref)


def test_hard_select_fp32_near_ties():
    from neuralattentionsearchlinear_amd import nats_util
    g = torch.Generator().manual_seed(1)
    x0 = torch.randn(200000, generator=g)
    ulps = torch.randint(-3, 4, (200000,), generator=g)
    x1 = (x0.view(torch.int32) + ulps.int()).view(torch.float32)
    lg = torch.stack([x0, x1], -1)
    ref = R.hard_select(lg)
    ty, _ = nats_util.hard_select(lg.view(1, -1, 1, 2).to(_dev()))
    assert torch.equal(ty.cpu().view(-1, 2), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,D,block", [(2, 512, 256, 64), (3, 200, 96, 64), (1, 1000, 130, 256)])
def test_mean_pool(B, T, D, block, dtype):
    from neuralattentionsearchlinear_amd import nats_util
    g = torch.Generator().manual_seed(2)
    x = torch.randn(B, T, D, generator=g).to(dtype)
    ref = R.mean_pool(x, block)
    out = nats_util.mean_pooling(x.to(_dev()), block)
    # sums of <=256 values in fp32: the summation order may differ, so allow 1 ulp of the output dtype
    tol = 2 ** -7 if dtype == torch.bfloat16 else 1e-6
    assert float((out.cpu().float() - ref.float()).abs().max()) <= tol * float(ref.float().abs().max())


@pytest.mark.parametrize("B,TN,HN,block,p", [(1, 4, 1, 64, 0.5), (8, 128, 16, 64, 0.25), (2, 1024, 4, 64, 0.1), (3, 33, 5, 256, 0.6), (2, 16, 2, 128, 0.0), (2, 16, 2, 64, 1.0)])
def test_route_tables(B, TN, HN, block, p):
    from neuralattentionsearchlinear_amd import nats_util
    T = TN * block
    for dtype in (torch.bfloat16, torch.float32):
        ty = make_types(B, TN, HN, p, seed=TN + HN, dtype=dtype)
        ref = R.route(ty, T, block)
        got = nats_util.route(ty.to(_dev()), T, block, tables=True)
        torch.cuda.synchronize()
        assert torch.equal(got['nats_block_indices'].cpu(), ref['nats_block_indices'])
        assert torch.equal(got['n_nats_blocks'].cpu(), ref['n_nats_blocks'])
        assert torch.equal(got['linear_chunk_offsets'].cpu(), ref['linear_chunk_offsets'])
        n = int(ref['linear_chunk_offsets'][-1])
        assert torch.equal(got['chunk_indices_linear_buffer'][:n].cpu(), ref['chunk_indices_linear'])
        assert torch.equal(got['starting_h_idx'].cpu(), ref['starting_h_idx'])
        assert torch.equal(got['attn_n_iters'].cpu(), ref['attn_n_iters'])
        # the torch re-statements of the two host helpers agree too
        ci = nats_util.prepare_nats_block_indices(got['n_nats_blocks'][..., 1], block, 64)
        assert torch.equal(ci.cpu().int(), ref['chunk_indices_linear'])
        off = nats_util.prepare_nats_chunk_offsets(got['n_nats_blocks'], None, block, 64, 1)
        assert torch.equal(off.cpu(), ref['linear_chunk_offsets'])


def test_route_known_answer():
    from neuralattentionsearchlinear_amd import nats_util
    types = torch.tensor([[1, 0], [0, 1], [1, 0], [1, 1]], dtype=torch.float32).view(1, 4, 1, 2)
    got = nats_util.route(types.to(_dev()), 256, 64, tables=True)
    assert got['nats_block_indices'][0, :, 0, 0].tolist() == [0, 2, 3, 4]
    assert got['nats_block_indices'][0, :, 0, 1].tolist() == [1, 3, 4, 4]
    assert got['n_nats_blocks'][0, 0].tolist() == [3, 2]
    assert got['linear_chunk_offsets'].tolist() == [0, 2]
    assert got['starting_h_idx'][0, :, 0].tolist() == [0, 0, 1, 1]
    assert got['attn_n_iters'][0, :, 0].tolist() == [0, 1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,TN,HN", [(1, 1, 1), (3, 1025, 2), (513, 3, 5), (8, 64, 6)])     # around a workgroup's threads and sequences
def test_layer_select(B, TN, HN, dtype):
    """One launch gives what the two selections and torch's arithmetic on the counts give, bit for bit."""
    from neuralattentionsearchlinear_amd import _front, nats_util
    g = torch.Generator().manual_seed(B)
    logits = torch.randn(B, TN, HN, 2, generator=g).to(dtype)
    raw = R.hard_select(logits)
    forced = R.force_last_block(raw)
    for want in (True, False):
        types, counts, fraction, before = _front._select(logits.to(_dev()), want)
        assert torch.equal(types.cpu(), forced) and torch.equal(counts.cpu(), R.n_blocks(forced))
        assert torch.equal(before.cpu(), raw) if want else before is None
        assert torch.equal(fraction, nats_util.hard_select(logits.to(_dev()), True)[1][..., 0].sum(0).float() / (TN * B))


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 512, 513])           # around a launch's 64 rows and the most that launches carry
def test_table_of_packed_sequences(n):
    from neuralattentionsearchlinear_amd import nats_util
    lens = torch.randint(1, 400, (n,), generator=torch.Generator().manual_seed(n)).tolist()
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    before = lambda unit: [sum(-(-x // unit) for x in lens[:i]) for i in range(n)]
    ref = torch.tensor([[cu[i], cu[i + 1], b, c, t, 0, 0, 0] for i, (b, c, t) in enumerate(zip(before(128), before(64), before(256)))])
    for make in (nats_util.pack_sequences, nats_util.pack_sequences_here):
        seqs = make(torch.tensor(cu, device=_dev()), None, 128, _dev())
        assert seqs.table.dtype == torch.int32 and torch.equal(seqs.table.cpu().long(), ref)
        assert (seqs.n_seqs, seqs.total_chunks, seqs.total_qtiles) == (n, before(64)[-1] + -(-lens[-1] // 64), before(256)[-1] + -(-lens[-1] // 256))


@pytest.mark.parametrize("n", [3, 512, 513])
def test_a_packed_table_is_complete_when_it_is_handed_out(n):
    """A table made on a stream that still has work in front of it is there for every other stream as soon as the call returns."""
    from neuralattentionsearchlinear_amd import nats_util
    cu = [100 * i for i in range(n + 1)]
    maker, taker = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(maker):
            torch.full((n, 8), -1, dtype=torch.int32, device=_dev())          # (what a table not yet written would hold)
            torch.cuda._sleep(20_000_000)
            seqs = nats_util.pack_sequences(cu, None, 64, _dev())
        with torch.cuda.stream(taker):
            got = seqs.table.cpu()
        assert got[:, 0].tolist() == cu[:-1] and got[:, 1].tolist() == cu[1:]
        torch.cuda.synchronize()


@pytest.mark.parametrize("lens", [[1] * 70, [64, 128, 64], [65, 1, 127, 300], [2500, 700, 3, 1900]])
def test_boundaries_on_the_gpu_or_on_the_host(lens):
    """Boundaries that the call reads back behind its preparations (its workspace sized by what they can be at most) give the same bits."""
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    g = torch.Generator(device=_dev()).manual_seed(3)
    rn = lambda *s: torch.randn(*s, device=_dev(), generator=g)
    T, NB = cu[-1], sum(-(-x // 64) for x in lens)
    q, k, v, beta = rn(1, T, 2, 64).bfloat16(), rn(1, T, 2, 64).bfloat16(), rn(1, T, 2, 64).bfloat16(), torch.sigmoid(rn(1, T, 2)).bfloat16()
    ty = torch.nn.functional.one_hot((rn(1, NB, 2) > 0).long(), 2).bfloat16()
    out = [nats_mixed_attn_gdn(q, k, v, q, k, v, None, -torch.nn.functional.softplus(rn(1, T, 2) * 0 + 1), beta, ty, None, cu_seqlens=c, nats_block_size=64,
                               ops_for_incomplete_chunks="all", output_final_state_gated_delta=True, decay_for_non_gdn_blocks=True)
           for c in (cu, torch.tensor(cu, device=_dev()), torch.tensor(cu, dtype=torch.int32, device=_dev()))]
    for o in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(o, out[0]))


@pytest.mark.parametrize("lens", [[1] * 70, [65, 1, 127, 300], [2500, 700, 3, 1900]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_boundaries_on_the_gpu_on_one_stream_and_two(lens, dtype, monkeypatch):
    """The same with the branches on one stream and side by side (the table is stored behind what the side stream waits for), with a state
    to start from, and with fp32 tensors, whose copies are laid out before the table is there."""
    from neuralattentionsearchlinear_amd import _mixed_common as MC
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    gen = torch.Generator(device=_dev()).manual_seed(3)
    rn = lambda *s: torch.randn(*s, device=_dev(), generator=gen)
    T, NB = cu[-1], sum(-(-x // 64) for x in lens)
    q, k, v, beta = rn(1, T, 2, 64).to(dtype), rn(1, T, 2, 64).to(dtype), rn(1, T, 2, 64).to(dtype), torch.sigmoid(rn(1, T, 2)).to(dtype)
    g, h0 = -torch.nn.functional.softplus(rn(1, T, 2)), rn(len(lens), 2, 64, 64)
    ty = torch.nn.functional.one_hot((rn(1, NB, 2) > 0).long(), 2).bfloat16()

    def outputs(c, side):
        monkeypatch.setattr(MC, 'CONCURRENT_BRANCHES', side)
        return nats_mixed_attn_gdn(q, k, v, q, k, v, h0, g, beta, ty, None, cu_seqlens=c, nats_block_size=64, ops_for_incomplete_chunks="all",
                                   output_final_state_gated_delta=True, decay_for_non_gdn_blocks=True)
    want = outputs(cu, False)
    for c, side in ((cu, True), (torch.tensor(cu, device=_dev()), False), (torch.tensor(cu, device=_dev()), True), (torch.tensor(cu, dtype=torch.int32, device=_dev()), True)):
        assert all(torch.equal(a, b) for a, b in zip(outputs(c, side), want))
    with pytest.raises(ValueError):
        nats_mixed_attn_gdn(q, k, v, q, k, v, h0[1:], g, beta, ty, None, cu_seqlens=torch.tensor(cu, device=_dev()), nats_block_size=64,
                            ops_for_incomplete_chunks="all", output_final_state_gated_delta=True, decay_for_non_gdn_blocks=True)
