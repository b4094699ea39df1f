"""The mixed operator's one native call: fp32 tensors converted inside it give what tensors rounded beforehand give, bit for bit, at
sizes where a conversion segment ends inside a thread's eight elements or a workgroup's 2048; and both placements of the softmax
branch (same stream, side stream) agree."""
import pytest
import torch

from tests._util import make_gates, make_qkv, make_types

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _case(kind, B, T, H, K, V, seed):
    q, k, v = make_qkv(B, T, H, K, V, seed, torch.float32)
    g, beta = make_gates(B, T, H, seed + 1, torch.float32)
    ty = make_types(B, -(-T // 64), H, 0.4, seed + 2)
    return [t.to(DEV) for t in (q, k, v, g, beta, ty)]


def _run(kind, q, k, v, g, beta, ty):
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    from neuralattentionsearchlinear_amd.mixed_attn_mamba import nats_mixed_attn_mamba
    if kind == 'gdn':
        return nats_mixed_attn_gdn(q, k, v, q, k, v, None, g, beta, ty, None, ops_for_incomplete_chunks='all',
                                   output_final_state_gated_delta=True, decay_for_non_gdn_blocks=True)
    return nats_mixed_attn_mamba(q, k, v, q, k, v, None, g, ty, None, output_final_state_mamba=True, decay_for_non_mamba_blocks=True)


@pytest.mark.parametrize("kind,B,T,H,K,V", [('gdn', 1, 1, 1, 64, 64), ('gdn', 1, 67, 3, 64, 64), ('gdn', 2, 129, 5, 128, 128), ('mamba', 1, 100, 3, 128, 64)])
@pytest.mark.parametrize("grad", [False, True])
def test_fp32_tensors_equal_rounded_tensors(kind, B, T, H, K, V, grad):
    q, k, v, g, beta, ty = _case(kind, B, T, H, K, V, T)
    r16 = lambda t: t.bfloat16()
    if grad:                                              # the differentiable operator keeps its copies as tensors of their own
        q.requires_grad_(True)
    out = _run(kind, q, k, v, g, beta, ty)
    ref = _run(kind, r16(q.detach()), r16(k), r16(v), g, r16(beta), ty)
    for name, a, b in zip(("o_linear", "o_attn", "state"), out, ref):
        assert a.dtype == torch.float32
        assert torch.equal(a.detach(), b.float()), name


@pytest.mark.parametrize("kind,B,H,K,V", [('gdn', 1, 2, 64, 64), ('mamba', 1, 3, 128, 64),
                                          # the scan's width depends on what it leaves: 1, 2, 4 waves, several rounds
                                          ('gdn', 5, 13, 64, 64), ('gdn', 9, 15, 128, 128), ('gdn', 11, 24, 128, 64),
                                          ('mamba', 5, 13, 128, 64), ('mamba', 9, 15, 64, 128)])
def test_side_stream_and_one_stream_agree(kind, B, H, K, V, monkeypatch):
    import neuralattentionsearchlinear_amd._mixed_common as MC
    q, k, v, g, beta, ty = _case(kind, B, 500 if B == 1 else 130, H, K, V, 9)
    outs = []
    for side in (False, True):
        monkeypatch.setattr(MC, 'CONCURRENT_BRANCHES', side)
        outs.append(_run(kind, q, k, v, g, beta, ty))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("T,seqs", [(1023, 17), (1024, 17)])
def test_captured_operator_replays_beside_other_launches(T, seqs):
    """A captured forward whose softmax branch is the persistent kernel, replayed while eager launches of that kernel run on another
    stream (more of them than the library has slots): the operator's work queues are its own."""
    from neuralattentionsearchlinear_amd import _capi
    from tests.test_gpu_softmax_stream import _call, _inputs
    H = 32
    assert _capi.lib().natsl_softmax_fwd_variant(seqs, T, H, H, 64, 0) == 2, "shape does not reach the persistent kernel on this GPU"
    q, k, v, g, beta, ty = _case('gdn', seqs, T, H, 64, 64, 3)
    args = [t.bfloat16() for t in (q, k, v)] + [g, beta.bfloat16(), ty.bfloat16()]
    _, _, _, _, qe, ke, ve, te = _inputs(4, 4096, 16, 16, 16, 64, 64, 64, 0.25, 5, torch.device(DEV))
    with torch.no_grad():
        ref = [t.clone() for t in _run('gdn', *args)]
        other_ref = _call(qe, ke, ve, te, 64, 64, True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = _run('gdn', *args)
        other = torch.cuda.Stream()                       # default priority
        for i in range(3):
            for t in out:
                t.fill_(float('nan'))
            torch.cuda.synchronize()
            with torch.cuda.stream(other):
                o = [_call(qe, ke, ve, te, 64, 64, True) for _ in range(35)]
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, ref)), f"replay {i}"
            assert all(torch.equal(a, b) for pair in o for a, b in zip(pair, other_ref)), f"beside replay {i}"
