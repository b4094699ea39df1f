"""Small calls' softmax tiles and linear prep in one launch against the same branches on two streams, where each has its own, bit for bit: one token, cut
chunks and tiles, the last size that one launch takes and the first that it does not, all pairs of head widths, both linear forms, with and without
the chunk states for a backward."""
import pytest
import torch

from tests._util import make_gates, make_qkv, make_types

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


# kind, B, T, H, head widths of the softmax branch, of the linear branch, block, whether one launch takes both (test_kernel_choices.py)
CASES = [
    ('gdn', 1, 1, 1, 64, 64, 64, 64, 64, True), ('gdn', 3, 65, 3, 64, 64, 64, 64, 64, True), ('gdn', 1, 256, 2, 64, 128, 64, 128, 64, True),
    ('gdn', 2, 333, 4, 128, 64, 128, 64, 128, True), ('gdn', 1, 1000, 4, 128, 128, 128, 128, 256, True), ('gdn', 2, 300, 6, 64, 128, 192, 128, 64, True),
    ('gdn', 1, 777, 6, 64, 128, 128, 256, 64, True), ('gdn', 1, 200, 2, 128, 128, 64, 64, 64, False), ('gdn', 1, 1344, 8, 64, 64, 64, 64, 64, True),
    ('gdn', 1, 1345, 8, 64, 64, 64, 64, 64, True), ('gdn', 120, 64, 1, 128, 128, 128, 128, 64, True), ('mamba', 1, 1, 1, 64, 64, 64, 64, 64, True),
    ('mamba', 2, 333, 17, 128, 64, 128, 64, 256, True), ('mamba', 1, 700, 5, 64, 128, 192, 128, 64, True), ('mamba', 1, 1500, 16, 128, 128, 128, 128, 64, True),
    ('gdn', 1, 3839, 16, 64, 64, 64, 64, 64, True), ('gdn', 1, 3841, 16, 64, 64, 64, 64, 64, False)]    # (of 16 heads: one tile of 256 queries a CU)


@pytest.mark.parametrize("gradients", [False, True])
@pytest.mark.parametrize("kind,B,T,H,KA,VA,K,V,block", [c[:-1] for c in CASES])
def test_one_launch_gives_what_two_give(kind, B, T, H, KA, VA, K, V, block, gradients, monkeypatch):
    import neuralattentionsearchlinear_amd._mixed_common as MC
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    from neuralattentionsearchlinear_amd.mixed_attn_mamba import nats_mixed_attn_mamba
    qa, ka, va = (t.to(DEV) for t in make_qkv(B, T, H, KA, VA, 1, torch.bfloat16))
    q, k, v = (t.to(DEV) for t in make_qkv(B, T, H, K, V, 2, torch.bfloat16))
    g, beta = (t.to(DEV) for t in make_gates(B, T, H, 3, torch.bfloat16))
    types = make_types(B, -(-T // block), H, 0.4, 4).to(DEV)

    def run(two_streams):
        monkeypatch.setattr(MC, 'CONCURRENT_BRANCHES', two_streams)
        leaves = [t.detach().clone().requires_grad_(gradients) for t in (qa, ka, va, q, k, v)]
        kw = dict(nats_block_size=block, ops_for_incomplete_chunks='all', compute_dnats_for_invalid_blocks_linear_att=False)
        with torch.set_grad_enabled(gradients):
            if kind == 'gdn':
                out = nats_mixed_attn_gdn(*leaves, None, g.float(), beta, types, None, output_final_state_gated_delta=True, **kw)
            else:
                out = nats_mixed_attn_mamba(*leaves, None, g.float(), types, None, output_final_state_mamba=True, **kw)
        if gradients:
            (out[0].float().sum() + out[1].float().square().sum()).backward()
        torch.cuda.synchronize()
        return [t for t in out if torch.is_tensor(t)] + [t.grad for t in leaves if gradients]
    one, two = run(False), run(True)
    assert len(one) == len(two) and all(torch.isfinite(a).all() and torch.equal(a, b) for a, b in zip(one, two))
