"""The softmax kernels of one workgroup a tile on the blocks' types alone against the same on a routing table, bit for bit: numbers of blocks around a
wave's 64 and the most that are taken without a table, both kernels, selector heads shared and not, types of either dtype, all and no attention."""
import pytest
import torch

from tests._util import make_gates, make_qkv, make_types

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


CASES = [
    (1, 1, 2, 2, 64, 0.5, False), (2, 3, 2, 1, 64, 1.0, True), (5, 40, 16, 16, 64, 0.4, False), (5, 40, 16, 4, 128, 0.4, False), (63, 1, 4, 2, 64, 0.3, True),
    (64, 2, 2, 2, 64, 0.0, False), (65, 1, 4, 4, 64, 0.5, False), (129, 1, 2, 1, 128, 0.2, False), (193, 2, 1, 1, 64, 1.0, True), (255, 1, 1, 1, 64, 0.7, False),
    (256, 1, 2, 2, 64, 0.1, False), (257, 1, 1, 1, 64, 0.3, False)]


@pytest.mark.parametrize("blocks,B,H,HN,block,share,wide", CASES)
def test_tiles_find_their_blocks_in_the_types(blocks, B, H, HN, block, share, wide, monkeypatch):
    import neuralattentionsearchlinear_amd._mixed_common as MC
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd.mixed_attn_gdn import nats_mixed_attn_gdn
    T = blocks * block - (17 if blocks > 1 else 0)
    q, k, v = (t.to(DEV) for t in make_qkv(B, T, H, 64, 64, blocks, torch.bfloat16))
    g, beta = (t.to(DEV) for t in make_gates(B, T, H, blocks + 1, torch.bfloat16))
    types = make_types(B, blocks, HN, share, blocks + 2).to(DEV)
    types = types.float() if wide else types.bfloat16()
    assert _capi.lib().natsl_mixed_softmax_variant(B, T, H, H, block, 0) != 2, "the case takes the persistent kernel on this GPU"

    def run():
        with torch.no_grad():
            return nats_mixed_attn_gdn(q, k, v, q, k, v, None, g.float(), beta, types, None, nats_block_size=block, ops_for_incomplete_chunks='all')
    native = run()
    monkeypatch.setattr(MC, '_plain_forward', lambda *a: None)
    general = run()

    class WithTables(MC._Mixed):
        private_tables = property(lambda self: 0, lambda self, x: None)
    monkeypatch.setattr(MC, '_Mixed', WithTables)
    tables = run()
    for a, b, c in zip(native[:2], general[:2], tables[:2]):
        assert torch.equal(a, c) and torch.equal(b, c)
