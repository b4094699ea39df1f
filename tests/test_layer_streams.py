"""CPU-only: which of a layer's native calls put the softmax branch on a second stream, at both sides of the rule's lines (256 compute units)."""
import pytest
import torch

import neuralattentionsearchlinear_amd._mixed_common as MC

HOW = dict(gdn_340M=dict(D=1024, widths=(768, 768, 1536, 1536), H=6, K=128, V=256), gdn_760M=dict(D=1536, widths=(1152, 1152, 2304, 2304), H=6, K=192, V=384),
           mamba=dict(D=1024, widths=(2048, 2048, 1024, 1024), H=16, K=128, V=64))


@pytest.mark.parametrize("geometry,B,T,training,forward", [
    ("gdn_340M", 1, 256, False, False), ("gdn_340M", 4, 1024, False, False), ("gdn_340M", 6, 1024, True, False), ("gdn_340M", 1, 1500, False, False), ("gdn_340M", 1, 2048, True, False),
    ("gdn_340M", 1, 3000, True, False), ("gdn_340M", 3, 2048, True, False), ("gdn_340M", 4, 2048, True, True), ("gdn_340M", 8, 4096, True, True),
    ("gdn_340M", 1, 16384, True, True), ("gdn_760M", 1, 1200, False, False), ("gdn_760M", 1, 1536, True, False), ("gdn_760M", 1, 3000, True, True), ("gdn_760M", 2, 1536, True, False),
    ("gdn_760M", 7, 4096, False, False),                   # 252 workgroups of the scan: it leaves four compute units
    ("mamba", 8, 2047, True, False), ("mamba", 8, 2048, True, True), ("mamba", 1, 1536, False, False), ("mamba", 2, 1536, True, False), ("mamba", 16, 4096, False, False)])
def test_where_a_layers_softmax_branch_runs(geometry, B, T, training, forward, monkeypatch):
    monkeypatch.setitem(MC._cu_counts, 0, 256)
    dev = torch.device('cuda:0')
    assert [MC._layer_runs_side_by_side(dev, B, T, HOW[geometry], g) for g in (True, False)] == [training, forward]
    for forced in (True, False):
        monkeypatch.setattr(MC, 'CONCURRENT_BRANCHES', forced)
        assert [MC._layer_runs_side_by_side(dev, B, T, HOW[geometry], g) for g in (True, False)] == [forced, forced]
