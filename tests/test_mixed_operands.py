"""CPU-only: which tensors the mixed operators take together (_mixed_common._check_operands), on tensors without memory."""
import pytest
import torch

import neuralattentionsearchlinear_amd._mixed_common as MC
from neuralattentionsearchlinear_amd.nats_util import pack_sequences

B, T, H, K, V, HQ, HKV, KA, VA, TN, HN = 2, 130, 4, 64, 128, 8, 2, 128, 64, 3, 2
NAMES = ('q_attn', 'k_attn', 'v_attn', 'q', 'k', 'v', 'g', 'beta', 'types')
SHAPES = dict(zip(NAMES, ((B, T, HQ, KA), (B, T, HKV, KA), (B, T, HKV, VA), (B, T, H, K), (B, T, H, K), (B, T, H, V), (B, T, H), (B, T, H), (B, TN, HN, 2))))


def _check(n_prefix=0, device=None, **changed):
    made = {n: None if s is None else torch.empty(s, device='meta') for n, s in {**SHAPES, **changed}.items()}
    if device:
        made[device] = torch.empty(made[device].shape)
    MC._check_operands(**made, n_prefix=n_prefix)


@pytest.mark.parametrize("fits", [dict(), dict(beta=None), dict(g=(B, T, H, 1)), dict(q_attn=(B, 140, HQ, KA), k_attn=(B, 140, HKV, KA), v_attn=(B, 140, HKV, VA)),
                                  dict(n_prefix=128, k_attn=(B, T + 128, HKV, KA), v_attn=(B, T + 128, HKV, VA)), dict(types=(B, 7, H, 2))])
def test_taken(fits):
    _check(**fits)


@pytest.mark.parametrize("name", [n for n in NAMES if n != 'q'])
def test_another_size_is_refused(name):
    shape = SHAPES[name]
    sizes = {'types': (0,), 'g': (0, 1, 2), 'beta': (0, 1, 2), 'v': (0, 1, 2), 'v_attn': (0, 1, 2), 'k_attn': (0, 1, 3), 'q_attn': (0,), 'k': (0, 1, 2, 3)}[name]
    for i in sizes:                                        # (the others are the tensor's own: head counts and value widths, which the entry points look at)
        for n in (shape[i] - 1, shape[i] + 1):
            with pytest.raises(ValueError):
                _check(**{name: shape[:i] + (n,) + shape[i + 1:]})
    for other in (shape[:-1], (*shape, 2), (shape[1], shape[0], *shape[2:])):
        with pytest.raises(ValueError):
            _check(**{name: other})
    with pytest.raises(ValueError, match="is on cpu"):
        _check(device=name)


def test_keys_without_their_prefix_are_refused():
    with pytest.raises(ValueError):
        _check(n_prefix=128)


def test_packed_sequences_lie_in_their_rows():
    seqs = pack_sequences([0, 70, 130], None, 64, 'cpu')
    MC._check_packed(None, 1, 1, 1)
    MC._check_packed(seqs, 130, 140, 3)
    for T_, T_attn, TN_ in ((129, 130, 3), (130, 129, 3), (130, 130, 2)):
        with pytest.raises(ValueError):
            MC._check_packed(seqs, T_, T_attn, TN_)
    for cu, nats in (([-64, 64], None), ([0, 64], [-1, 0])):
        with pytest.raises(ValueError):
            MC._check_packed(pack_sequences(cu, nats, 64, 'cpu'), 1000, 1000, 100)
