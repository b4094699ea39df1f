"""CPU-only: how a one-token step is launched, by batch, cached tokens and geometry, seen from what a HIP runtime that launches nothing
(tests/fake_hip.c) is asked to launch.  The expected splits are those that a sweep over all of them found within a few percent of the
fastest."""
import json
import os
import subprocess
import sys

import pytest

from tests.test_stream_order import fake_hip  # noqa: F401

CHILD = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
lib.natsl_layer_step_workspace_bytes.restype = ctypes.c_size_t
for step in json.loads(sys.argv[3]):
    fake.fake_reset(0)
    s = ctypes.create_string_buffer(bytes.fromhex(step))
    rc = lib.natsl_layer_step_fwd(s, ctypes.c_void_p(1 << 20), ctypes.c_size_t(lib.natsl_layer_step_workspace_bytes(s)), ctypes.c_void_p(0x10))
    out.append([rc, fake.fake_launches().decode()])
print(json.dumps(out))
"""
# H, K, V, HQ, the delta rule
GEOMETRY = dict(gdn_340M=(6, 128, 256, 12, 1), gdn_760M=(6, 192, 384, 18, 1), mamba=(16, 128, 64, 16, 0), wide=(8, 128, 128, 8, 1))


def _splits(fake_hip, cases):
    """[splits of the one launch, or None where the step is several launches] of cases (geometry, sequences, cached tokens)."""
    from neuralattentionsearchlinear_amd import _build, _capi
    from neuralattentionsearchlinear_amd._layer_step import _TENSORS, _WEIGHTS, LayerStep
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    steps = []
    for geometry, B, tokens in cases:
        s = LayerStep()
        for n in _WEIGHTS + _TENSORS:
            setattr(s, n, 1 << 20)
        s.H, s.K, s.V, s.HQ, s.is_delta = GEOMETRY[geometry]
        s.B, s.T, s.D, s.HN, s.block, s.conv_width = B, 1, 1024, 1, 64, 4
        s.n_kept, s.n_in, s.cache_tokens = (tokens - 1) // 64, (tokens - 1) % 64, -(-tokens // 64) * 64
        s.types_dtype = s.norm_dtype = s.gate_dtype = s.out_norm_dtype = _capi.BF16
        steps.append(bytes(s).hex())
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, _capi.LIB_PATH, json.dumps(steps)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = []
    for (geometry, B, _), (rc, text) in zip(cases, json.loads(r.stdout)):
        assert rc == 0
        H, K, V, HQ, _ = GEOMETRY[geometry]
        one = [line for line in text.splitlines() if "step_one_kernel" in line]
        assert len(text.splitlines()) == (3 if one else 5)
        attention = int(one[0].split()[2]) - B * (-(-H * K // 256) + H * -(-V // 64)) if one else 0
        assert attention % (B * HQ) == 0
        out.append(attention // (B * HQ) if one else None)
    return out


@pytest.mark.parametrize("geometry,B,tokens,splits", [
    ("mamba", 1, 2473, 10), ("mamba", 8, 1461, 4), ("mamba", 16, 537, 1), ("mamba", 16, 1589, 3), ("mamba", 16, 3113, 5), ("mamba", 32, 5357, 5),
    ("mamba", 64, 973, 2), ("gdn_340M", 1, 473, 2), ("gdn_340M", 8, 5229, 5), ("gdn_340M", 16, 2793, 4), ("gdn_340M", 24, 5421, 5),
    ("gdn_340M", 28, 600, 1), ("gdn_340M", 29, 600, None), ("gdn_340M", 64, 2857, None), ("gdn_760M", 1, 1333, 6), ("gdn_760M", 4, 2665, 4),
    ("gdn_760M", 8, 537, 1), ("gdn_760M", 8, 5101, 5), ("gdn_760M", 12, 9525, 5), ("gdn_760M", 13, 9525, None), ("wide", 4, 3697, 13),
    ("wide", 12, 7393, 5), ("wide", 25, 1245, 2), ("wide", 26, 1245, None)])
def test_splits_of_the_one_token_step(fake_hip, geometry, B, tokens, splits):  # noqa: F811
    assert _splits(fake_hip, [(geometry, B, tokens)]) == [splits]
