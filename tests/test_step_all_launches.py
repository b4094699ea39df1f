"""CPU-only: which one-token steps are one launch when the caller keeps memory for them, seen from what a HIP runtime that launches nothing
(tests/fake_hip.c) is asked to launch.  Whatever waits in such a launch is at most half of what the chip holds."""
import json
import subprocess
import sys

import pytest

from tests.test_step_splits import GEOMETRY
from tests.test_stream_order import fake_hip  # noqa: F401

CHILD = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
lib.natsl_layer_step_workspace_bytes.restype = lib.natsl_layer_step_sync_bytes.restype = ctypes.c_size_t
P, Z = ctypes.c_void_p, ctypes.c_size_t
for step in json.loads(sys.argv[3]):
    s = ctypes.create_string_buffer(bytes.fromhex(step))
    ws, shared = lib.natsl_layer_step_workspace_bytes(s), lib.natsl_layer_step_sync_bytes(s)
    row = [shared]
    for n in (shared, shared - 1) if shared else (0,):
        fake.fake_reset(0)
        rc = lib.natsl_layer_step_sync_fwd(s, P(1 << 20), Z(ws), P(1 << 21 if shared else 0), Z(n), ctypes.c_uint64(1000), P(0x10))
        row.append([rc, fake.fake_launches().decode()])
    out.append(row)
print(json.dumps(out))
"""


@pytest.mark.parametrize("geometry,B,T,tokens,D,one", [
    ("gdn_340M", 1, 1, 473, 1024, True), ("gdn_340M", 4, 1, 300, 1024, True), ("gdn_340M", 4, 1, 2000, 1024, False), ("gdn_340M", 8, 1, 300, 1024, False),
    ("gdn_340M", 1, 2, 473, 1024, False), ("gdn_760M", 1, 1, 473, 1536, True), ("gdn_760M", 2, 1, 100, 1536, True), ("gdn_760M", 3, 1, 100, 1536, False),
    ("mamba", 1, 1, 473, 1024, True), ("mamba", 6, 1, 100, 1024, False), ("mamba", 17, 1, 100, 1024, False), ("wide", 1, 1, 64, 4096, False)])
def test_which_steps_are_one_launch(fake_hip, geometry, B, T, tokens, D, one):  # noqa: F811
    from neuralattentionsearchlinear_amd import _build, _capi
    from neuralattentionsearchlinear_amd._layer_step import _TENSORS, _WEIGHTS, LayerStep
    import os
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    s = LayerStep()
    for n in _WEIGHTS + _TENSORS:
        setattr(s, n, 1 << 20)
    H, K, V, HQ, s.is_delta = GEOMETRY[geometry]
    s.H, s.K, s.V, s.HQ, s.B, s.T, s.D, s.HN, s.block, s.conv_width = H, K, V, HQ, B, T, D, 1, 64, 4
    s.n_kept, s.n_in, s.cache_tokens = (tokens - T) // 64, min((tokens - T) % 64, 64 - T), -(-tokens // 64) * 64 + 64
    s.types_dtype = s.norm_dtype = s.gate_dtype = s.out_norm_dtype = _capi.BF16
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, _capi.LIB_PATH, json.dumps([bytes(s).hex()])], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    ((shared, (rc, text), *short),) = json.loads(r.stdout)
    assert rc == 0
    lines = text.splitlines()
    assert ([line for line in lines if "step_all_kernel" in line] == lines and len(lines) == 1) == one and len(lines) == (1 if one else 5 if T > 1 else 3)
    if short:                                              # (less memory than asked for: refused, nothing launched)
        assert short[0][0] != 0 and short[0][1] == ""
    if one:
        tiles = sum(-(-n // 16) for n in (H * K, H * K, H * V, H * V, H) + ((H,) if s.is_delta else ()))
        waiting = int(lines[0].split()[2]) - tiles
        assert shared > 0 and 0 < waiting <= 280 and waiting <= 128 * (2 if K == 192 or (K, V) == (128, 128) else 3)
