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


def _step(geometry, B, T, tokens, D):
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
    return s


@pytest.mark.parametrize("geometry,B,T,tokens,D,one", [
    ("gdn_340M", 1, 1, 473, 1024, True), ("gdn_340M", 4, 1, 300, 1024, True), ("gdn_340M", 4, 1, 2000, 1024, False), ("gdn_340M", 8, 1, 300, 1024, False),
    ("gdn_340M", 1, 2, 473, 1024, False), ("gdn_760M", 1, 1, 473, 1536, True), ("gdn_760M", 2, 1, 100, 1536, True), ("gdn_760M", 3, 1, 100, 1536, False),
    ("mamba", 1, 1, 473, 1024, True), ("mamba", 6, 1, 100, 1024, False), ("mamba", 17, 1, 100, 1024, False), ("wide", 1, 1, 64, 4096, False)])
def test_which_steps_are_one_launch(fake_hip, geometry, B, T, tokens, D, one):  # noqa: F811
    from neuralattentionsearchlinear_amd import _capi
    s = _step(geometry, B, T, tokens, D)
    H, K, V = s.H, s.K, s.V
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


TURNS = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
lib.natsl_layer_step_workspace_bytes.restype = lib.natsl_layer_step_sync_bytes.restype = ctypes.c_size_t
P, Z = ctypes.c_void_p, ctypes.c_size_t
s = ctypes.create_string_buffer(bytes.fromhex(sys.argv[3]))
for stream, done, capturing, no_memory, device in json.loads(sys.argv[4]):
    fake.fake_reset(device)
    ctypes.c_int.in_dll(fake, "fake_capturing").value, ctypes.c_int.in_dll(fake, "fake_no_host_memory").value = capturing, no_memory
    if done is not None:
        ctypes.c_ulonglong.in_dll(fake, "fake_host_words").value = done
    shared = lib.natsl_layer_step_sync_bytes(s)
    rc = lib.natsl_layer_step_sync_fwd(s, P(1 << 20), Z(lib.natsl_layer_step_workspace_bytes(s)), P(1 << 21), Z(shared), ctypes.c_uint64(1000), P(stream))
    out.append((rc, len(fake.fake_launches().decode().splitlines())))
lib.natsl_layer_step_gave_up.restype = ctypes.c_ulonglong
before = lib.natsl_layer_step_gave_up(0)
(ctypes.c_ulonglong * 8).in_dll(fake, "fake_host_words")[1] = 4
out.append([before, *(lib.natsl_layer_step_gave_up(d) for d in (0, 1, -1, 64))])
print(json.dumps(out))
"""


def test_one_launch_at_a_time_waits_to_start(fake_hip):  # noqa: F811
    """Steps whose parts wait for each other are under way one at a time or one behind another on a stream: those of a second stream are three launches until
    the last of the first has started all of its parts; so are captured ones, and all of them where the host has no word to look at."""
    from neuralattentionsearchlinear_amd import _capi
    A, B, PER_THREAD = 0x10, 0x20, 2
    calls = [  # (stream, what the GPU has written before the call, whether the stream is captured, no pinned memory, device) -> launches
        ((A, None, 0, 1, 0), 3), ((A, None, 0, 0, 0), 1), ((A, None, 0, 0, 0), 1), ((B, None, 0, 0, 0), 3), ((B, 1, 0, 0, 0), 3), ((A, None, 1, 0, 0), 3),
        ((A, None, 0, 0, 0), 1), ((B, 2, 0, 0, 0), 3), ((B, 3, 0, 0, 0), 1), ((A, None, 0, 0, 0), 3), ((B, None, 0, 0, 0), 1), ((A, 5, 0, 0, 0), 1),
        ((PER_THREAD, 5, 0, 0, 0), 3), ((PER_THREAD, 6, 0, 0, 0), 1), ((PER_THREAD, None, 0, 0, 0), 3), ((PER_THREAD, 7, 0, 0, 0), 1)]
    r = subprocess.run([sys.executable, "-c", TURNS, fake_hip, _capi.LIB_PATH, bytes(_step("gdn_340M", 1, 1, 473, 1024)).hex(),
                        json.dumps([c for c, _ in calls])], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert json.loads(r.stdout) == [[0, n] for _, n in calls] + [[0, 4, 0, 0, 0]]       # (and what a launch that gives up leaves there)


@pytest.mark.parametrize("cus,one", [(256, True), (128, False), (32, False)])
def test_waiting_parts_are_half_of_the_chip_that_is_there(fake_hip, cus, one):  # noqa: F811
    """(a part of the card that is a device of its own has fewer compute units)"""
    from neuralattentionsearchlinear_amd import _capi
    child = CHILD.replace("lib, out =", "ctypes.c_int.in_dll(fake, 'fake_cus').value = %d\nlib, out =" % cus)
    r = subprocess.run([sys.executable, "-c", child, fake_hip, _capi.LIB_PATH, json.dumps([bytes(_step("gdn_760M", 1, 1, 473, 1536)).hex()])],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    shared, *calls = json.loads(r.stdout)[0]
    assert calls[0][0] == 0 and ("step_all_kernel" in calls[0][1]) == one
