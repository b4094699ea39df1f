"""CPU-only: how the mixed operator's native call orders its two streams, run against a HIP runtime that launches nothing
(tests/fake_hip.c) in a process of its own."""
import json
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CONVERT, ROUTE, SOFTMAX, LINEAR, JOIN = 1, 2, 4, 8, 16
ALL = CONVERT | ROUTE | SOFTMAX | LINEAR | JOIN
CHILD = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_notes.restype = ctypes.c_char_p
lib = ctypes.CDLL(sys.argv[2])
call, out = ctypes.create_string_buffer(bytes.fromhex(sys.argv[3])), []
for phases, stream, side, current in json.loads(sys.argv[4]):
    fake.fake_reset(current)
    rc = lib.natsl_mixed_fwd(call, phases, ctypes.c_void_p(stream), ctypes.c_void_p(side))
    out.append([rc, fake.fake_notes().decode().strip(), fake.fake_current()])
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", os.path.join(HERE, "fake_hip.c"), "-o", lib], check=True)
    return lib


def _run(fake_hip, calls, **fields):
    """[(return code, what was launched and ordered, the current device afterwards)] of calls (phases, stream, side, current device)."""
    from neuralattentionsearchlinear_amd import _build, _capi
    from neuralattentionsearchlinear_amd._mixed_common import _POINTERS, _Mixed
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    m = _Mixed()
    for name in _POINTERS:
        setattr(m, name, 1 << 20)
    m.h0 = m.ht = m.h_block_start = m.g_block_sum = m.chunk_states = m.chunk_v_new = None
    size = dict(is_delta=1, B=1, T=256, H=2, HN=2, K=64, V=64, TN=4, block=64, flags=7, T_attn=256, TN_attn=4, HQ=2, HKV=2, KA=64, VA=64,
                same_block_visible=1, types_dtype=_capi.BF16, scale_attn=0.1, scale_linear=0.1, workspace_bytes=1 << 30)
    for name, value in dict(size, **fields).items():
        setattr(m, name, value)
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, _capi.LIB_PATH, bytes(m).hex(), json.dumps(calls)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout)


def test_streams_are_ordered_on_their_own_device(fake_hip):
    """The caller's current device may be another than the streams': the call enters theirs and leaves the caller's as it was."""
    calls = [(ALL, 0x2001, 0x2002, 0), (ALL, 0x1001, 0x1002, 1), (ALL, 0, 0x3002, 0), (ALL, 0x2001, 0x2001, 0)]
    for (_, stream, side, current), (rc, notes, after) in zip(calls, _run(fake_hip, calls)):
        device = (side or stream) >> 12
        assert rc == 0 and after == current
        launched = re.findall(r"launch (\w+):(\d+)", notes)
        assert {int(s, 16) for s, _ in launched} == {stream, side} and {int(d) for _, d in launched} == {device}, notes
        if side != stream:
            assert notes.startswith(f"record {stream:x} wait {side:x} ") and notes.endswith(f"record {side:x} wait {stream:x}"), notes
    assert _run(fake_hip, [(ALL, 0x1001, 0x2001, 0)])[0][0] == -1                    # streams of two devices


@pytest.mark.parametrize("fields", [dict(K=96), dict(VA=96), dict(HQ=3), dict(workspace_bytes=16)])
def test_an_error_leaves_nothing_unwaited_on_the_side_stream(fake_hip, fields):
    """What the side stream got before a branch refused its arguments is waited for by the caller's stream all the same: the caller
    frees what it works on."""
    s, side = 0x1001, 0x1002
    steps = [(ALL, s, side, 1), (CONVERT | ROUTE, s, side, 1), (SOFTMAX | LINEAR, s, side, 1), (CONVERT | ROUTE | SOFTMAX, s, side, 1), (LINEAR, s, side, 1)]
    failed = 0
    for rc, notes, _ in _run(fake_hip, steps, **fields):
        if rc != 0:
            failed += 1
            assert notes.endswith(f"record {side:x} wait {s:x}"), notes
    assert failed >= 2
    # on one stream there is nothing to wait for
    rc, notes, _ = _run(fake_hip, [(ALL, s, s, 1)], **fields)[0]
    assert rc != 0 and "wait" not in notes


def test_chunk_states_release_the_other_stream_before_the_scan(fake_hip):
    """The linear branch's states for a backward: the other stream waits for what is in front of the scan and not for the scan; without one
    nothing is ordered, and what is refused has ordered nothing."""
    child = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_notes.restype = ctypes.c_char_p
f = ctypes.CDLL(sys.argv[2]).natsl_linear_chunk_states
p, n, i, out = ctypes.c_void_p(1 << 20), ctypes.c_void_p(None), ctypes.c_int, []
for kind, K, side in ((1, 64, 0x1002), (0, 128, 0x1002), (1, 192, 0), (1, 96, 0x1002)):
    fake.fake_reset(0)
    rc = f(i(kind), p, p, p, p, p, n, n, p, p, p, i(1), i(1), i(256), i(2), i(2), i(K), i(64), i(4), i(64), ctypes.c_float(0.1), i(7), p,
           ctypes.c_size_t(1 << 30), i(1), n, i(0), i(4), ctypes.c_void_p(0x1001), ctypes.c_void_p(side))
    out.append([rc, fake.fake_notes().decode().strip(), fake.fake_current()])
print(json.dumps(out))
"""
    from neuralattentionsearchlinear_amd import _build, _capi
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    assert _capi.BF16 == 1
    r = subprocess.run([sys.executable, "-c", child, fake_hip, _capi.LIB_PATH], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    beside, ordered = "launch 1001:1 record 1001 wait 1002 launch 1001:1", "launch 1001:1 launch 1001:1"
    got = json.loads(r.stdout)
    assert [g[1] for g in got] == [beside, beside, ordered, ""] and [g[0] == 0 for g in got] == [True] * 3 + [False] and {g[2] for g in got} == {0}


@pytest.mark.parametrize("kind,B,H,K,V,alone,beside", [(1, 4, 8, 128, 128, 256, 128), (1, 1, 8, 192, 384, 192, 96), (0, 2, 32, 128, 64, 256, 128), (1, 1, 2, 128, 128, 64, 64)])
def test_a_scan_next_to_other_work_leaves_it_compute_units(fake_hip, kind, B, H, K, V, alone, beside):
    """Workgroups of the scan, by itself and with the other stream's work behind the kernel in front of it (256 compute units)."""
    child = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
f = ctypes.CDLL(sys.argv[2]).natsl_linear_chunk_states
kind, B, H, K, V = json.loads(sys.argv[3])
p, n, i, out = ctypes.c_void_p(1 << 20), ctypes.c_void_p(None), ctypes.c_int, []
for side in (0, 0x1002):
    fake.fake_reset(1)
    rc = f(i(kind), p, p, p, p, p, n, n, p, p, p, i(1), i(B), i(4096), i(H), i(H), i(K), i(V), i(64), i(64), ctypes.c_float(0.1), i(7), p,
           ctypes.c_size_t(1 << 40), i(1), n, i(0), i(B * 64), ctypes.c_void_p(0x1001), ctypes.c_void_p(side))
    scan = [line.split() for line in fake.fake_launches().decode().splitlines() if "linear_scan_kernel" in line]
    out.append([rc, len(scan), int(scan[0][2])])
print(json.dumps(out))
"""
    from neuralattentionsearchlinear_amd import _build, _capi
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    r = subprocess.run([sys.executable, "-c", child, fake_hip, _capi.LIB_PATH, json.dumps([kind, B, H, K, V])], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert json.loads(r.stdout) == [[0, 1, alone], [0, 1, beside]]
