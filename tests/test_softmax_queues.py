"""CPU-only: whose memory the persistent softmax kernel's work queues are, seen from what a HIP runtime that launches nothing
(tests/fake_hip.c) is asked to launch; and the order in which that kernel deals tiles out where it has no queues."""
import json
import os
import re
import subprocess
import sys

import pytest

from tests.test_stream_order import ALL, fake_hip  # noqa: F401

CHILD = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
lib.natsl_linear_workspace_bytes.restype = lib.natsl_mixed_workspace_bytes.restype = ctypes.c_size_t
lib.natsl_linear_workspace_bytes.argtypes = lib.natsl_mixed_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int]
p, f = ctypes.c_void_p(1 << 20), ctypes.c_float(0.1)
for kind, arg in json.loads(sys.argv[3]):
    fake.fake_reset(0)
    if kind == "mixed":
        rc = lib.natsl_mixed_fwd(ctypes.create_string_buffer(bytes.fromhex(arg)), 31, ctypes.c_void_p(0x10), ctypes.c_void_p(0x20))
    else:
        B, T, H, n_seqs, tiles, TN = arg
        rc = lib.natsl_softmax_sparse_fwd(p, p, p, p, p, p, 1, p, p, B, T, H, H, H, 64, 64, TN, 64, f, 1, 1, p if n_seqs else None, n_seqs, tiles,
                                          ctypes.c_void_p(0x10))
    out.append([rc, fake.fake_launches().decode()])
print(json.dumps(out))
"""
WORKSPACE, SLOTS = 1 << 24, 4096          # (the fake's address of the library's slots)


def _launches(fake_hip, calls):
    from neuralattentionsearchlinear_amd import _build, _capi
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, _capi.LIB_PATH, json.dumps(calls)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = []
    for rc, text in json.loads(r.stdout):
        assert rc == 0
        rows = [line.split() for line in text.splitlines()]
        out.append([(re.search("stream_queue_clear|softmax_stream|softmax_sparse", n)[0], int(s, 16), int(q, 16)) for n, s, _, q in rows if "softmax" in n or "queue" in n])
    return out


def _mixed(B, T, H, n_seqs, workspace_bytes):
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._mixed_common import _POINTERS, _Mixed
    m = _Mixed()
    for name in _POINTERS:
        setattr(m, name, 1 << 20)
    m.workspace, m.workspace_bytes = WORKSPACE, workspace_bytes
    m.h0 = m.ht = m.h_block_start = m.g_block_sum = m.chunk_states = m.chunk_v_new = None
    TN = -(-T // 64) + n_seqs
    for name, v in dict(is_delta=1, B=B, T=T, H=H, HN=H, K=64, V=64, TN=TN if n_seqs else -(-T // 64), block=64, flags=7, T_attn=T, HQ=H, HKV=H, KA=64,
                        VA=64, same_block_visible=1, types_dtype=_capi.BF16, scale_attn=0.1, scale_linear=0.1).items():
        setattr(m, name, v)
    m.TN_attn = m.TN
    if n_seqs:
        m.seqs, m.n_seqs, m.total_chunks, m.total_qtiles = 1 << 20, n_seqs, -(-T // 64) + n_seqs, -(-T // 256) + n_seqs
    return ["mixed", bytes(m).hex()]


# (batch, tokens, heads, packed sequences): all of enough tiles for the persistent kernel
FORMS = [(16, 4096, 16, 0), (16, 4000, 16, 0), (16, 4095, 16, 0), (1, 65536, 16, 4), (1, 65521, 16, 3)]


@pytest.mark.parametrize("B,T,H,n_seqs", FORMS)
def test_an_operators_queues_are_in_its_own_workspace(fake_hip, B, T, H, n_seqs):  # noqa: F811
    chunks = -(-T // 64) + n_seqs if n_seqs else B * -(-T // 64)
    from neuralattentionsearchlinear_amd import _capi
    linear, need = _capi.lib().natsl_linear_workspace_bytes(chunks, H), _capi.lib().natsl_mixed_workspace_bytes(chunks, H)
    (clear, kernel), short = _launches(fake_hip, [_mixed(B, T, H, n_seqs, need), _mixed(B, T, H, n_seqs, need - 1)])
    assert clear == ("stream_queue_clear", 0x20, WORKSPACE + linear) and kernel == ("softmax_stream", 0x20, WORKSPACE + linear)
    assert need >= linear + 8 * 4                                       # a counter per XCD
    # a workspace without that room: the call runs as the softmax entry by itself
    if T % 256 or n_seqs:
        assert short == [("softmax_stream", 0x20, 0)]
    else:
        assert [n for n, _, _ in short] == ["stream_queue_clear", "softmax_stream"] and short[0][2] == short[1][2] and short[0][2] < WORKSPACE


@pytest.mark.parametrize("T,per_cu", [(2048, 6), (4096, 6), (16384, 6), (8191, 4), (32769, 6), (3000, 8), (4160, 8), (512, 8)])
def test_operators_take_the_persistent_kernel_from_their_own_line_on(fake_hip, T, per_cu):  # noqa: F811
    """Six tiles' worth of queries per CU on long whole or cut lengths (four where the last tile is more than half full), eight on others
    (256 CUs), whatever the softmax entry by itself is held to by its tests."""
    H = 8
    from neuralattentionsearchlinear_amd import _capi
    calls, first = [], -(-per_cu * 256 * 256 // (H * T))                # batches that reach the line, and the largest that does not
    for B in (first - 1, first):
        need = _capi.lib().natsl_mixed_workspace_bytes(B * -(-T // 64), H)
        calls.append(_mixed(B, T, H, 0, need))
    below, at = _launches(fake_hip, calls)
    assert [r[0] for r in below] == ["softmax_sparse"] and [r[0] for r in at] == ["stream_queue_clear", "softmax_stream"]


@pytest.mark.parametrize("B,T,H,kernel", [
    (1, 8192, 18, "softmax_stream"), (1, 12392, 18, "softmax_stream"), (1, 16385, 12, "softmax_stream"), (4, 4096, 9, "softmax_stream"),
    (1, 8192, 24, "softmax_sparse"), (1, 12392, 24, "softmax_sparse"), (5, 4096, 9, "softmax_sparse"), (1, 4096, 18, "softmax_sparse")])
def test_operators_with_pairs_that_leave_xcds_idle_take_it_earlier(fake_hip, B, T, H, kernel):  # noqa: F811
    """(sequence, head) pairs that do not divide over the eight XCDs: from two tiles per CU on whole tiles, three on cut lengths."""
    from neuralattentionsearchlinear_amd import _capi
    (rows,) = _launches(fake_hip, [_mixed(B, T, H, 0, _capi.lib().natsl_mixed_workspace_bytes(B * -(-T // 64), H))])
    assert rows[-1][0] == kernel


def test_only_whole_tile_launches_of_the_softmax_entry_take_slots(fake_hip):  # noqa: F811
    """Packed sequences and lengths that are no multiple of a tile share no memory with any other launch, whatever streams and graphs
    they are on."""
    calls = []
    for B, T, H, n in FORMS:
        calls.append(["softmax", (B, T, H, n, -(-T // 256) + n, -(-T // 64) + n if n else -(-T // 64))])
    for (_, T, _, n), rows in zip(FORMS, _launches(fake_hip, calls)):
        if T % 256 or n:
            assert rows == [("softmax_stream", 0x10, 0)]
        else:
            assert [r[0] for r in rows] == ["stream_queue_clear", "softmax_stream"] and SLOTS <= rows[0][2] == rows[1][2] < SLOTS + 64 * 64


@pytest.mark.parametrize("workgroups,pairs,tiles", [(256, 128, 32), (256, 8, 256), (256, 9, 240), (250, 704, 4), (256, 1, 3), (3, 5, 7), (1, 2, 2)])
def test_dealt_tiles_are_each_taken_once(workgroups, pairs, tiles):
    """The kernel's arithmetic (next_dealt and what resolve_ticket makes of it): every tile of every pair once, no workgroup asked for
    more than it has, and with tiles that cost what causal ones do no workgroup far behind the others."""
    seen, most = {}, 0
    for w in range(workgroups):
        rounds = load = 0
        while True:
            t = rounds * workgroups + (workgroups - 1 - w if rounds & 1 else w)
            rounds += 1
            if t >= pairs * tiles:
                break
            key = (t % pairs, tiles - 1 - t // pairs)
            assert key not in seen and 0 <= key[1] < tiles
            seen[key] = w
            load += key[1] + 1
        most = max(most, load)
    assert len(seen) == pairs * tiles
    mean = pairs * tiles * (tiles + 1) / 2 / workgroups
    assert most <= mean + tiles                             # (list scheduling of jobs of at most `tiles`)
