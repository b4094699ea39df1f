"""CPU-only: that the sizes at which the GPU tests compare two kernels take the kernel that they are about, seen from what a HIP runtime that launches
nothing (tests/fake_hip.c; 256 compute units) is asked to launch: the softmax tiles' launch with the linear prep, lists made from the blocks' types,
the weight gradients' tile widths."""
import ctypes
import json
import os
import subprocess
import sys

import pytest

from tests.test_gpu_softmax_prep import CASES as PREP
from tests.test_gpu_softmax_types import CASES as TYPES
from tests.test_gpu_wgrad_tiles import CASES as WGRAD
from tests.test_stream_order import ALL, fake_hip  # noqa: F401

MIXED = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
for call in json.loads(sys.argv[3]):
    fake.fake_reset(0)
    rc = lib.natsl_mixed_fwd(ctypes.create_string_buffer(bytes.fromhex(call)), %d, ctypes.c_void_p(0x10), ctypes.c_void_p(0x10))
    out.append([rc, [line.split()[0] for line in fake.fake_launches().decode().splitlines()]])
print(json.dumps(out))
""" % ALL
WEIGHTS = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
lib, out = ctypes.CDLL(sys.argv[2]), []
lib.natsl_wgrad_workspace_bytes.restype = ctypes.c_size_t
class Seg(ctypes.Structure):
    _fields_ = [("dy", ctypes.c_void_p), ("out", ctypes.c_void_p), ("n", ctypes.c_int32), ("ld", ctypes.c_int32)]
N, P = ctypes.c_int64, ctypes.c_void_p
for T, D, widths in json.loads(sys.argv[3]):
    segs = (Seg * len(widths))()
    for s, n in zip(segs, widths):
        s.dy = s.out = 1 << 20
        s.n = s.ld = n
    size = lib.natsl_wgrad_workspace_bytes(segs, len(widths), N(T), D)
    fake.fake_reset(0)
    rc = lib.natsl_wgrad(segs, len(widths), P(1 << 20), N(T), D, D, P(1 << 20), ctypes.c_size_t(size), P(0x10))
    other = [lib.natsl_narrow_wgrad_pays(N(T), D, n, 0, len(widths) == 1) for n in widths]
    out.append([rc, size, other, [line.split()[0] for line in fake.fake_launches().decode().splitlines()]])
print(json.dumps(out))
"""


def _run(child, fake, cases):
    from neuralattentionsearchlinear_amd import _build, _capi
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    r = subprocess.run([sys.executable, "-c", child, fake, _capi.LIB_PATH, json.dumps(cases)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout)


def _mixed(kind, B, T, H, KA, VA, K, V, block, HQ=None, HN=None, tables=False, states=False):
    from neuralattentionsearchlinear_amd import _capi
    from neuralattentionsearchlinear_amd._mixed_common import _POINTERS, _Mixed
    m = _Mixed()
    for name in _POINTERS:
        setattr(m, name, 1 << 20)
    m.h0 = m.ht = m.h_block_start = m.g_block_sum = None
    if not states:
        m.chunk_states = m.chunk_v_new = None
    if kind != 'gdn':
        m.beta = None
    TN, HQ = -(-T // block), HQ or H
    size = dict(is_delta=int(kind == 'gdn'), B=B, T=T, H=H, HN=HN or H, K=K, V=V, TN=TN, block=block, flags=7, T_attn=T, TN_attn=TN, HQ=HQ, HKV=HQ, KA=KA,
                VA=VA, same_block_visible=1, types_dtype=_capi.BF16, scale_attn=0.1, scale_linear=0.1, workspace_bytes=1 << 40, private_tables=int(not tables))
    for name, value in size.items():
        setattr(m, name, value)
    return bytes(ctypes.string_at(ctypes.addressof(m), ctypes.sizeof(m))).hex()


@pytest.mark.parametrize("gradients", [False, True])
def test_softmax_tiles_and_prep_are_one_launch(fake_hip, gradients):  # noqa: F811
    # (gradients: the routing tables and the chunk states are kept.)  Many linear heads on few attention heads: two launches
    calls = [_mixed(*c[:-1], tables=gradients, states=gradients) for c in PREP] + [_mixed('gdn', 1, 256, 40, 64, 64, 64, 64, 64, HQ=8, HN=8)]
    for case, (rc, names) in zip(PREP + [(False,)], _run(MIXED, fake_hip, calls)):
        assert rc == 0
        joint = [n for n in names if "softmax_prep_kernel" in n]
        own = [n for n in names if "linear_prep_kernel" in n or "mamba_scale_kernel" in n or "softmax_sparse_fwd_kernel" in n]
        assert (len(joint), len(own)) == ((1, 0) if case[-1] else (0, 2)), (case, names)


@pytest.mark.parametrize("tables", [False, True])
def test_no_routing_launch_where_tiles_read_the_types(fake_hip, tables):  # noqa: F811
    calls = [_mixed('gdn', B, blocks * block - (17 if blocks > 1 else 0), H, 64, 64, 64, 64, block, HN=HN, tables=tables) for blocks, B, H, HN, block, _, _ in TYPES]
    for (blocks, *_), (rc, names) in zip(TYPES, _run(MIXED, fake_hip, calls)):
        assert rc == 0 and any("route_kernel" in n for n in names) == (tables or blocks > 256), (blocks, names)
        assert not any("softmax_stream_kernel" in n for n in names)


def test_weight_gradient_tiles(fake_hip):  # noqa: F811
    columns = set()
    for (T, D, widths, width, slices), (rc, size, other, names) in zip(WGRAD, _run(WEIGHTS, fake_hip, [c[:3] for c in WGRAD])):
        if width is None:
            assert all(other)
            continue
        nb, tiles = width // 64, -(-D // width)
        assert rc == 0 and not any(other) and [f"wgrad_kernelILi{nb}E" in names[0], f"wgrad_reduce_kernelILi{nb}E" in names[1]] == [True, True], (T, D, widths, names)
        assert size == slices * tiles * sum(-(-n // 32) for n in widths) * 32 * width * 4, (T, D, widths)
        columns.add((width, slices > 1, D % width > 0))
    assert {(w, True, last) for w in (192, 256) for last in (False, True)} <= columns      # both widths: several slices, whole and part last tiles
