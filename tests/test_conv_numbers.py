"""CPU-only: which of a segment's numbers (natsl_conv_seg.scale) the convolutions' kernels are handed, seen from what a HIP runtime that
launches nothing (tests/fake_hip.c) is asked to launch.  They are rows of D / (8 norm_lanes) for what follows the convolution."""
import ctypes
import json
import os
import subprocess
import sys

import pytest

from tests.test_stream_order import fake_hip  # noqa: F401

CHILD = """
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_segments.restype = ctypes.c_void_p
lib = ctypes.CDLL(sys.argv[2])
lib.natsl_conv_norm_bwd_workspace_bytes.restype = ctypes.c_size_t
one, p, i = ctypes.create_string_buffer(bytes.fromhex(sys.argv[3])), ctypes.c_void_p(1 << 20), ctypes.c_int
fake.fake_reset(0)
if sys.argv[4] == "1":
    n = lib.natsl_conv_norm_bwd_workspace_bytes(one, i(1), i(2), i(100), i(3))
    rc = lib.natsl_conv_norm_bwd(one, i(1), i(2), i(100), i(3), i(1), i(1), p, ctypes.c_size_t(n), ctypes.c_void_p(0x10))
else:
    rc = lib.natsl_conv_norm_fwd(one, i(1), i(2), i(100), i(3), i(1), i(1), ctypes.c_void_p(0x10))
print(json.dumps([rc, ctypes.string_at(fake.fake_segments(), len(one) - 1).hex()]))
"""
X, SCALE, DSCALE = 1 << 20, 1 << 21, 1 << 22


@pytest.mark.parametrize("bwd,dscale,follows,lanes,gets", [
    (0, False, True, 8, (SCALE, None, 8)), (0, False, False, 8, (None, None, 1)), (0, False, False, 7, (None, None, 1)),
    (1, True, True, 8, (SCALE, DSCALE, 8)), (1, False, True, 8, (SCALE, None, 8)), (1, False, False, 8, (None, None, 1)),
    (1, True, False, 8, (SCALE, DSCALE, 8)), (1, True, False, 7, None)])
def test_numbers_are_read_where_something_is_multiplied_by_them(fake_hip, bwd, dscale, follows, lanes, gets):
    """gets: (scale, dscale, norm_lanes) of the kernel's segment; None: refused.  Without a tensor that follows the numbers norm_lanes is one,
    which makes their rows D / 8 wide, and the numbers must not be read; the gradient of unused ones is zero, for which norm_lanes has to be right."""
    from neuralattentionsearchlinear_amd import _build, _capi
    from neuralattentionsearchlinear_amd._front import _ConvSeg
    if not os.path.exists(_capi.LIB_PATH):
        _build.build()
    s = _ConvSeg()
    s.x = s.weight = X
    if bwd:
        s.dy_a = s.dx = s.dweight = X
        s.dy_norm = X if follows else None
    else:
        s.y, s.y_norm = X, X if follows else None
    s.D, s.norm_lanes, s.scale, s.dscale = 128, lanes, SCALE, DSCALE if dscale else None
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, _capi.LIB_PATH, bytes(s).hex(), str(bwd)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    rc, given = json.loads(r.stdout)
    assert (rc == 0) == (gets is not None)
    if gets is not None:
        got = _ConvSeg.from_buffer_copy(bytes.fromhex(given)[:ctypes.sizeof(_ConvSeg)])
        assert (got.scale, got.dscale, got.norm_lanes) == gets
