"""CPU-only: what the layers' native calls (csrc/host/layer_core.cpp) refuse before they look at a tensor."""
import json
import os
import subprocess
import sys

CHILD = """
import json, torch
from neuralattentionsearchlinear_amd import _capi
core = _capi.step_core()
layer = core.make_layer(_capi.lib()._handle, _capi.check, (0,) * 21, (1.,) * 4)
x, out = torch.zeros(1, 64, 32), {}
calls = dict(train=lambda n: core.layer_train(layer, x, [None] * n, 0, 0, False, None, False),
             wants=lambda n: core.layer_train(layer, x, [None] * 21, 0, 0, False, (True,) * n, False),
             front=lambda n: core.layer_front(layer, x, [None] * n, 0),
             rest=lambda n: core.layer_rest(layer, x, [None] * n, [None] * 8, 0, 0, False, False),
             backward=lambda n: core.layer_backward(layer, x, [None] * n, (True,) * 22, 0, 0, False, False))
for name, call in calls.items():
    for n in (0, 20, 23):
        try:
            call(n)
            out[f"{name} {n}"] = "taken"
        except Exception as e:
            out[f"{name} {n}"] = type(e).__name__
        print(json.dumps(out), flush=True)
"""


def test_another_number_of_tensors_is_refused():
    """The calls address the weights by number: fewer would be read past their end."""
    from neuralattentionsearchlinear_amd import _build, _capi
    if not (os.path.exists(_capi.LIB_PATH) and os.path.exists(_capi.STEP_CORE_PATH)):
        _build.build()
    r = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    got = json.loads(r.stdout.splitlines()[-1]) if r.stdout else {}
    assert r.returncode == 0 and len(got) == 15 and set(got.values()) == {"ValueError"}, (got, r.stderr[-300:])
