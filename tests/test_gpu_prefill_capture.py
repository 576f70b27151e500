"""A prefill layer whose formats come from both families, captured where the
scratch holds the bf16 path's regions but not the f16 path's: it is taken on
the bf16 kernels, and the scratch does not grow. In a process of its own, so
that the scratch has its smallest size, 4 MiB."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = r"""
import ctypes, sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from sepia_amd import hip
from test_gpu_parity import make_layer, run_prefill

T, H = int(sys.argv[2]), 512
dev = hip.Device()
L, stream = dev.L, ctypes.c_void_p(dev.stream())
R = ctypes.CDLL("libamdhip64.so")
rng = np.random.default_rng(T)
X = rng.standard_normal((T, H)).astype(np.float32)
desc, spec, bufs = make_layer(dev, rng, hidden=H, inter=H, n_routed=4, n_shared=0, tg=12, tu=12, td=13, ts=12, topk=2)
run_prefill(dev, desc, X[:2])   # the weights are on the device, the scratch is there
xs, ys = dev.shared_from(X), dev.alloc(X.nbytes)
xp, yp = dev.alloc(X.nbytes, private=True), dev.alloc(X.nbytes, private=True)
dev.run(L.sepia_gpu_copy, xs, 0, xp, 0, X.size)
size = L.sepia_hip_scratch_bytes()
graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
dev.begin()
assert R.hipStreamBeginCapture(stream, 1) == 0
ok = L.sepia_gpu_moe_prefill(ctypes.byref(desc), T, xp, yp, None)
assert R.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
dev.end()
assert ok == 1 and L.sepia_hip_scratch_bytes() == size
assert R.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
got = []
for i in range(3):
    assert R.hipGraphLaunch(exe, stream) == 0
    dev.run(L.sepia_gpu_copy, yp, 0, ys, 0, X.size)
    got.append(dev.download(ys, X.size).copy())
R.hipGraphExecDestroy(exe)
want, _, _ = run_prefill(dev, desc, X)
grown = L.sepia_hip_scratch_bytes() > size
# a product of the bf16 kernels is within 3 * 2^-17 = 2.3e-5 (both factors' splits and the dropped lo * lo); errors of
# random sign average out in a contraction, and two contractions follow each other
err = max(float(np.abs(y - want.ravel()).max()) for y in got) / float(np.abs(want).max())
print("grown %d err %.2e" % (grown, err), flush=True)
assert err <= 4e-5
assert grown == (sys.argv[3] == "bf16")
"""


# hidden = inter = 512, two slots: 10240 bytes a token on the bf16 path and
# 11008 on the f16 path, and about 48 for the routing: 4 MiB hold 407 and 379
@pytest.mark.parametrize("tokens,path", [(370, "f16"), (395, "bf16")])
def test_mixed_layer_at_the_scratch_limit(tokens, path):
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT, str(tokens), path], capture_output=True, text=True,
                       cwd=ROOT, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
