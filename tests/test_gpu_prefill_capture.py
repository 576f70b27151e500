"""Prefill layers captured where the scratch holds the bf16 kernels' regions for
the batch but not the f16 kernels': they run on the f16 kernels all the same,
in parts of the batch, so that the bits do not depend on the scratch there is,
and the scratch does not grow. In a process of its own, so that the scratch
has its smallest size, 4 MiB."""
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
from test_gpu_parity import Launches, make_layer, run_prefill

T, H, I, routed, shared, topk, tg, td, ts, tsd = [int(a) for a in sys.argv[3:]]
dev = hip.Device()
L, stream = dev.L, ctypes.c_void_p(dev.stream())
R = ctypes.CDLL("libamdhip64.so")
rng = np.random.default_rng(T)
X = rng.standard_normal((T, H)).astype(np.float32)
desc, spec, bufs = make_layer(dev, rng, hidden=H, inter=I, n_routed=routed, n_shared=shared, tg=tg, tu=tg, td=td, ts=ts,
                              tsd=tsd, topk=topk)
run_prefill(dev, desc, X[:2])   # the weights are on the device, the scratch is there
xs, ys = dev.shared_from(X), dev.alloc(X.nbytes)
n_route = T * (2 * topk + shared)
rs = dev.alloc(4 * n_route)
xp, yp = dev.alloc(X.nbytes, private=True), dev.alloc(X.nbytes, private=True)
rp = dev.alloc(4 * n_route, private=True)
dev.run(L.sepia_gpu_copy, xs, 0, xp, 0, X.size)
size = L.sepia_hip_scratch_bytes()
graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
dev.begin()
assert R.hipStreamBeginCapture(stream, 1) == 0
ok = L.sepia_gpu_moe_prefill(ctypes.byref(desc), T, xp, yp, rp)
assert R.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
dev.end()
assert ok == 1 and L.sepia_hip_scratch_bytes() == size
assert R.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
got = []
for i in range(3):
    assert R.hipGraphLaunch(exe, stream) == 0
    dev.run(L.sepia_gpu_copy, yp, 0, ys, 0, X.size)
    dev.run(L.sepia_gpu_copy, rp, 0, rs, 0, n_route)
    got.append((dev.download(ys, X.size).copy(), dev.download(rs, n_route).copy()))
R.hipGraphExecDestroy(exe)
with Launches(dev) as n:
    want, idx, w = run_prefill(dev, desc, X)
assert n.count("sepia_ph_gateup") == 1 and n.count("sepia_ph_down") == 1
grown = L.sepia_hip_scratch_bytes() > size
route = np.concatenate([idx.ravel().view(np.float32), w.ravel()])
for y, r in got:
    print("max diff %.2e of %.2e" % (np.abs(y - want.ravel()).max(), np.abs(want).max()), flush=True)
    assert np.array_equal(y.view(np.uint32), want.ravel().view(np.uint32))
    assert np.array_equal(r.view(np.uint32), route.view(np.uint32))
assert grown == (sys.argv[2] == "parts")
"""

# hidden = inter = 512, two slots: 10240 bytes a token on the bf16 path and
# 11008 on the f16 path, and about 48 for the routing: 4 MiB hold 407 and 379.
# One long side of 5120 beside 256, one slot: at most 42000 bytes a token on the
# bf16 path and about 44700 on the f16 path: 4 MiB hold 93 there.
CASES = [("whole", 370, 512, 512, 4, 0, 2, 12, 13, 12, 12), ("parts", 395, 512, 512, 4, 0, 2, 12, 13, 12, 12),
         ("parts", 285, 512, 512, 4, 1, 2, 12, 13, 10, 14), ("whole", 92, 256, 5120, 2, 0, 1, 23, 13, 13, 14),
         ("parts", 95, 256, 5120, 2, 0, 1, 23, 13, 13, 14), ("parts", 95, 5120, 256, 2, 0, 1, 13, 23, 13, 14),
         ("parts", 95, 256, 5120, 2, 0, 1, 8, 8, 8, 8)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_layer_at_the_scratch_limit(case):
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT] + [str(a) for a in case], capture_output=True, text=True,
                       cwd=ROOT, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
