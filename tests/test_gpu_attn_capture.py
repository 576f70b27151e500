"""Banded attention captured where the scratch does not hold the splits it
would take: fewer splits, the same outputs up to the order of double sums, and
the scratch does not grow. In a process of its own, so that the scratch has
its smallest size, 4 MiB."""
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
import oracle
from sepia_amd import hip
from test_gpu_attn_tiles import make

T, H, Hkv, n, window = [int(a) for a in sys.argv[2:]]
oracle.build()
dev = hip.Device()
L, stream = dev.L, ctypes.c_void_p(dev.stream())
R = ctypes.CDLL("libamdhip64.so")
args = make(np.random.default_rng(T), T, H, Hkv, 128, 64, n, window)
q, k, v, rl, lo, hi, tau, _, _, _, Dh, rel, qpb, kv_dim = args
assert L.sepia_hip_reserve_scratch(1) == 1
size = L.sepia_hip_scratch_bytes()
bufs = [dev.alloc(a.nbytes, private=True) for a in (q, k, v, rl)]
for a, p in zip((q, k, v, rl), bufs):
    s = dev.shared_from(a)
    dev.run(L.sepia_gpu_copy, s, 0, p, 0, a.size)
    dev.free(s)
out, host = dev.alloc(q.nbytes, private=True), dev.alloc(q.nbytes)
c = [ctypes.cast(a, ctypes.c_void_p) for a in ((ctypes.c_int64 * T)(*lo), (ctypes.c_int64 * T)(*hi),
                                               (ctypes.c_float * T)(*tau))]
graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
dev.begin()
assert R.hipStreamBeginCapture(stream, 1) == 0
ok = L.sepia_gpu_banded_attn(*bufs, out, *c, T, H, Hkv, Dh, rel, qpb, kv_dim, 1.0 / Dh)
assert R.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
dev.end()
assert ok == 1 and L.sepia_hip_scratch_bytes() == size
assert R.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
got = []
for i in range(3):
    assert R.hipGraphLaunch(exe, stream) == 0
    dev.run(L.sepia_gpu_copy, out, 0, host, 0, q.size)
    got.append(dev.download(host, q.size).copy())
R.hipGraphExecDestroy(exe)
dev.run(L.sepia_gpu_banded_attn, *bufs, out, *c, T, H, Hkv, Dh, rel, qpb, kv_dim, 1.0 / Dh)
assert L.sepia_hip_scratch_bytes() > size   # uncaptured it takes all its splits
want = oracle.banded_attn(*args, 1.0 / Dh)
for y in got:
    assert np.array_equal(y.view(np.uint32), got[0].view(np.uint32))
    assert np.abs(y.astype(np.float64) - want).max() <= 5e-6 * np.abs(want).max()
"""


# (T, H, Hkv, kv positions, window): one token of 64 heads over 64 splits of 66560 bytes (the wave kernel), and token
# counts whose bounds are in the scratch too, over 57 and 29 splits of 0.6 and 1.2 MB (the tile kernel)
@pytest.mark.parametrize("case", [(1, 64, 8, 20480, 20480), (70, 8, 1, 9000, 9000), (70, 16, 2, 4000, 1500)], ids=str)
def test_fewer_splits(case):
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT] + [str(a) for a in case], capture_output=True, text=True,
                       cwd=ROOT, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
