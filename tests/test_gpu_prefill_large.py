"""Expert matrices of more than 4 GiB on each of the prefill's three paths: a
row's offset in its matrix does not fit 32 bits. One routed expert on random
blocks; h and y against the library's own matvec over slices of the same
matrices that start at their own 64-bit offsets."""
import ctypes

import numpy as np
import pytest

from sepia_amd import hip, synth
from test_gpu_parity import Launches, assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


def matvec(dev, t, w, rows, cols, x, step=16384):
    """w . x over slices of rows."""
    rb = synth.row_bytes(t, cols)
    xb, yb = dev.shared_from(x), dev.alloc(4 * step)
    out = []
    for r in range(0, rows, step):
        n = min(step, rows - r)
        dev.run(dev.L.sepia_gpu_matvec_q, t, w, r * rb, xb, yb, n, cols)
        out.append(dev.download(yb, n).copy())
    dev.free(xb)
    dev.free(yb)
    return np.concatenate(out)


# format, hidden = inter (so that each of the three matrices passes 4 GiB), kernel
@pytest.mark.parametrize("t,n,kernel", [(12, 87552, "sepia_pf_gateup_q"), (8, 63744, "sepia_ph_gateup"),
                                        (14, 72960, "sepia_pf_gateup")], ids=["int8", "f16", "bf16"])
def test_matrices_over_4_gib(dev, t, n, kernel):
    L = dev.L
    rb, (elems, _) = synth.row_bytes(t, n), synth.GEOM[t]
    assert n * rb > 1 << 32
    ws = [dev.alloc(n * rb, private=True) for _ in range(3)]
    rng = np.random.default_rng(n)
    rw, rbias = np.zeros((1, n), np.float32), np.zeros(1, np.float32)
    x = rng.standard_normal((2, n)).astype(np.float32)
    bufs = [dev.shared_from(a) for a in (rw, rbias, x)] + [dev.alloc(x.nbytes), dev.alloc(256)]
    try:
        for i, w in enumerate(ws):
            dev.run(L.sepia_hip_synth_blocks, t, w, 0, n * (n // elems), 7 + i, synth.SCALE_LO, synth.SCALE_HI)
        d = hip.MoeLayerDesc(hidden=n, inter=n, n_routed=1, n_shared=0, topk=1, route_scale=1.0, global_scale=1.0,
                             router_w=bufs[0], router_bias=bufs[1])
        for name, w in zip(("gate", "up", "down"), ws):
            setattr(d, name, hip.ExpertTensor(w, 0, n * rb, t))
        with Launches(dev) as count:
            dev.run(L.sepia_gpu_moe_prefill, ctypes.byref(d), 2, bufs[2], bufs[3], bufs[4])
        assert count.count(kernel) == 1
        y = dev.download(bufs[3], 2 * n).reshape(2, n)
        weight = dev.download(bufs[4], 2, offset=8)
        for k in range(2):
            g, u = (matvec(dev, t, w, n, n, x[k]).astype(np.float64) for w in ws[:2])
            # either side: exact products (bf16: within 2.3e-5, of random sign), f32 sums of 7e4 terms in two
            # contractions; a row that is not the right one is of the outputs' own size off
            want = weight[k] * matvec(dev, t, ws[2], n, n, (g / (1 + np.exp(-np.maximum(g, -600.0))) * u).astype(np.float32))
            assert_close(y[k], want, tol=1e-4, what="token %d" % k, gate=False)
    finally:
        for b in ws + bufs:
            dev.free(b)
