"""RMSNorm's three kernels at the edges of their ranges: rows around the 512
floats a wave holds, around the 8192 a workgroup holds in registers, row
counts around the four of a workgroup, lengths that are no multiple of four
and weights or rows off 16 bytes (the general kernel), each also in place."""
import numpy as np
import pytest

from sepia_amd import hip
from test_gpu_parity import Launches

pytestmark = pytest.mark.gpu
KERNELS = ("sepia_rmsnorm_f32", "sepia_rmsnorm_wave", "sepia_rmsnorm_row")


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


@pytest.mark.parametrize("n", [1, 3, 4, 64, 128, 252, 256, 260, 508, 510, 512, 516, 1020, 1024, 4100, 6144, 8192, 8196,
                               20000])
@pytest.mark.parametrize("rows", [1, 4, 5, 67])
@pytest.mark.parametrize("w_off", [0, 4, 16])
def test_rmsnorm(dev, n, rows, w_off):
    rng = np.random.default_rng(n + rows)
    x = (rng.standard_normal((rows, n)) * np.exp(rng.standard_normal((rows, 1)))).astype(np.float32)
    w = rng.standard_normal(n + w_off // 4).astype(np.float32)
    eps = np.float32(1e-6)
    bx, bw, by = dev.shared_from(x), dev.shared_from(w), dev.alloc(x.nbytes)
    with Launches(dev) as got:
        dev.run(dev.L.sepia_gpu_rmsnorm_off, bw, w_off, bx, by, rows, n, eps)
    want = KERNELS[0] if n % 4 or w_off == 4 else KERNELS[1] if n <= 512 else KERNELS[2]
    for k in KERNELS:
        assert got.count(k) == (k == want), k
    y = dev.download(by, x.size).reshape(rows, n)
    x2 = x.astype(np.float64)
    ref = w[w_off // 4:] * (x2 / np.sqrt((x2 ** 2).mean(axis=1, keepdims=True) + np.float64(eps)))
    # the sum of squares passes at most 79 + 8 roundings of 2^-24 (n / 256 terms a thread, then the tree), all terms
    # positive; its square root halves them; divide, add, sqrt, reciprocal and the two products add under 6
    assert np.all(np.abs(y - ref) <= (87 / 2 + 6) * 2.0 ** -24 * np.abs(ref) + 1e-37)
    dev.run(dev.L.sepia_gpu_rmsnorm_off, bw, w_off, bx, bx, rows, n, eps)
    assert np.array_equal(dev.download(bx, x.size).view(np.uint32), y.reshape(-1).view(np.uint32))
    for b in (bx, bw, by):
        dev.free(b)
