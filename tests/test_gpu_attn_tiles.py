"""The matrix-core attention kernels at the sizes where their tiling can go
wrong: head dims off the 16-wide steps, query heads per kv head that do not
divide a tile, token counts at the edges of the 16- and 64-row tiles and of
the bounds in the kernel arguments (64, then 256 a launch), kv ranges off the
16- and 32-row steps and split over workgroups, and NaN or infinite v rows
that only some of a tile's rows see. All against the oracle's restatement of
the reference's loop (src/sepia.c:1203-1247)."""
import ctypes

import numpy as np
import pytest

from sepia_amd import hip
from test_gpu_attn import banded

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


def make(rng, T, H, Hkv, Dh, R, n, window, extra=0):
    kv_dim = Hkv * Dh + extra
    q = (rng.standard_normal(T * H * Dh) * 0.5).astype(np.float32)
    k = (rng.standard_normal(n * kv_dim) * 0.5).astype(np.float32)
    v = (rng.standard_normal(n * kv_dim) * 0.5).astype(np.float32)
    rl = (rng.standard_normal(T * H * R) * 0.5).astype(np.float32)
    qpb = n - T
    hi = [qpb + t for t in range(T)]
    lo = [max(0, h - window + 1) for h in hi]
    tau = np.linspace(1.0, 1.5, T).astype(np.float32)
    return q, k, v, rl, lo, hi, tau, T, H, Hkv, Dh, R, qpb, kv_dim


def check(dev, orc, args):
    got = banded(dev, *args)
    want = orc.banded_attn(*args, 1.0 / args[10])
    # f32 scores of at most a few units: each weight is within about 1e-6
    # relative, and the weighted sums and their quotient are double
    fin = np.isfinite(want)
    assert np.array_equal(fin, np.isfinite(got)) and np.array_equal(np.isnan(want), np.isnan(got))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    err = np.abs(got[fin].astype(np.float64) - want[fin])
    assert not fin.any() or err.max() <= 5e-6 * np.abs(want[fin]).max()


# (T, H, Hkv, Dh, R, kv positions, window): one 16-row tile and its edges
# (rows = T H / Hkv = 16, 17, 32), the 64-row kernel from 33 rows, its tile
# edges (64, 65, 128 rows), bounds in the arguments up to 64 tokens and in
# scratch beyond (65, 256, 257), kv ranges around the steps and long ones
SHAPES = [
    (1, 8, 8, 128, 16, 1, 1), (1, 8, 8, 128, 16, 17, 17), (1, 64, 8, 128, 1024, 4097, 4097), (2, 8, 1, 128, 7, 40, 40),
    (17, 4, 4, 128, 33, 80, 64), (4, 16, 2, 128, 100, 200, 31), (33, 2, 2, 128, 64, 97, 50), (11, 9, 3, 36, 20, 70, 33),
    (4, 16, 1, 100, 300, 333, 333), (5, 16, 1, 4, 8, 64, 64), (3, 48, 3, 124, 9, 150, 20), (64, 3, 3, 64, 40, 65, 32),
    (65, 4, 1, 128, 128, 400, 100), (256, 2, 2, 128, 30, 300, 70), (257, 4, 4, 20, 12, 290, 290), (66, 7, 1, 8, 5, 99, 40),
]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_shapes(dev, orc, shape):
    T, H, Hkv, Dh, R, n, window = shape
    check(dev, orc, make(np.random.default_rng(T * 31 + n), T, H, Hkv, Dh, R, n, window, extra=4 * (T % 3)))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf], ids=["nan", "inf", "-inf"])
@pytest.mark.parametrize("T,H,Hkv,n,window", [(2, 16, 2, 60, 40), (1, 8, 1, 300, 300), (40, 8, 4, 200, 64),
                                              (70, 8, 2, 150, 150)], ids=str)
def test_nonfinite_rows(dev, orc, bad, T, H, Hkv, n, window):
    """A bad v element reaches exactly the tokens whose range holds its row (a
    matrix op would also give 0 * bad to the tile's other tokens), a bad k
    element exactly the scores it enters; neighbours outside every range stay
    unread."""
    rng = np.random.default_rng(T + n)
    args = make(rng, T, H, Hkv, 128, 64, n, window)
    k, v, kv_dim = args[1], args[2], args[13]
    first = args[4][0]
    for row in {n - 1, n - 1 - T // 2, first, max(0, first - 1), min(n - 1, first + T // 2)}:
        v[row * kv_dim + 5 * (row % 20)] = bad
    check(dev, orc, args)
    args = make(rng, T, H, Hkv, 128, 64, n, window)
    args[1][(n - 1) * args[13] + 3] = bad
    args[1][max(0, args[4][0] - 1) * args[13]] = bad
    check(dev, orc, args)


@pytest.mark.parametrize("low", [-np.inf, float(np.finfo(np.float32).min)], ids=["-inf", "lowest"])
@pytest.mark.parametrize("T,H,Hkv,n,window", [(1, 8, 1, 20, 20), (1, 64, 8, 4097, 4097), (2, 16, 2, 60, 40),
                                              (40, 8, 4, 200, 64), (70, 8, 2, 150, 150)], ids=str)
def test_masked_scores(dev, orc, low, T, H, Hkv, n, window):
    """A band bias of -inf or the lowest float takes whole steps, waves and splits out of a row, at its start, at its
    end, everywhere but one position or everywhere: the reference's maximum is over the whole row, so a row gives NaN
    only where every score is -inf."""
    args = make(np.random.default_rng(T + n), T, H, Hkv, 128, n, n, window)
    rel = args[3].reshape(T, H, n)   # by distance from the token
    rel[:, 0, min(window, n) // 2:] = low
    rel[:, 1, :min(window, n) // 2 + 1] = low
    rel[:, 2, :] = low
    rel[:, 2, min(5, T - 1):1 + min(5, T - 1)] = 0.25
    rel[T - 1, 3, :] = low
    check(dev, orc, args)


@pytest.mark.parametrize("T,H,Hkv,n", [(1, 8, 1, 20), (3, 16, 2, 70), (60, 4, 2, 200)], ids=str)
@pytest.mark.parametrize("shared", ["q", "k", "v", "rel_logits"])
def test_output_in_an_input(dev, orc, shared, T, H, Hkv, n):
    """attn_out may be one of the inputs: every input is read before the first output is written (q, which a
    workgroup reads for its own outputs only, in any case)."""
    args = make(np.random.default_rng(T + n), T, H, Hkv, 128, 128, n, n)
    q, k, v, rl, lo, hi, tau, _, _, _, Dh, R, qpb, kv_dim = args
    names = ["q", "k", "v", "rel_logits"]
    bufs = [dev.shared_from(a) for a in (q, k, v, rl)]
    out = bufs[names.index(shared)]
    c = [ctypes.cast(a, ctypes.c_void_p) for a in ((ctypes.c_int64 * T)(*lo), (ctypes.c_int64 * T)(*hi),
                                                   (ctypes.c_float * T)(*tau))]
    dev.run(dev.L.sepia_gpu_banded_attn, *bufs, out, *c, T, H, Hkv, Dh, R, qpb, kv_dim, 1.0 / Dh)
    got = dev.download(out, T * H * Dh)
    want = orc.banded_attn(*args, 1.0 / Dh)
    assert np.abs(got.astype(np.float64) - want).max() <= 5e-6 * np.abs(want).max()
    for b in bufs:
        dev.free(b)


@pytest.mark.parametrize("T,H,Hkv", [(16384, 64, 4), (16, 32768, 16384)], ids=["tile", "wave"])
def test_weights_correctly_rounded(dev, T, H, Hkv):
    """The weights are double exponentials rounded to f32: with scores 0 and -x, x >= 40, and v rows of 0 and 1 a
    head's output is its second weight, e^-x (1 + e^-x rounds to 1 within 5e-18), which a double good to 2^-51 rounds
    like the exact value but for one x in 10^8."""
    x = np.random.default_rng(T).uniform(40.0, 80.0, T * H).astype(np.float32)
    q = np.zeros((T * H, 4), np.float32)
    q[:, 0] = -4.0 * x   # 1 / head dim is 1/4
    k, v = np.zeros((2, Hkv, 4), np.float32), np.zeros((2, Hkv, 4), np.float32)
    k[1, :, 0] = v[1] = 1.0
    got = banded(dev, q.reshape(-1), k.reshape(-1), v.reshape(-1), np.zeros(T * H, np.float32), [0] * T, [1] * T,
                 [1.0] * T, T, H, Hkv, 4, 1, 1, Hkv * 4).reshape(T * H, 4)
    want = np.exp(-x.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got, np.broadcast_to(want[:, None], got.shape)), int((got[:, 0] != want).sum())


def test_more_tokens_than_a_launch(dev, orc):
    """Over 32768 tokens, the most a launch takes: the second one starts at its own q, bounds and positions."""
    T = 32768 + 70
    check(dev, orc, make(np.random.default_rng(8), T, 1, 1, 4, 8, T, 9))
