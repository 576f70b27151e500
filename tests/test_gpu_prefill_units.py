"""The f16 prefill kernels at the sizes where their tiling can go wrong: units
at every edge of their 16-pair tiles (16, 17, 32, 33, 48, 49, 64, 65 pairs of
one expert), rows of few and of odd numbers of blocks (weight groups of 1, 2
and 4 blocks end inside them), every format as gate/up and as down, and layers
whose formats come from both families, which run on these kernels too. Each
token against the oracle's layer; the launch counts show the path."""
import numpy as np
import pytest

from sepia_amd import hip
from test_gpu_parity import Launches, assert_close, check_route, make_layer, run_prefill

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


def check(dev, orc, hidden, inter, types, T, n_routed=2, n_shared=1):
    """Two routed experts, both selected by every token: each has T pairs."""
    tg, td, ts, tsd = types
    rng = np.random.default_rng(hidden + 13 * T + tg + 3 * td)
    desc, spec, bufs = make_layer(dev, rng, hidden=hidden, inter=inter, n_routed=n_routed, n_shared=n_shared, tg=tg,
                                  tu=tg, td=td, ts=ts, tsd=tsd, topk=n_routed)
    X = rng.standard_normal((T, hidden)).astype(np.float32)
    with Launches(dev) as n:
        y, idx, w = run_prefill(dev, desc, X)
    assert n.count("sepia_ph_gateup") == 1 and n.count("sepia_ph_down") == 1
    for t in range(T):
        y_ref, logits, idx_ref, _ = orc.moe_layer(spec, X[t])
        chosen = check_route(orc, spec, logits, idx[t], w[t])
        if chosen != list(idx_ref):
            y_ref, _, _, _ = orc.moe_layer(spec, X[t], force_idx=chosen)
        # f32 sums of exact products, each term within 2^-22 of the row's largest: 2e-5 of ||y||_inf is ample
        assert_close(y[t], y_ref, tol=2e-5, what="%s T=%d token %d" % (types, T, t), gate=False)
    for b in bufs.values():
        dev.free(b)


@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 48, 49, 64, 65])
@pytest.mark.parametrize("types", [(17, 18, 13, 14), (10, 14, 12, 13), (11, 23, 17, 12)], ids=str)
def test_unit_edges(dev, orc, types, T):
    check(dev, orc, 512, 512, types, T)


# (hidden, inter): rows of 2 and 4, 6 and 2, 10 and 6 blocks; of 3, 5 and 7 where the rows stay 4-byte aligned
@pytest.mark.parametrize("shape,types", [
    ((512, 1024), (17, 18, 17, 18)), ((1536, 512), (18, 17, 18, 17)), ((2560, 1536), (17, 18, 13, 14)),
    ((1536, 1536), (14, 11, 11, 14)), ((512, 1536), (8, 8, 8, 8)), ((2560, 512), (23, 8, 8, 23)),
    ((768, 1280), (12, 13, 13, 12)), ((1280, 1792), (10, 23, 23, 10)), ((768, 768), (13, 12, 10, 13)),
    ((256, 256), (12, 13, 12, 13))], ids=str)
@pytest.mark.parametrize("T", [5, 40, 70])
def test_row_lengths(dev, orc, shape, types, T):
    check(dev, orc, shape[0], shape[1], types, T)


def test_many_units(dev, orc):
    """More units than the launch order keeps (they are then dealt to the XCDs): 3 routed and 2 shared experts
    with 1700 pairs each."""
    rng = np.random.default_rng(3)
    desc, spec, bufs = make_layer(dev, rng, hidden=512, inter=256, n_routed=3, n_shared=2, tg=12, tu=12, td=13, ts=13,
                                  tsd=12, topk=3)
    X = rng.standard_normal((1700, 512)).astype(np.float32)
    y, idx, w = run_prefill(dev, desc, X)
    for t in range(0, 1700, 61):
        y_ref, logits, idx_ref, _ = orc.moe_layer(spec, X[t])
        chosen = check_route(orc, spec, logits, idx[t], w[t])
        if chosen != list(idx_ref):
            y_ref, _, _, _ = orc.moe_layer(spec, X[t], force_idx=chosen)
        assert_close(y[t], y_ref, tol=2e-5, what="token %d" % t, gate=False)
    for b in bufs.values():
        dev.free(b)
