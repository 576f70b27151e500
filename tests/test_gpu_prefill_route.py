"""The prefill's router and grouping launches at the edges of their tiles:
tokens and router rows around 16, row lengths of few and of odd numbers of
128-column chunks (fewer than the loads in flight, and none left over), both
tile sizes, more experts than one scan thread holds, and routers at a 4-byte
offset, which keep the f32 tile kernel. Selection, weights and outputs per
token against the oracle's layer; the launch counts show the kernel."""
import numpy as np
import pytest

from sepia_amd import hip
from test_gpu_parity import Launches, assert_close, check_route, make_layer, run_prefill

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


def check(dev, orc, hidden, n_routed, n_shared, topk, T, kernel, rw_off=0, step=1):
    rng = np.random.default_rng(hidden + 17 * T + n_routed)
    desc, spec, bufs = make_layer(dev, rng, hidden=hidden, inter=256, n_routed=n_routed, n_shared=n_shared, tg=12,
                                  tu=12, td=13, ts=12, tsd=13, topk=topk, rw_off=rw_off)
    X = rng.standard_normal((T, hidden)).astype(np.float32)
    with Launches(dev) as n:
        y, idx, w = run_prefill(dev, desc, X)
    for k in ("sepia_pf_route", "sepia_pf_route_m", "sepia_pf_route_m2"):
        assert n.count(k) == (1 if k == kernel else 0), k
    for t in sorted({0, T - 1, *range(0, T, step)}):
        y_ref, logits, idx_ref, _ = orc.moe_layer(spec, X[t])
        chosen = check_route(orc, spec, logits, idx[t], w[t])   # weights within 1e-4: logits within about that
        if chosen != list(idx_ref):
            y_ref, _, _, _ = orc.moe_layer(spec, X[t], force_idx=chosen)
        # f32 sums of exact products, each term within 2^-22 of the row's largest: 2e-5 of ||y||_inf is ample
        assert_close(y[t], y_ref, tol=2e-5, what="token %d" % t, gate=False)
    for b in bufs.values():
        dev.free(b)


# chunks of 128 columns: 2, 6, 8, 10; router rows 3, 16, 17, 35
@pytest.mark.parametrize("hidden,n_routed,n_shared", [(256, 3, 0), (768, 15, 1), (1024, 15, 2), (1280, 32, 3)], ids=str)
@pytest.mark.parametrize("T", [1, 15, 16, 17, 50])
def test_tile_edges(dev, orc, hidden, n_routed, n_shared, T):
    check(dev, orc, hidden, n_routed, n_shared, 3, T, "sepia_pf_route_m")


@pytest.mark.parametrize("hidden,T", [(256, 577), (512, 592), (768, 593)], ids=str)
def test_large_tiles(dev, orc, hidden, T):
    """Over 1152 tiles of 16 x 16: the 32 x 32 kernel; 500 routed experts and over 4096 pairs in the grouping."""
    check(dev, orc, hidden, 500, 3, 8, T, "sepia_pf_route_m2", step=37)


def test_unaligned_router(dev, orc):
    check(dev, orc, 768, 15, 1, 3, 17, "sepia_pf_route", rw_off=4)
