"""The f16 prefill path's row scales: rows whose largest magnitude is a
denormal or close to the largest float, and rows whose largest element the
weights do not look at. One routed and one shared expert, so that h of either
follows from two of the oracle's matvecs; each token against the oracle's
layer."""
import numpy as np
import pytest

from sepia_amd import hip, synth
from test_gpu_parity import Launches, check_route, make_layer, run_prefill

pytestmark = pytest.mark.gpu
# (gate/up, down, shared gate/up, shared down): both families mixed, and the real checkpoint's formats
TYPES = [(12, 13, 10, 14), (11, 18, 13, 12), (17, 18, 13, 14), (23, 8, 8, 18)]
H = I = 512


@pytest.fixture(scope="module")
def dev():
    return hip.Device()


def layer(dev, rng, types):
    tg, td, ts, tsd = types
    desc, spec, bufs = make_layer(dev, rng, hidden=H, inter=I, n_routed=1, n_shared=1, tg=tg, tu=tg, td=td, ts=ts,
                                  tsd=tsd, topk=1)
    spec["router_w"][:] = 0.0   # both experts weigh the same, whatever x
    dev.upload(bufs["rw"], spec["router_w"])
    return desc, spec, bufs


def rescale(dev, spec, bufs, name, t, factor, columns=None):
    """The f16 scales of a projection's blocks (those of the first columns of each row) times a factor."""
    elems, nbytes = synth.GEOM[t]
    blocks = spec[name][0].reshape(H, -1, nbytes)
    n = blocks.shape[1] if columns is None else columns // elems
    for off in synth.F16_FIELDS[t]:
        f = blocks[:, :n, off:off + 2].copy().view(np.float16) * np.float16(factor)
        blocks[:, :n, off:off + 2] = f.view(np.uint8)
    dev.upload(bufs[name], spec[name][0])


def gate_up(orc, spec, x):
    for g, u, t in (("gate", "up", spec["t_gate"]), ("s_gate", "s_up", spec["ts_gate"])):
        yield (orc.qlinear(t, spec[g][0], I, H, x).astype(np.float64), orc.qlinear(t, spec[u][0], I, H, x).astype(np.float64))


def run(dev, desc, X):
    with Launches(dev) as n:
        out = run_prefill(dev, desc, X)
    assert n.count("sepia_ph_gateup") == 1 and n.count("sepia_ph_down") == 1
    return out


def weight_sums(orc, spec):
    """Largest row sum of |w| of the routed and the shared down projection."""
    for name, t in (("down", spec["t_down"]), ("s_down", spec["ts_down"])):
        yield float(np.abs(orc.dequantize(t, spec[name][0], H * I).reshape(H, I)).sum(axis=1).max())


@pytest.mark.parametrize("types", TYPES, ids=str)
def test_tiny_rows(dev, orc, types):
    """x scaled so that h's largest magnitude is about 2^-k, x itself a denormal, and a token of zeros."""
    rng = np.random.default_rng(sum(types))
    desc, spec, bufs = layer(dev, rng, types)
    base = rng.standard_normal(H).astype(np.float32)
    top = max(np.abs(g * u).max() for g, u in gate_up(orc, spec, base)) / 2   # silu(g) is g / 2 for a tiny g
    rows = [base * np.float32(np.sqrt(2.0 ** -k / top)) for k in (60, 120, 127, 129, 131, 138)]
    rows += [base * np.float32(2.0 ** -130), np.zeros(H, np.float32), base]
    X = np.stack(rows).astype(np.float32)
    y, idx, w = run(dev, desc, X)
    sums = list(weight_sums(orc, spec))
    for t in range(len(X)):
        y_ref, logits, _, _ = orc.moe_layer(spec, X[t])
        check_route(orc, spec, logits, idx[t], w[t])
        assert np.all(np.isfinite(y[t])), t
        # 2e-5 as in the other prefill tests, and for results among the denormals: either side rounds each h, each
        # slot's row and their weighted sum to a multiple of 2^-149
        slack = 2.0 ** -149 * (2 * float(np.dot(w[t], sums)) + 2 * float(w[t].sum()) + 4)
        err = np.abs(y[t].astype(np.float64) - y_ref).max()
        assert err <= 2e-5 * np.abs(y_ref).max() + slack, (t, err)
    for b in bufs.values():
        dev.free(b)


@pytest.mark.parametrize("types", TYPES, ids=str)
def test_huge_rows(dev, orc, types):
    """x scaled so that h's largest magnitude comes close to the largest float, and down weights small enough for a
    finite y."""
    rng = np.random.default_rng(sum(types) + 1)
    desc, spec, bufs = layer(dev, rng, types)
    rescale(dev, spec, bufs, "down", types[1], 2.0 ** -8)
    rescale(dev, spec, bufs, "s_down", types[3], 2.0 ** -8)
    base = rng.standard_normal(H).astype(np.float32)
    base /= np.abs(base).max()
    pos = [np.where(g > 0, g * u, 0.0) for g, u in gate_up(orc, spec, base)]   # silu(g) is g or 0 for a large g
    top = max(np.abs(h).max() for h in pos)
    X = np.stack([base * np.float32(np.sqrt(m / top)) for m in (1.0e37, 1.6e38, 2.9e38, 3.3e38)])
    # a small route weight: y itself stays in range
    desc.global_scale = spec["global_scale"] = 2.0 ** -12
    y, idx, w = run(dev, desc, X)
    for t in range(len(X)):
        y_ref, logits, _, _ = orc.moe_layer(spec, X[t])
        assert np.all(np.isfinite(y_ref)), "the reference overflows: scale the case down"
        assert np.all(np.isfinite(y[t])), t
        # silu(g) u: g and u are each within 2e-6 of the oracle's
        err = np.abs(y[t].astype(np.float64) - y_ref).max()
        assert err <= 2e-5 * np.abs(y_ref).max(), (t, err)
    for b in bufs.values():
        dev.free(b)


@pytest.mark.parametrize("types", TYPES, ids=str)
def test_outliers(dev, orc, types):
    """One element of x many times the rest, in a block whose weights are zero: the other elements keep their
    precision."""
    rng = np.random.default_rng(sum(types) + 2)
    desc, spec, bufs = layer(dev, rng, types)
    for name in ("gate", "up", "s_gate", "s_up"):
        rescale(dev, spec, bufs, name, spec["ts_gate" if name[1] == "_" else "t_gate"], 0.0, columns=256)
    X = rng.standard_normal((4, H)).astype(np.float32)
    X[1:, 77] = (1e3, -1e4, 1e5)
    y, idx, w = run(dev, desc, X)
    for t in range(len(X)):
        y_ref, logits, _, _ = orc.moe_layer(spec, X[t])
        check_route(orc, spec, logits, idx[t], w[t])
        # an element's two planes hold it within 2^-23 of itself or 2^-39 of the row's largest (2e-7 here), the sums
        # are f32: a few 2^-24 a contraction
        err = np.abs(y[t].astype(np.float64) - y_ref).max()
        assert err <= 4e-6 * np.abs(y_ref).max(), (t, err / np.abs(y_ref).max())
    for b in bufs.values():
        dev.free(b)
