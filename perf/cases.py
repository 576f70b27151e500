"""The work that is measured: what a user of this library has it do, through
its C ABI (sepia_amd.hip), over the sizes, formats and directions that an
inference engine of a routed-MoE model meets.

A pass is one batch of the ABI (begin, the ops, end), as an engine issues it:
end waits for the work. Weights, inputs and outputs are private device
buffers, made from the seed; outputs come back as views of the output
buffers. Weight blocks are random bytes with f16 scales in [2^-10, 2^-6],
activations are N(0, 1), routers N(0, 0.02) with a bias in [-0.1, 0.1].
"""
import ctypes
import math
import os
import re

import numpy as np
import torch

from sepia_amd import hip

Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, IQ2_XS, IQ3_XXS, IQ4_XS = 8, 10, 11, 12, 13, 14, 17, 18, 23
# ggml type: (weights of a block, its bytes, offsets of its f16 scales)
BLOCK = {Q8_0: (32, 34, (0,)), Q2_K: (256, 84, (80, 82)), Q3_K: (256, 110, (108,)), Q4_K: (256, 144, (0, 2)),
         Q5_K: (256, 176, (0, 2)), Q6_K: (256, 210, (208,)), IQ2_XS: (256, 74, (0,)), IQ3_XXS: (256, 98, (0,)),
         IQ4_XS: (256, 136, (0,))}
SCALE_LO, SCALE_HI = 2.0 ** -10, 2.0 ** -6
ROUTE_SCALE = 8.0
NAMES = {Q8_0: "q8_0", Q2_K: "q2_k", Q3_K: "q3_k", Q4_K: "q4_k", Q5_K: "q5_k", Q6_K: "q6_k", IQ2_XS: "iq2_xs",
         IQ3_XXS: "iq3_xxs", IQ4_XS: "iq4_xs"}
TYPES = {name: t for t, name in NAMES.items()}


def listed():
    real = dict(gate="iq2_xs", down="iq3_xxs", s_gate="q5_k", s_down="q6_k")
    low = dict(gate="q2_k", down="q3_k", s_gate="q4_k", s_down="q4_k")
    moe = dict(hidden=6144, inter=3072, routed=256, shared=2, topk=6)
    return [
        # decode, the smallest calls: the k projections of 8 layers
        dict(name="matvec_kv_q8_0", op="matvec", type="q8_0", rows=2048, cols=6144, count=8),
        # decode: square projections in a codebook format
        dict(name="matvec_iq3_6144", op="matvec", type="iq3_xxs", rows=6144, cols=6144, count=8),
        # decode: the output head, an odd vocabulary
        dict(name="matvec_head_q4_k", op="matvec", type="q4_k", rows=100003, cols=6144, count=1),
        # decode with the routing on the host: the six experts of a token, one call each
        dict(name="expert_ffn_x6", op="ffn", gate="q2_k", down="q3_k", hidden=6144, inter=3072, experts=32, count=6),
        # decode: one token through the MoE halves of 4 layers
        dict(name="moe_decode", op="moe", tokens=0, layers=4, **moe, **low),
        dict(name="moe_decode_real", op="moe", tokens=0, layers=4, **moe, **real),
        # a few tokens at once (several users' tokens, or drafted ones)
        dict(name="moe_batch_9", op="moe", tokens=9, layers=1, **moe, **real),
        # prefill: an ordinary chunk in the low-bit formats
        dict(name="moe_prefill_512", op="moe", tokens=512, layers=1, **moe, **low),
        # prefill: the longest chunk, the formats of the real checkpoint, a ragged length
        dict(name="moe_prefill_1999_real", op="moe", tokens=1999, layers=1, **moe, **real),
        # prefill of a layer whose formats come from two families (4-bit gate and up, 6-bit down)
        dict(name="moe_prefill_mixed", op="moe", tokens=300, layers=1, gate="q4_k", down="q6_k", s_gate="q4_k",
             s_down="q6_k", hidden=4096, inter=2048, routed=64, shared=1, topk=4),
        # the attention half of a decode token: norm, projections, short convolutions, attention over a long
        # context, output projection, residual
        dict(name="attn_block_decode", op="block", sliding=False, pos=20000, hidden=6144, heads=64, kv_heads=8,
             window=1024),
        # attention of a prefill chunk over a longer context
        dict(name="attn_prefill_500", op="attn", sliding=False, tokens=500, pos=1500, heads=64, kv_heads=8,
             window=1024),
    ]


MIXES = [("q2_k", "q3_k", "q4_k", "q4_k"), ("q3_k", "q2_k", "q2_k", "q3_k"), ("iq2_xs", "iq3_xxs", "q5_k", "q6_k"),
         ("iq2_xs", "iq4_xs", "q8_0", "q8_0"), ("iq3_xxs", "iq3_xxs", "q5_k", "q6_k"), ("q4_k", "q6_k", "q4_k", "q6_k"),
         ("q3_k", "q5_k", "q5_k", "q6_k"), ("q4_k", "q4_k", "q6_k", "q6_k")]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "ffn", "moe", "moe", "moe", "block", "attn"])
    if op == "matvec":
        cols = 256 * _log(rng, 4, 48)
        if rng.random() < 0.7:
            cols = max(1024, cols // 1024 * 1024)
        rows = _log(rng, 64, max(64, min(100000, 600000000 // cols)))
        return dict(op=op, type=rng.choice(sorted(TYPES)), rows=rows, cols=cols,
                    count=rng.randint(4, 12) if rows < 16384 else 1)
    if op == "ffn":
        mix = rng.choice(MIXES)
        return dict(op=op, gate=mix[0], down=mix[1], hidden=1024 * rng.randint(1, 6), inter=1024 * rng.randint(1, 3),
                    experts=16, count=rng.randint(2, 8))
    if op == "moe":
        mix = rng.choice(MIXES)
        tokens = 0 if rng.random() < 0.35 else _log(rng, 2, 1600)
        hidden, inter = 256 * rng.randint(4, 24), 256 * rng.randint(2, 12)
        if rng.random() < 0.6 or tokens == 0:
            hidden, inter = max(1024, hidden // 1024 * 1024), max(1024, inter // 1024 * 1024)
        routed = rng.choice([16, 40, 64, 128, 256])
        if hidden * inter * routed > 2500000000:
            routed = 64
        return dict(op=op, tokens=tokens, layers=rng.randint(2, 4) if tokens == 0 else 1, hidden=hidden, inter=inter,
                    routed=routed, shared=rng.randint(0, 2), topk=rng.randint(2, 6), gate=mix[0], down=mix[1],
                    s_gate=mix[2], s_down=mix[3])
    sliding = rng.random() < 0.5
    kv_heads, window = (16, 512) if sliding else (8, 1024)
    if op == "block":
        return dict(op=op, sliding=sliding, pos=_log(rng, 30, 30000), hidden=1024 * rng.randint(1, 6), heads=64,
                    kv_heads=kv_heads, window=window)
    tokens = _log(rng, 2, 500)
    return dict(op=op, sliding=sliding, tokens=tokens, pos=_log(rng, 1, 1000000 // tokens if tokens > 60 else 16000),
                heads=64, kv_heads=kv_heads, window=window)


# ------------------------------------------------------------------ buffers --
_device = None


def _dev():
    global _device
    if _device is None:
        _device = hip.Device()
    return _device


class _Memory:
    """A private device buffer of the library as torch takes it. torch holds this object for as long as any tensor
    over it lives (outputs outlive the state that made them), and the buffer is given back after that."""

    def __init__(self, nbytes):
        self.dev = _dev()
        self.handle = self.dev.alloc(nbytes, private=True)
        addr = self.dev.L.sepia_gpu_gpu_addr(self.handle)
        self.__cuda_array_interface__ = dict(shape=(nbytes,), typestr="|u1", data=(addr, False), version=2)

    def __del__(self):
        if getattr(self, "handle", None):
            torch.cuda.synchronize()   # torch's work on it is done
            self.dev.L.sepia_gpu_free(self.handle)


class Buf:
    """A private device buffer: the library's handle and torch's view of it."""

    def __init__(self, nbytes):
        memory = _Memory(nbytes)
        self.handle = memory.handle
        self.bytes = torch.as_tensor(memory, device="cuda")

    def f32(self, *shape):
        return self.bytes.view(torch.float32).view(*shape)

    def fill(self, t):
        self.bytes.view(t.dtype).copy_(t.reshape(-1))
        return self


def _of(t):
    return Buf(t.numel() * t.element_size()).fill(t)


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(seed * 1000003 + salt)


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _row_bytes(t, cols):
    elems, nbytes, _ = BLOCK[t]
    return cols // elems * nbytes


def _raw(g, t, n_weights, out=None):
    """Random blocks of n_weights weights: bytes at random, scales in [SCALE_LO, SCALE_HI]."""
    elems, nbytes, scales = BLOCK[t]
    n = n_weights // elems
    if out is None:
        out = torch.empty(n * nbytes, dtype=torch.uint8, device="cuda")
    whole = out.numel() // 8 * 8
    out[:whole].view(torch.int64).random_(-2 ** 63, None, generator=g)
    out[whole:].random_(0, 256, generator=g)
    blocks = out.view(n, nbytes)
    for off in scales:
        s = torch.rand(n, 1, generator=g, device="cuda") * (SCALE_HI - SCALE_LO) + SCALE_LO
        blocks[:, off:off + 2] = s.to(torch.float16).view(torch.uint8).view(n, 2)
    return out


def _weights(seed, salt, t, n_weights):
    elems, nbytes, _ = BLOCK[t]
    b = Buf(n_weights // elems * nbytes)
    _raw(_gen(seed, salt), t, n_weights, b.bytes)
    return b


# ------------------------------------------------------------------- inputs --
# Each pass's inputs by name, as torch tensors on the GPU (weights apart), the
# same for prepare() and exact().
def _router(case, seed, layer):
    g = _gen(seed, 100 + 10 * layer)
    n, h = case["routed"] + case["shared"], case["hidden"]
    return _normal(g, n, h, scale=0.02), torch.rand(case["routed"], generator=g, device="cuda") * 0.2 - 0.1


def _tokens(case, seed, layer, router, bias):
    """The layer's tokens. Those whose selection or its order two correct implementations may see differently
    (neighbouring scores closer than f32 sums tell apart) are passed over."""
    n = max(1, case["tokens"])
    x = _normal(_gen(seed, 101 + 10 * layer), n + n // 8 + 32, case["hidden"])
    score = torch.sigmoid(x.double() @ router[:case["routed"]].double().T) + bias.double()
    top = score.topk(min(case["topk"] + 1, case["routed"]), dim=1).values
    gap = (top[:, :-1] - top[:, 1:]).min(dim=1).values
    return x[torch.nonzero(gap > 2e-5)[:n, 0]].contiguous()


def _moe_types(case):
    return [TYPES[case[k]] for k in ("gate", "gate", "down", "s_gate", "s_gate", "s_down")]


def _moe_shapes(case):
    h, i = case["hidden"], case["inter"]
    return [(i, h), (i, h), (h, i), (i, h), (i, h), (h, i)]


def _attn_inputs(case, seed, tokens):
    g = _gen(seed, 1)
    h, hk, w, dh = case["heads"], case["kv_heads"], case["window"], 128
    n = case["pos"] + tokens
    return dict(q=_normal(g, tokens, h, dh, scale=0.3), k=_normal(g, n, hk * dh, scale=0.5),
                v=_normal(g, n, hk * dh, scale=0.5), rel=_normal(g, tokens, h, w, scale=0.5))


def _bounds(case, tokens):
    """kv ranges and bias scales of the chunk's tokens: the window of a sliding layer, everything before the
    token and a bias that grows with the logarithm of the context of a global one."""
    pos = [case["pos"] + t for t in range(tokens)]
    lo = [max(0, p - case["window"] + 1) if case["sliding"] else 0 for p in pos]
    tau = [1.0 if case["sliding"] else 1.0 + 0.1 * math.log(max(1.0, (p + 1) / 128.0)) for p in pos]
    return lo, pos, tau


BLOCK_TAPS, BLOCK_D_REL = 4, 16


def _block_shapes(case):
    """Projections of an attention block: name -> (rows, columns); all Q8_0, as the real checkpoint's."""
    h, q, kv = case["hidden"], case["heads"] * 128, case["kv_heads"] * 128
    return dict(q=(q, h), k=(kv, h), v=(kv, h), r=(case["heads"] * BLOCK_D_REL, h), o=(h, q))


def _block_inputs(case, seed):
    g = _gen(seed, 2)
    h, kv, taps = case["hidden"], case["kv_heads"] * 128, BLOCK_TAPS
    one = lambda n: 1.0 + _normal(g, n, scale=0.1)  # noqa: E731
    return dict(x=_normal(g, h), norm=one(h), q_norm=one(128), k_norm=one(128),
                conv_k=_normal(g, kv, taps, scale=0.3), conv_v=_normal(g, kv, taps, scale=0.3),
                conv_o=_normal(g, h, taps, scale=0.3), hist_k=_normal(g, taps - 1, kv), hist_v=_normal(g, taps - 1, kv),
                hist_o=_normal(g, taps - 1, h), rel_proj=_normal(g, BLOCK_D_REL, case["window"], scale=0.05),
                k=_normal(g, case["pos"] + 1, kv), v=_normal(g, case["pos"] + 1, kv))


# ------------------------------------------------------------------ prepare --
def prepare(case, seed):
    state = {"case": dict(case)}
    op = case["op"]
    if op == "matvec":
        t = TYPES[case["type"]]
        n = case["rows"] * case["cols"]
        state["w"] = [_weights(seed, 10 + i, t, n) for i in range(case["count"])]
        x = _normal(_gen(seed, 1), case["count"], case["cols"])
        state["x"] = [_of(x[i]) for i in range(case["count"])]
        state["y"] = [Buf(4 * case["rows"]) for _ in range(case["count"])]
    elif op == "ffn":
        tg, td = TYPES[case["gate"]], TYPES[case["down"]]
        n = case["experts"] * case["hidden"] * case["inter"]
        state["w"] = [_weights(seed, 10, tg, n), _weights(seed, 11, tg, n), _weights(seed, 12, td, n)]
        size = [_row_bytes(tg, case["hidden"]) * case["inter"]] * 2 + [_row_bytes(td, case["inter"]) * case["hidden"]]
        state["stacks"] = [hip.ExpertTensor(b.handle, 0, s, t) for b, s, t in zip(state["w"], size, (tg, tg, td))]
        state["x"] = _of(_normal(_gen(seed, 1), case["hidden"]))
        state["y"] = [Buf(4 * case["hidden"]) for _ in range(case["count"])]
    elif op == "moe":
        state["layers"] = [_prepare_layer(case, seed, i) for i in range(case["layers"])]
    elif op == "attn":
        state["in"] = {k: _of(v) for k, v in _attn_inputs(case, seed, case["tokens"]).items()}
        state["y"] = Buf(4 * case["tokens"] * case["heads"] * 128)
        state["bounds"] = _c_bounds(case, case["tokens"])
    else:
        state["w"] = {k: _weights(seed, 10 + i, Q8_0, r * c) for i, (k, (r, c)) in enumerate(_block_shapes(case).items())}
        state["in"] = {k: _of(v) for k, v in _block_inputs(case, seed).items()}
        h, q, kv = case["hidden"], case["heads"] * 128, case["kv_heads"] * 128
        sizes = dict(xn=h, q=q, qn=q, k=kv, kc=kv, kn=kv, v=kv, vc=kv, r=case["heads"] * BLOCK_D_REL,
                     rel=case["heads"] * case["window"], a=q, o=h, oc=h, y=h)
        state["t"] = {k: Buf(4 * n) for k, n in sizes.items()}
        state["bounds"] = _c_bounds(case, 1)
    torch.cuda.synchronize()
    return state


def _c_bounds(case, tokens):
    lo, hi, tau = _bounds(case, tokens)
    arrays = (ctypes.c_int64 * tokens)(*lo), (ctypes.c_int64 * tokens)(*hi), (ctypes.c_float * tokens)(*tau)
    return arrays, [ctypes.cast(a, ctypes.c_void_p) for a in arrays]


def _prepare_layer(case, seed, layer):
    router, bias = _router(case, seed, layer)
    x = _tokens(case, seed, layer, router, bias)
    n, sel = x.shape[0], case["topk"] + case["shared"]
    bufs = dict(router=_of(router), bias=_of(bias), x=_of(x), y=Buf(4 * x.numel()), route=Buf(4 * n * (case["topk"] + sel)))
    d = hip.MoeLayerDesc(hidden=case["hidden"], inter=case["inter"], n_routed=case["routed"], n_shared=case["shared"],
                         topk=case["topk"], route_scale=ROUTE_SCALE, global_scale=1.0, router_w=bufs["router"].handle,
                         router_bias=bufs["bias"].handle)
    for i, (key, t, (rows, cols)) in enumerate(zip(("gate", "up", "down", "s_gate", "s_up", "s_down"), _moe_types(case),
                                                   _moe_shapes(case))):
        experts = case["routed"] if i < 3 else case["shared"]
        if experts:
            bufs[key] = _weights(seed, 110 + 10 * layer + i, t, experts * rows * cols)
            setattr(d, key, hip.ExpertTensor(bufs[key].handle, 0, rows * _row_bytes(t, cols), t))
    return dict(desc=d, bufs=bufs, n=n)


# ---------------------------------------------------------------------- run --
def run(state):
    case, dev = state["case"], _dev()
    L, op = dev.L, case["op"]
    dev.begin()
    if op == "matvec":
        t = TYPES[case["type"]]
        for w, x, y in zip(state["w"], state["x"], state["y"]):
            dev.check(L.sepia_gpu_matvec_q(t, w.handle, 0, x.handle, y.handle, case["rows"], case["cols"]), op)
        out = [y.f32(-1) for y in state["y"]]
    elif op == "ffn":
        g, u, d = (ctypes.byref(s) for s in state["stacks"])
        for i, y in enumerate(state["y"]):
            dev.check(L.sepia_gpu_expert_ffn(g, u, d, case["experts"], (5 * i + 3) % case["experts"], case["hidden"],
                                             case["inter"], state["x"].handle, y.handle), op)
        out = [y.f32(-1) for y in state["y"]]
    elif op == "moe":
        out = []
        for s in state["layers"]:
            b = s["bufs"]
            if case["tokens"]:
                ok = L.sepia_gpu_moe_prefill(ctypes.byref(s["desc"]), s["n"], b["x"].handle, b["y"].handle, b["route"].handle)
            else:
                ok = L.sepia_gpu_moe_decode(ctypes.byref(s["desc"]), b["x"].handle, b["y"].handle, b["route"].handle)
            dev.check(ok, op)
            chosen = s["n"] * case["topk"]
            out.append(dict(y=b["y"].f32(s["n"], -1), idx=b["route"].bytes[:4 * chosen].view(torch.int32),
                            w=b["route"].bytes[4 * chosen:].view(torch.float32)))
    elif op == "attn":
        i = state["in"]
        _attention(L, case, i["q"], i["k"], i["v"], i["rel"], state["y"], state["bounds"][1], case["tokens"])
        out = state["y"].f32(case["tokens"], -1)
    else:
        out = _run_block(dev, case, state)
    dev.end()
    return out


def _attention(L, case, q, k, v, rel, y, bounds, tokens):
    kv_heads = case["kv_heads"]
    _dev().check(L.sepia_gpu_banded_attn(q.handle, k.handle, v.handle, rel.handle, y.handle, *bounds, tokens,
                                         case["heads"], kv_heads, 128, case["window"], case["pos"], kv_heads * 128,
                                         1.0 / 128), "banded_attn")


def _run_block(dev, case, state):
    L, i, t, w = dev.L, state["in"], state["t"], state["w"]
    h, heads, kv_heads = case["hidden"], case["heads"], case["kv_heads"]
    kv, taps, eps = kv_heads * 128, BLOCK_TAPS, 1e-6
    do = lambda ok: dev.check(ok, "block")  # noqa: E731

    def project(name, x, y):
        rows, cols = _block_shapes(case)[name]
        do(L.sepia_gpu_matvec_q(Q8_0, w[name].handle, 0, x.handle, y.handle, rows, cols))

    do(L.sepia_gpu_rmsnorm(i["norm"].handle, i["x"].handle, t["xn"].handle, 1, h, eps))
    for name in ("q", "k", "v", "r"):
        project(name, t["xn"], t[name])
    do(L.sepia_gpu_sconv(i["conv_k"].handle, i["hist_k"].handle, t["k"].handle, t["kc"].handle, kv, taps, 1))
    do(L.sepia_gpu_sconv(i["conv_v"].handle, i["hist_v"].handle, t["v"].handle, t["vc"].handle, kv, taps, 1))
    do(L.sepia_gpu_rmsnorm(i["q_norm"].handle, t["q"].handle, t["qn"].handle, heads, 128, eps))
    do(L.sepia_gpu_rmsnorm(i["k_norm"].handle, t["kc"].handle, t["kn"].handle, kv_heads, 128, eps))
    do(L.sepia_gpu_copy(t["kn"].handle, 0, i["k"].handle, 4 * kv * case["pos"], kv))
    do(L.sepia_gpu_copy(t["vc"].handle, 0, i["v"].handle, 4 * kv * case["pos"], kv))
    do(L.sepia_gpu_rel_project(t["r"].handle, i["rel_proj"].handle, t["rel"].handle, 1, heads, BLOCK_D_REL, case["window"]))
    _attention(L, case, t["qn"], i["k"], i["v"], t["rel"], t["a"], state["bounds"][1], 1)
    project("o", t["a"], t["o"])
    do(L.sepia_gpu_sconv(i["conv_o"].handle, i["hist_o"].handle, t["o"].handle, t["oc"].handle, h, taps, 1))
    do(L.sepia_gpu_add(i["x"].handle, t["oc"].handle, t["y"].handle, h))
    return dict(y=t["y"].f32(-1), attn=t["a"].f32(-1), k=i["k"].f32(-1, kv)[case["pos"]:], v=i["v"].f32(-1, kv)[case["pos"]:])


# --------------------------------------------------------------------- work --
def _expert_bytes(case, shared):
    t, s = _moe_types(case), _moe_shapes(case)
    return sum(r * _row_bytes(t[i], c) for i, (r, c) in enumerate(s) if (i >= 3) == shared)


def work(case):
    op = case["op"]
    if op == "matvec":
        r, c, n = case["rows"], case["cols"], case["count"]
        return {"bytes": n * (r * _row_bytes(TYPES[case["type"]], c) + 4 * (r + c)), "flops": 2 * n * r * c}
    if op == "ffn":
        h, i, n = case["hidden"], case["inter"], case["count"]
        one = 2 * i * _row_bytes(TYPES[case["gate"]], h) + h * _row_bytes(TYPES[case["down"]], i)
        return {"bytes": n * (one + 4 * h) + 4 * h, "flops": 6 * n * h * i}
    if op == "moe":
        n, h, i = max(1, case["tokens"]), case["hidden"], case["inter"]
        # experts that n tokens touch, each token taking topk of them
        touched = case["routed"] * (1.0 - (1.0 - case["topk"] / case["routed"]) ** n)
        total, sel = case["routed"] + case["shared"], case["topk"] + case["shared"]
        one = (touched * _expert_bytes(case, False) + case["shared"] * _expert_bytes(case, True) + 4 * total * h +
               4 * case["routed"] + 8 * n * h + 4 * n * (case["topk"] + sel))
        return {"bytes": int(case["layers"] * one), "flops": case["layers"] * n * (6 * sel * h * i + 2 * total * h)}
    tokens = case.get("tokens", 1)
    lo, hi, _ = _bounds(case, tokens)
    heads, kv = case["heads"], case["kv_heads"] * 128
    rows = sum(b - a + 1 for a, b in zip(lo, hi))
    band = sum(min(b - a + 1, case["window"]) for a, b in zip(lo, hi))
    nbytes = 8 * kv * (hi[-1] - lo[0] + 1) + 8 * tokens * heads * 128 + 4 * heads * band
    flops = 4 * rows * heads * 128
    if op == "block":
        shapes = _block_shapes(case).values()
        nbytes += sum(r * _row_bytes(Q8_0, c) for r, c in shapes) + 4 * (2 * case["hidden"] + 8 * kv + 8 * case["hidden"])
        flops += sum(2 * r * c for r, c in shapes)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # About four times the error measured against exact(): f32 sums 2e-7 (matvec), 3e-7 (the FFN), 5e-7 (a MoE
    # layer); attention up to 1.3e-6, where its scores are large; 7e-6 for prefill layers whose formats come from
    # two families, which may carry weights and activations as bf16 pairs (2^-17).
    if case["op"] in ("attn", "block"):
        return {"rel": 5e-6, "max": 5e-4}
    if case["op"] == "moe" and case["tokens"]:
        kinds = {case[k] in ("q2_k", "q3_k", "q4_k") for k in ("gate", "down") + ("s_gate", "s_down") * (case["shared"] > 0)}
        if len(kinds) > 1:
            return {"rel": 3e-5, "max": 1e-3}
    return {"rel": 2e-6, "max": 2e-4}


# -------------------------------------------------------------------- exact --
_TABLES = {}


def _table(name):
    """A codebook of the formats, from the table file they are published in here."""
    if name not in _TABLES:
        root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
        with open(os.path.join(root, "sepia_amd", "csrc", "iq_tables.h")) as f:
            text = f.read()
        body = re.search(r"#define %s \{(.*?)\}" % name, text, re.S).group(1)
        values = [int(v.rstrip("ULul"), 0) for v in re.findall(r"-?\w+", body)]
        entry = {512: 8, 256: 4, 16: 1}[len(values)]
        a = np.array(values, dtype=np.int64 if entry == 1 else np.uint64)
        if entry > 1:
            a = a.view(np.uint8).reshape(-1, 8)[:, :entry].astype(np.int64)
        _TABLES[name] = torch.from_numpy(a).to("cuda")
    return _TABLES[name]


def _signs(index):
    """+-1 for the 8 weights of each 7-bit sign index: the eighth bit makes the count of negative ones even."""
    bits = (index[..., None] >> torch.arange(7, device=index.device)) & 1
    return 1 - 2 * torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)


def _six_bit(s):
    """The eight 6-bit (scale, minimum) pairs of the 12 scale bytes of Q4_K and Q5_K."""
    low, high = s[:, 0:4], s[:, 4:8]
    sc = torch.cat([low & 63, (s[:, 8:12] & 15) | ((low >> 6) << 4)], 1)
    mn = torch.cat([high & 63, (s[:, 8:12] >> 4) | ((high >> 6) << 4)], 1)
    return sc, mn


def _decode(t, raw):
    """Blocks -> f64 weights [blocks, weights of a block]."""
    b = raw.view(-1, BLOCK[t][1])
    n = b.shape[0]
    f16 = lambda off: b[:, off:off + 2].contiguous().view(torch.float16).double()  # noqa: E731
    u = lambda lo, hi: b[:, lo:hi].to(torch.int32)  # noqa: E731
    at = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    if t == Q8_0:
        return f16(0) * b[:, 2:].view(torch.int8).double()
    if t in (Q2_K, Q3_K):
        shifts = at(0, 2, 4, 6).view(1, 1, 4, 1)
        if t == Q2_K:
            q = ((u(16, 80).view(n, 2, 1, 32) >> shifts) & 3).view(n, 16, 16)
            s = u(0, 16)
            return ((f16(80) * (s & 15))[..., None] * q - (f16(82) * (s >> 4))[..., None]).view(n, 256)
        q = (u(32, 96).view(n, 2, 1, 32) >> shifts) & 3
        top = (u(0, 32).view(n, 1, 1, 32) >> at(*range(8)).view(1, 2, 4, 1)) & 1
        s = u(96, 108)
        sc = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1) | \
            (((s[:, 8:12].view(n, 1, 4) >> at(0, 2, 4, 6).view(1, 4, 1)) & 3) << 4).view(n, 16)
        return ((f16(108) * (sc - 32))[..., None] * (q + 4 * top - 4).view(n, 16, 16)).view(n, 256)
    if t in (Q4_K, Q5_K):
        sc, mn = _six_bit(u(4, 16))
        q = u(16, 144) if t == Q4_K else u(48, 176)
        q = ((q.view(n, 4, 1, 32) >> at(0, 4).view(1, 1, 2, 1)) & 15).view(n, 8, 32)
        if t == Q5_K:
            q = q + 16 * ((u(16, 48).view(n, 1, 32) >> at(*range(8)).view(1, 8, 1)) & 1)
        return ((f16(0) * sc)[..., None] * q - (f16(2) * mn)[..., None]).view(n, 256)
    if t == Q6_K:
        low = u(0, 128).view(n, 2, 1, 2, 32) >> at(0, 4).view(1, 1, 2, 1, 1)
        top = (u(128, 192).view(n, 2, 1, 1, 32) >> at(0, 2, 4, 6).view(1, 1, 2, 2, 1)) & 3
        q = ((low & 15) | (top << 4)) - 32
        return ((f16(208) * b[:, 192:208].contiguous().view(torch.int8))[..., None] * q.view(n, 16, 16)).view(n, 256)
    if t == IQ2_XS:
        v = u(2, 66).view(n, 32, 2)
        v = v[..., 0] | (v[..., 1] << 8)
        sc = torch.stack([u(66, 74) & 15, u(66, 74) >> 4], 2).repeat_interleave(2, 2).view(n, 32)
        w = _table("SEPIA_IQ2XS_GRID_INIT")[(v & 511).long()] * _signs(v >> 9)
        return ((f16(0) * (0.5 + sc) * 0.25)[..., None] * w).view(n, 256)
    if t == IQ3_XXS:
        a = u(66, 98).to(torch.int64).view(n, 8, 4)
        a = a[..., 0] | (a[..., 1] << 8) | (a[..., 2] << 16) | (a[..., 3] << 24)
        s = _signs((a[..., None] >> at(0, 7, 14, 21)) & 127).view(n, 8, 32)
        w = _table("SEPIA_IQ3XXS_GRID_INIT")[u(2, 66).long()].view(n, 8, 32) * s
        return ((f16(0) * (0.5 + (a >> 28)) * 0.5)[..., None] * w).view(n, 256)
    sh = u(2, 4)
    sc = ((u(4, 8).view(n, 4, 1) >> at(0, 4)) & 15).view(n, 8) | \
        ((((sh[:, :1] | (sh[:, 1:] << 8)) >> (2 * at(*range(8)))) & 3) << 4)
    q = (u(8, 136).view(n, 8, 1, 16) >> at(0, 4).view(1, 1, 2, 1)) & 15
    return ((f16(0) * (sc - 32))[..., None] * _table("SEPIA_IQ4NL_VALUES_INIT")[q.long()].view(n, 8, 32)).view(n, 256)


def _linear(t, raw, cols, x):
    """x [n, cols] times the quantized rows of raw, in f64, a slab of rows at a time."""
    rb = _row_bytes(t, cols)
    rows = raw.numel() // rb
    step = max(1, (1 << 24) // cols)
    return torch.cat([x @ _decode(t, raw[r * rb:(r + step) * rb]).view(-1, cols).T for r in range(0, rows, step)], 1)


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    op = case["op"]
    if op == "matvec":
        t, n = TYPES[case["type"]], case["rows"] * case["cols"]
        x = _normal(_gen(seed, 1), case["count"], case["cols"]).double()
        return [_linear(t, _raw(_gen(seed, 10 + i), t, n), case["cols"], x[i:i + 1])[0] for i in range(case["count"])]
    if op == "ffn":
        tg, td = TYPES[case["gate"]], TYPES[case["down"]]
        h, i = case["hidden"], case["inter"]
        g, u, d = (_raw(_gen(seed, s), t, case["experts"] * h * i).view(case["experts"], -1)
                   for s, t in ((10, tg), (11, tg), (12, td)))
        x = _normal(_gen(seed, 1), h).double()[None]
        out = []
        for k in range(case["count"]):
            e = (5 * k + 3) % case["experts"]
            out.append(_linear(td, d[e], i, _silu(_linear(tg, g[e], h, x)) * _linear(tg, u[e], h, x))[0])
        return out
    if op == "moe":
        return [_exact_layer(case, seed, layer) for layer in range(case["layers"])]
    if op == "attn":
        a = {k: v.double() for k, v in _attn_inputs(case, seed, case["tokens"]).items()}
        return _exact_attn(case, a["q"], a["k"], a["v"], a["rel"])
    a = {k: v.double() for k, v in _block_inputs(case, seed).items()}
    w = {k: (_raw(_gen(seed, 10 + i), Q8_0, r * c), c) for i, (k, (r, c)) in enumerate(_block_shapes(case).items())}
    project = lambda name, x: _linear(Q8_0, w[name][0], w[name][1], x.view(1, -1))[0]  # noqa: E731
    norm = lambda x, g: g * x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)  # noqa: E731
    conv = lambda x, taps, hist: x + (taps * torch.cat([hist, x[None]]).T).sum(1)  # noqa: E731
    xn = norm(a["x"], a["norm"])
    q = norm(project("q", xn).view(-1, 128), a["q_norm"])
    k = norm(conv(project("k", xn), a["conv_k"], a["hist_k"]).view(-1, 128), a["k_norm"]).view(-1)
    v = conv(project("v", xn), a["conv_v"], a["hist_v"])
    a["k"][case["pos"]], a["v"][case["pos"]] = k, v
    rel = (project("r", xn).view(-1, BLOCK_D_REL) @ a["rel_proj"])[None]
    attn = _exact_attn(case, q[None], a["k"], a["v"], rel)[0]
    y = a["x"] + conv(project("o", attn), a["conv_o"], a["hist_o"])
    return dict(y=y, attn=attn, k=k[None], v=v[None])


def _exact_layer(case, seed, layer):
    router, bias = _router(case, seed, layer)
    x = _tokens(case, seed, layer, router, bias).double()
    nr, k, h, i = case["routed"], case["topk"], case["hidden"], case["inter"]
    logits = x @ router.double().T
    idx = (torch.sigmoid(logits[:, :nr]) + bias.double()).topk(k, dim=1).indices
    picked = torch.cat([logits.gather(1, idx), logits[:, nr:]], 1)
    w = torch.softmax(torch.nn.functional.logsigmoid(picked), 1) * ROUTE_SCALE
    raw, types, shapes = [], _moe_types(case), _moe_shapes(case)
    for j in range(6 if case["shared"] else 3):
        experts, (r, c) = nr if j < 3 else case["shared"], shapes[j]
        raw.append(_raw(_gen(seed, 110 + 10 * layer + j), types[j], experts * r * c).view(experts, -1))
    y = torch.zeros_like(x)
    for e in range(nr + case["shared"]):
        if e < nr:
            token, slot = torch.nonzero(idx == e, as_tuple=True)
        else:
            token, slot = torch.arange(x.shape[0], device="cuda"), torch.full((x.shape[0],), k + e - nr, device="cuda")
        if not token.numel():
            continue
        j, at = (0, e) if e < nr else (3, e - nr)
        hid = _silu(_linear(types[j], raw[j][at], h, x[token])) * _linear(types[j], raw[j + 1][at], h, x[token])
        y.index_add_(0, token, w[token, slot][:, None] * _linear(types[j + 2], raw[j + 2][at], i, hid))
    return dict(y=y, idx=None, w=w.reshape(-1))


def _exact_attn(case, q, k, v, rel):
    tokens, heads, window = q.shape[0], case["heads"], case["window"]
    lo, hi, tau = _bounds(case, tokens)
    n = hi[-1] + 1
    pos = torch.arange(n, device="cuda")[None]
    lo, hi = (torch.tensor(a, device="cuda")[:, None] for a in (lo, hi))
    tau = torch.tensor(tau, dtype=torch.float32, device="cuda").double()[:, None]
    dist = hi - pos
    seen, near = (pos >= lo) & (pos <= hi), (dist >= 0) & (dist < window)
    out = torch.empty(tokens, heads, 128, dtype=torch.float64, device="cuda")
    for head in range(heads):
        at = slice(128 * (head * case["kv_heads"] // heads), 128 * (head * case["kv_heads"] // heads) + 128)
        bias = rel[:, head].gather(1, dist.clamp(0, window - 1)) * tau
        s = q[:, head] @ k[:n, at].T / 128 + torch.where(near, bias, torch.zeros_like(bias))
        out[:, head] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ v[:n, at]
    return out.view(tokens, -1)
