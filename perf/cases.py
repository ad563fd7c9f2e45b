"""The workloads whose speed matters, as a user's program runs them through the public entry points.

Eight families: ``linear`` (a Linear layer, forward and backward), ``rows`` (a Linear layer on the few rows of an
inference step, forward), ``matmul`` (one matrix product), ``broadcast`` (a (B, M, K) activation times a shared (K, N)
matrix, forward and backward), ``attention`` (the rank-4 products of attention with the softmax and the reshape between
them, forward and backward), ``encoder`` (a transformer encoder block, a training step), ``encode`` (the block's forward
alone) and ``conv`` (a convolution layer, forward and backward).

``listed()`` holds the sizes of this repository's own benchmark and tests; ``draw()`` gives others of the same ranges.
Gradient storage is declared zero and not filled, the way ``EncoderBlock`` takes it (``zeros_many(..., deferred=True)``).
"""
from __future__ import annotations

import math

import torch

from dfdx_amd import EncoderBlock, Rocm, View
from dfdx_amd.encoder import PARAMS

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "f64": torch.float64}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "f64": 8}


def listed():
    return [
        # The smallest call in earnest: a small network's Linear layer on a batch of 64.  Launches and host time count.
        {"name": "linear_64x512x256_f32", "kind": "linear", "rows": 64, "inp": 512, "out": 256, "dtype": "f32"},
        # One token through a 4096-wide Linear: the matrix is read once, its bytes are the bound.
        {"name": "rows_1x4096x4096_f16", "kind": "rows", "rows": 1, "inp": 4096, "out": 4096, "dtype": "f16"},
        # A language model's output layer, vocabulary of 50257: every matrix but one has an odd extent.
        {"name": "linear_2048x1024x50257_f16", "kind": "linear", "rows": 2048, "inp": 1024, "out": 50257, "dtype": "f16"},
        # The large square product, in the half type and in the library's default type with a transposed right operand.
        {"name": "matmul_4096_f16", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "ta": False, "tb": False, "dtype": "f16"},
        {"name": "matmul_4096_f32_nt", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "ta": False, "tb": True, "dtype": "f32"},
        # A (batch, seq, hidden) activation times one matrix.
        {"name": "broadcast_32x512x1024_f16", "kind": "broadcast", "batch": 32, "m": 512, "k": 1024, "n": 1024, "dtype": "f16"},
        # Attention written out as its ops: 8 sequences of 1024 tokens, 16 heads of 64.
        {"name": "attention_8x16x1024x64_f16", "kind": "attention", "batch": 8, "heads": 16, "seq": 1024, "dim": 64, "dtype": "f16"},
        # A training step of a transformer encoder block.
        {"name": "encoder_16x512x1024_bf16", "kind": "encoder", "batch": 16, "seq": 512, "d": 1024, "heads": 16, "ff": 4096, "dtype": "bf16"},
        # The same of a small block, where the many launches count.
        {"name": "encoder_4x100x256_bf16", "kind": "encoder", "batch": 4, "seq": 100, "d": 256, "heads": 4, "ff": 1024, "dtype": "bf16"},
        # Inference on images cut into 196 patches and a class token: the odd sequence length of vision transformers.
        {"name": "encode_16x197x768_f16", "kind": "encode", "batch": 16, "seq": 197, "d": 768, "heads": 12, "ff": 3072, "dtype": "f16"},
        # A residual network's 3 x 3 layer, and its first layer (few channels, large filter, strided).
        {"name": "conv_64x64x56_k3_f16", "kind": "conv", "batch": 64, "cin": 64, "cout": 64, "hw": 56, "k": 3, "stride": 1, "groups": 1, "dtype": "f16"},
        {"name": "conv_64x3x224_k7s2_f16", "kind": "conv", "batch": 64, "cin": 3, "cout": 64, "hw": 224, "k": 7, "stride": 2, "groups": 1, "dtype": "f16"},
    ]


def _log(rng, lo, hi):
    """A whole number, spread over the logarithm of [lo, hi]; half of them multiples of 64 (of 8 below 256), the rest as they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        g = 64 if v >= 256 else 8
        v = max(g, v // g * g)
    return min(max(v, lo), hi)


def _draw(rng):
    kind = rng.choice(("linear", "rows", "matmul", "broadcast", "attention", "encoder", "encode", "conv"))
    half = rng.choice(("f16", "bf16"))
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 16, 16384), "inp": _log(rng, 16, 4096), "out": _log(rng, 10, 50257), "dtype": rng.choice((half, half, "f32"))}
    if kind == "rows":
        return {"kind": kind, "rows": _log(rng, 1, 16), "inp": _log(rng, 512, 16384), "out": _log(rng, 512, 16384), "dtype": rng.choice((half, half, "f32"))}
    if kind == "matmul":
        c = {"kind": kind, "m": _log(rng, 64, 8192), "k": _log(rng, 64, 8192), "n": _log(rng, 64, 8192), "ta": rng.random() < 0.5, "tb": rng.random() < 0.5,
             "dtype": rng.choice((half, half, half, "f32", "f32", "f64"))}
        if c["ta"] and c["tb"]:
            c["ta"] = False
        return c
    if kind == "broadcast":
        return {"kind": kind, "batch": _log(rng, 2, 64), "m": _log(rng, 16, 1024), "k": _log(rng, 64, 4096), "n": _log(rng, 64, 4096), "dtype": rng.choice((half, half, "f32"))}
    if kind == "attention":
        return {"kind": kind, "batch": rng.randint(1, 16), "heads": rng.randint(2, 16), "seq": _log(rng, 32, 1024), "dim": rng.choice((32, 64, 64, 64, 80, 128)),
                "dtype": rng.choice((half, half, half, "f32"))}
    if kind in ("encoder", "encode"):
        dim = rng.choice((32, 64, 64, 64, 128))
        d = dim * rng.choice((4, 6, 8, 12, 16) if dim < 128 else (4, 6, 8))
        c = {"kind": kind, "batch": _log(rng, 1, 32), "seq": _log(rng, 16, 1024), "d": d, "heads": d // dim, "ff": 4 * d, "dtype": rng.choice((half, half, half, "f32"))}
        if kind == "encoder":
            # A step's gradients are compared: on few tokens, and in bf16, one pre-activation that rounds to the other side
            # of a ReLU is more than any tolerance can tell from a mistake (bf16 is in the listed cases and the other families).
            c["batch"] = max(c["batch"], -(-512 // c["seq"]))
            if c["dtype"] == "bf16":
                c["dtype"] = "f16"
        return c
    k, stride = rng.choice(((1, 1), (3, 1), (3, 1), (3, 1), (3, 2), (1, 2), (5, 1), (7, 2)))
    hw = rng.choice((7, 14, 28, 32, 56, 56, 64, 96, 112, 224))
    cin, cout = (rng.choice((16, 32, 64, 64, 96, 128, 192, 256, 512)) for _ in range(2))
    if k == 7 or hw == 224:
        cin, cout = 3, min(cout, 64)
    groups = cin if k == 3 and rng.random() < 0.15 else 1
    return {"kind": kind, "batch": _log(rng, 1, 64), "cin": cin, "cout": cin if groups > 1 else cout, "hw": hw, "k": k, "stride": stride, "groups": groups,
            "dtype": rng.choice((half, half, "f32"))}


def draw(rng):
    """One case more; one that would take more than the largest listed ones (by operations at the type's rate, or by bytes) is drawn again."""
    while True:
        c = _draw(rng)
        w = work(c)
        rate = {"f32": 140e12, "f64": 50e12}.get(c["dtype"], 1000e12)
        moved = w["bytes"]
        if c["kind"] in ("attention", "encoder", "encode"):
            moved += 8 * c["batch"] * c["heads"] * c["seq"] ** 2 * BYTES[c["dtype"]]
        if c["kind"] == "conv":
            moved += 2 * c["k"] ** 2 * c["batch"] * c["cin"] * (c["hw"] // c["stride"]) ** 2 * BYTES[c["dtype"]]
        if w["flops"] / rate < 0.6e-3 and moved < 2.2e9:
            return c


def _conv_out(c):
    pad = c["k"] // 2
    return (c["hw"] + 2 * pad - c["k"]) // c["stride"] + 1


def work(c):
    kind, es = c["kind"], BYTES[c["dtype"]]
    if kind == "linear":      # in: x, W, b, dy; out: y, dx, dW, db
        r, i, o = c["rows"], c["inp"], c["out"]
        return {"bytes": 2 * es * (r * i + i * o + o + r * o), "flops": 6 * r * i * o}
    if kind == "rows":
        r, i, o = c["rows"], c["inp"], c["out"]
        return {"bytes": es * (r * i + i * o + o + r * o), "flops": 2 * r * i * o}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": es * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "broadcast":
        r, k, n = c["batch"] * c["m"], c["k"], c["n"]
        return {"bytes": 2 * es * (r * k + k * n + r * n), "flops": 6 * r * k * n}
    if kind == "attention":   # in: q, k, v, dy; out: probabilities (which the backward op takes from the caller), y, dq, dk, dv
        bh, s, d = c["batch"] * c["heads"], c["seq"], c["dim"]
        return {"bytes": es * bh * (8 * s * d + s * s), "flops": 12 * bh * s * s * d}
    if kind in ("encoder", "encode"):
        t, d, ff, s = c["batch"] * c["seq"], c["d"], c["ff"], c["seq"]
        fwd = 2 * t * d * (4 * d + 2 * ff) + 4 * t * s * d
        par = 4 * d * d + 2 * d * ff + 9 * d + ff
        if kind == "encode":
            return {"bytes": es * (2 * t * d + par), "flops": fwd}
        return {"bytes": es * (4 * t * d + 2 * par), "flops": 3 * fwd}
    oh = _conv_out(c)         # in: image, filters, dy; out: y, dimage, dfilters
    img, out = c["batch"] * c["cin"] * c["hw"] ** 2, c["batch"] * c["cout"] * oh * oh
    fil = c["cout"] * (c["cin"] // c["groups"]) * c["k"] ** 2
    return {"bytes": 2 * es * (img + fil + out), "flops": 6 * out * (c["cin"] // c["groups"]) * c["k"] ** 2}


def tolerance(c):
    """About four times the distance from the same path in 64 bits, for the largest of a case's outputs."""
    if c["dtype"] == "f64":
        return {"rel": 1e-13}
    kind = c["kind"]
    # Behind a ReLU a gradient moves by a whole term wherever a pre-activation rounds across zero: its distance is the
    # square root of the share of such values (3.9 % measured in bf16, 0.004 % in f32; 3 % is stated).
    if c["dtype"] == "f32":
        return {"rel": 2e-4, "max": 0.05} if kind == "encoder" else {"rel": 5e-6}   # 1.1e-6 measured over 4096 terms
    # One rounding to the half type per result, 2^-9 (bf16) or 2^-12 (f16) of a value at most: 0.43 eps measured.  The
    # chains add the roundings of what they hand on: 1.3 eps through attention, 0.95 eps through the block's forward.
    eps = 2.0 ** -8 if c["dtype"] == "bf16" else 2.0 ** -11
    if kind == "encoder":
        return {"rel": 0.03, "max": 0.99}
    if kind == "attention":
        return {"rel": 5 * eps, "max": 60 * eps}
    if kind == "encode":
        return {"rel": 4 * eps, "max": 20 * eps}
    return {"rel": 2 * eps, "max": 12 * eps}


_dev = None


def _device():
    global _dev
    if _dev is None:
        _dev = Rocm(0)
    return _dev


def _view(t, dtype):
    return View(t.view(torch.uint8).reshape(-1), dtype, tuple(t.shape), tuple(t.stride()))


def _flat(dtype, *views):
    """The results' storages as flat tensors of their element type."""
    return [v.storage.view(TORCH[dtype]) for v in views]


def prepare(case, seed):
    dev, dt = _device(), case["dtype"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape, scale=1.0):
        return _view((torch.randn(*shape, device="cuda", generator=gen, dtype=torch.float32) * scale).to(TORCH[dt]), dt)

    def uni(*shape, bound):
        return _view(((torch.rand(*shape, device="cuda", generator=gen, dtype=torch.float32) * 2 - 1) * bound).to(TORCH[dt]), dt)

    kind = case["kind"]
    st = {"case": case, "dev": dev}
    if kind in ("linear", "rows"):   # x ~ N(0, 1), Kaiming-uniform weight and bias
        r, i, o = case["rows"], case["inp"], case["out"]
        st.update(x=rnd(r, i), w=uni(o, i, bound=i ** -0.5), b=uni(o, bound=i ** -0.5))
        if kind == "linear":
            st["g"] = rnd(r, o)
    elif kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        a = uni(k, m, bound=1.0).permute(1, 0) if case["ta"] else uni(m, k, bound=1.0)
        b = uni(n, k, bound=1.0).permute(1, 0) if case["tb"] else uni(k, n, bound=1.0)
        st.update(a=a, b=b)
    elif kind == "broadcast":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        st.update(a=rnd(b, m, k), b=rnd(k, n, scale=k ** -0.5), g=rnd(b, m, n))
    elif kind == "attention":
        b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
        st.update(q=rnd(b, h, s, d), k=rnd(b, h, s, d), v=rnd(b, h, s, d), g=rnd(b, s, h * d), scale=d ** -0.5)
    elif kind in ("encoder", "encode"):
        d, ff = case["d"], case["ff"]
        p = {n: rnd(*shape, scale=0.02) for n, shape in (("wq", (d, d)), ("wk", (d, d)), ("wv", (d, d)), ("wo", (d, d)), ("w1", (ff, d)), ("w2", (d, ff)))}
        p.update({n: rnd(size, scale=0.02) for n, size in (("bq", d), ("bk", d), ("bv", d), ("bo", d), ("b1", ff), ("b2", d))})
        for n in ("g1", "g2"):
            p[n] = _view(torch.ones(d, device="cuda", dtype=TORCH[dt]), dt)
        for n in ("be1", "be2"):
            p[n] = _view(torch.zeros(d, device="cuda", dtype=TORCH[dt]), dt)
        st.update(x=rnd(case["batch"], case["seq"], d), block=EncoderBlock(dev, dt, d, case["heads"], ff, p))
        if kind == "encoder":
            st["g"] = rnd(case["batch"], case["seq"], d)
    else:
        cin, cout, k, hw = case["cin"], case["cout"], case["k"], case["hw"]
        fan = cin // case["groups"] * k * k
        st.update(img=rnd(case["batch"], cin, hw, hw), fil=rnd(cout, cin // case["groups"], k, k, scale=fan ** -0.5), g=rnd(case["batch"], cout, _conv_out(case), _conv_out(case)))
    return st


def run(st):
    case, dev = st["case"], st["dev"]
    kind, dt = case["kind"], case["dtype"]
    if kind == "rows":
        return _flat(dt, dev.linear_forward(st["x"], st["w"], st["b"]))
    if kind == "linear":
        x, w, b = st["x"], st["w"], st["b"]
        y = dev.linear_forward(x, w, b)
        gx, gw, gb = dev.zeros_many([x, w, b], deferred=True)
        dev.linear_backward(x, gx, w, gw, gb, st["g"])
        dev.settle_zeros()
        return _flat(dt, y, gx, gw, gb)
    if kind == "matmul":
        return _flat(dt, dev.forward(st["a"], st["b"]))
    if kind == "broadcast":
        a, b = st["a"], st["b"]
        y = dev.forward(a, b)
        ga, gb = dev.zeros_many([a, b], deferred=True)
        dev.backward(a, ga, b, gb, st["g"])
        dev.settle_zeros()
        return _flat(dt, y, ga, gb)
    if kind == "attention":
        q, k, v, g = st["q"], st["k"], st["v"], st["g"]
        kt = k.permute(0, 1, 3, 2)
        scores = dev.forward(q, kt)
        probs = dev.softmax_forward(scores, st["scale"])
        tokens = dev.forward(probs, v)
        heads = tokens.permute(0, 2, 1, 3)
        y = dev.reshape_forward(heads, g.shape)
        gt, gp, gs, gq, gk, gv = dev.zeros_many([tokens, probs, scores, q, k, v], deferred=True)
        dev.reshape_backward(heads, gt, g)
        dev.backward(probs, gp, v, gv, gt)
        dev.softmax_backward(probs, gs, gp, st["scale"])
        dev.backward(q, gq, kt, gk, gs)
        dev.settle_zeros()
        return _flat(dt, probs, y, gq, gk, gv)
    if kind == "encode":
        return _flat(dt, st["block"].forward(st["x"])[0])
    if kind == "encoder":
        y, saved = st["block"].forward(st["x"])
        grads, gx = st["block"].backward(saved, st["g"])
        # the key bias has no gradient (it shifts all scores of a row alike): what is computed for it is the rounding of zero
        return _flat(dt, y, gx, *[grads[n] for n in PARAMS if n != "bk"])
    img, fil = st["img"], st["fil"]
    how = dict(stride=case["stride"], padding=case["k"] // 2, groups=case["groups"])
    y = dev.conv2d_forward(img, fil, **how)
    gi, gf = dev.zeros_many([img, fil], deferred=True)
    dev.conv2d_backward(img, gi, fil, gf, st["g"], **how)
    dev.settle_zeros()
    return _flat(dt, y, gi, gf)
