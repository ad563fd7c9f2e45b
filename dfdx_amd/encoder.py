"""Host-side mirror of dfdx's ``TransformerEncoderBlock`` on the Rocm device: one call into the C ABI forward, one backward.

    TransformerEncoderBlock   dfdx/src/nn/layers/transformer.rs:24-48
        = ResidualAdd<MultiHeadAttention>, LayerNorm1D, ResidualAdd<(Linear, ReLU, Linear)>, LayerNorm1D
    MultiHeadAttention        dfdx/src/nn/layers/multi_head_attention.rs:105-146
    Linear / LayerNorm1D / ResidualAdd   linear.rs:82-89, layer_norm1d.rs:87-91, residual_add.rs:38-45

The library strings the block's ops together (``dfdx_rocm_encoder_forward`` / ``_backward``); here live the parameters, the
storage and the names of what the forward keeps.  The forward keeps what the backward needs; the other values of the
reference's tape (the attention probabilities where the fused attention runs, the pre-activation of the ReLU) are made
when somebody asks for them.  Gradients are stored, not added into zeros, so the step pays neither a fill nor the read of
the zeros.  A backward from other values than the forward's own goes op by op.
"""
from __future__ import annotations

import ctypes
import math
from collections.abc import ItemsView, KeysView, ValuesView
from typing import Dict, Tuple

from .rocm import DTYPES, ITEMSIZE, Encoder, EncoderLayout, Rocm, View, _row_major

PARAMS = ("wq", "bq", "wk", "bk", "wv", "bv", "wo", "bo", "g1", "be1", "w1", "b1", "w2", "b2", "g2", "be2")


class _Plan:
    """What one (batch, seq) shape of a block needs to know: sizes and places, no data."""

    def __init__(self, block: "EncoderBlock", B: int, S: int):
        d, H, ff = block.d, block.h, block.ff
        self.desc = Encoder(DTYPES[block.dtype], 0, B, S, d, H, ff)
        self.layout = EncoderLayout()
        dev = block.dev
        dev._check(dev.lib.dfdx_rocm_encoder_plan(dev.ctx, ctypes.byref(self.desc), ctypes.byref(self.layout)))
        self.shapes = {"wq": (d, d), "wk": (d, d), "wv": (d, d), "wo": (d, d), "w1": (ff, d), "w2": (d, ff), "b1": (ff,)}
        self.shapes = {n: self.shapes.get(n, (d,)) for n in PARAMS}
        # gradients: one allocation, the pieces in the order of PARAMS, then that of x, on 16-byte boundaries
        es = ITEMSIZE[block.dtype]
        self.pieces = []
        for shape in list(self.shapes.values()) + [(B, S, d)]:
            n = math.prod(shape) * es or 16   # (an empty batch's gradient has an address all the same)
            self.pieces += [n, -n % 16]
        self.grad_bytes = sum(self.pieces)
        self.params = tuple((n, s, _row_major(s)) for n, s in self.shapes.items())
        self.offsets = tuple(sum(self.pieces[:n]) for n in range(0, len(self.pieces), 2))
        self.grad_views = tuple((n, at, size, s, strides) for (n, s, strides), at, size in
                                zip(self.params + (("x", (B, S, d), (S * d, d, 1)),), self.offsets, self.pieces[::2]))
        self.raw = bytes(self.desc)


KEPT = ("x", "qv", "kv", "vv", "probs", "tokens", "tok", "h1", "n1", "f1", "r1", "h2", "scale", "folded")


def _version(storage):
    """torch's count of changes in place (``None`` where it keeps none)."""
    try:
        return storage._version
    except RuntimeError:   # an inference tensor
        return None


class _Saved(dict):
    """What the forward keeps, by name (``KEPT``; ``lse`` too where the fused attention ran): a dict whose values are made when somebody
    asks for them, most of them Views into the one allocation ``arena``.  ``backward`` takes it as it is, or with values replaced or
    changed, or any dict with the same names."""

    __slots__ = ("made", "block", "plan", "arena", "version", "versions", "behind_f1")

    def __init__(self, block: "EncoderBlock", plan: _Plan, x: View, arena):
        self.made = {"x": x}
        super().__init__(self.made)
        self.block, self.plan, self.arena = block, plan, arena
        self.version = _version(arena)   # its contents stand for what the forward left, and those of `versions`
        self.versions = {}
        w1, b1 = block.p["w1"], block.p["b1"]
        self.behind_f1 = w1, _version(w1.storage), b1, _version(b1.storage)

    def __missing__(self, name):
        value = self._make(name)
        self.made[name] = self[name] = value
        if name in ("probs", "f1"):   # (made from what the forward left: changing them changes nothing that it left)
            self.versions[name] = value.storage, _version(value.storage)
        return value

    def untouched(self) -> bool:
        """Whether the names still stand for what the forward left."""
        if _version(self.arena) != self.version:
            return False
        made = self.made
        if len(made) == dict.__len__(self) == 1:   # (x, which nobody has asked about)
            return dict.get(self, "x") is made["x"]
        return all(dict.get(self, n, v) is v for n, v in made.items()) and all(n in made for n in dict.keys(self) if n in KEPT) and \
            all(_version(storage) == v for storage, v in self.versions.values())

    def _make(self, name):
        dev, dtype, l = self.block.dev, self.block.dtype, self.plan.layout
        B, S, d = self.made["x"].shape
        H = self.plan.desc.heads
        D, ff = d // H, self.plan.desc.d_ff

        def at(offset, shape, strides=None, kind=dtype):
            n = max(math.prod(shape) * ITEMSIZE[kind], 16)
            return View(self.arena[offset:offset + n], kind, shape, strides or _row_major(shape))

        heads = (S * d, D, d, 1)
        if name in ("qv", "vv"):                     # (B, H, S, D), head-interleaved strides
            return at(l.q if name == "qv" else l.v, (B, H, S, D), heads)
        if name == "kv":                             # (B, H, D, S)
            return at(l.k, (B, H, D, S), (S * d, D, 1, d))
        if name in ("tok", "h1", "n1", "h2"):
            return at(getattr(l, name), (B, S, d))
        if name == "r1":
            return at(l.r1, (B, S, ff))
        if name == "f1":
            w1, b1 = self.block.p["w1"], self.block.p["b1"]
            at_w1, version_w1, at_b1, version_b1 = self.behind_f1
            if w1 is not at_w1 or b1 is not at_b1 or (_version(w1.storage), _version(b1.storage)) != (version_w1, version_b1):
                raise RuntimeError("f1 is formed on request, from w1 and b1: they have changed since the forward")
            return dev.linear_forward(self["n1"], self.block.p["w1"], self.block.p["b1"])
        if name == "scale":
            return 1.0 / math.sqrt(D)
        if name == "folded":
            return _folded(dtype, D)
        if l.fused_attention:
            if name == "lse":
                return at(l.lse, (B, H, S), kind="f32")
            if name == "probs":
                return dev.softmax_forward(dev.forward(self["qv"], self["kv"]), self["scale"])
            if name == "tokens":
                return dev.reshape_forward(at(l.tok, (B, H, S, D), heads), (B, H, S, D))
        elif name in ("probs", "tokens"):
            return at(getattr(l, name), (B, H, S, S if name == "probs" else D))
        raise KeyError(name)

    # the names are there whether or not their values have been made
    def __contains__(self, name):
        return name in KEPT or dict.__contains__(self, name)

    def __iter__(self):
        yield from KEPT
        yield from [n for n in dict.keys(self) if n not in KEPT]

    def __len__(self):
        return len(list(iter(self)))

    def get(self, name, default=None):
        return self[name] if name in self else default

    def keys(self):
        return KeysView(self)

    def values(self):
        return ValuesView(self)

    def items(self):
        return ItemsView(self)

    def copy(self):
        return dict(self)

    __copy__ = copy


def _folded(dtype: str, head_dim: int) -> bool:
    """Whether the softmax entry, which takes its scale as a C float, may scale: not for an f64 block whose 1/sqrt(head dim) has no
    exact float value, which multiplies by the double scalar in an op of its own, as the reference does
    (multi_head_attention.rs:133-134)."""
    scale = 1.0 / math.sqrt(head_dim)
    return dtype != "f64" or ctypes.c_float(scale).value == scale


class EncoderBlock:
    """Parameters are device ``View``s: w* are (out, in) row-major Linear weights, b* biases, g*/be* the LayerNorm
    gamma / beta.  ``deferred_zeros``: where the backward adds into zeros (``_backward_by_ops``), whether they are declared or filled."""

    def __init__(self, dev: Rocm, dtype: str, d_model: int, heads: int, d_ff: int, params: Dict[str, View],
                 deferred_zeros: bool = True):
        assert d_model % heads == 0, f"left: {d_model % heads}\n right: 0"
        missing = [n for n in PARAMS if n not in params]
        assert not missing, f"missing parameters: {missing}"
        self.dev, self.dtype, self.d, self.h, self.ff, self.p = dev, dtype, d_model, heads, d_ff, params
        self.deferred_zeros = deferred_zeros
        self._plans: Dict[tuple, _Plan] = {}

    def _plan(self, B: int, S: int) -> _Plan:
        plan = self._plans.get((B, S))
        if plan is None:
            if len(self._plans) >= 64:   # shapes come and go: keep no more than a loader's buckets
                self._plans.clear()
            plan = self._plans[(B, S)] = _Plan(self, B, S)
        return plan

    def _desc(self, plan: _Plan) -> bytes:
        desc = self.dev._f.parameters(plan.raw, self.p, self.dtype, plan.params)
        if desc is None:   # (not of that type and shape, or with strides that are no tuple)
            ptrs = []
            for name, shape, strides in plan.params:
                v = self.p[name]
                assert v.shape == shape and v.dtype == self.dtype and tuple(v.strides) == strides, f"{name}: left: {v.shape}\n right: {shape}"
                ptrs.append(v.ptr)
            desc = Encoder.from_buffer_copy(plan.raw)
            desc.params[:] = ptrs
            desc = bytes(desc)
        return desc

    def forward(self, x: View) -> Tuple[View, dict]:
        """x: (batch, seq, d_model) contiguous.  Returns the block's output and the tensors the backward needs."""
        dev = self.dev
        B, S, d = x.shape
        assert d == self.d, f"left: {d}\n right: {self.d}"
        strides = (S * d, d, 1)
        assert x.strides == strides and x.dtype == self.dtype, "encoder input must be contiguous"
        plan = self._plan(B, S)
        l = plan.layout
        out = dev._bytes(max(B * S * d * ITEMSIZE[self.dtype], 16))
        arena = dev._bytes(max(l.saved_bytes, 16))
        scratch = dev._bytes(l.forward_scratch_bytes) if l.forward_scratch_bytes else None
        dev._check(dev._f.encoder_forward(dev._at, self._desc(plan), x, out.data_ptr(), arena.data_ptr(),
                                          scratch.data_ptr() if scratch is not None else None))
        return View(out, self.dtype, (B, S, d), strides), _Saved(self, plan, x, arena)

    def backward(self, saved: dict, grad_out: View) -> Tuple[Dict[str, View], View]:
        """grad_out: d(loss)/d(out), contiguous like the output.  Returns ({parameter: gradient}, d(loss)/d(x)).  ``saved``: what the
        forward returned, or a dict of the same names."""
        if not (isinstance(saved, _Saved) and saved.untouched()):
            return self._backward_by_ops(saved, grad_out)
        dev = self.dev
        plan, x, dtype = saved.plan, saved.made["x"], self.dtype
        assert grad_out.shape == x.shape and grad_out.strides == x.strides and grad_out.dtype == dtype
        grads = dev._bytes(plan.grad_bytes)
        scratch = dev._bytes(plan.layout.backward_scratch_bytes)
        base = grads.data_ptr()
        ptrs = tuple([base + at for at in plan.offsets])
        dev._check(dev._f.encoder_backward(dev._at, self._desc(plan), x, saved.arena.data_ptr(), grad_out, ptrs[:-1], ptrs[-1], scratch.data_ptr()))
        views = dev._f.pieces(View, grads, dtype, plan.grad_views)
        return views, views.pop("x")

    def _backward_by_ops(self, s: dict, grad_out: View) -> Tuple[Dict[str, View], View]:
        """The same, op by op from the values in ``s``: what the caller has put in the place of the forward's own."""
        dev, p, dtype = self.dev, self.p, self.dtype
        x, n1, tok, probs, qv, kv, vv, r1 = (s[n] for n in ("x", "n1", "tok", "probs", "qv", "kv", "vv", "r1"))
        B, H, S, D = qv.shape
        f1 = r1 if isinstance(s, _Saved) and "f1" not in s.made and not dict.__contains__(s, "f1") else s["f1"]   # (positive in the same places)
        tokens = View(tok.storage, dtype, (B, H, S, D), _row_major((B, H, S, D)))   # (its shape is all that counts)
        # every gradient buffer of the pass: one allocation, pieces aligned to 256 B, zero by declaration (or one fill)
        acts = dict(gh2=s["h2"], gf2=s["h2"], gn1=n1, gr1=r1, gf1=r1, gh1=s["h1"], gattn=s["h1"], gx=x, gtok=tok, gtokens=tokens, gp=probs,
                    gscores=probs, gq=x, gk=x, gv=x)   # gq, gk, gv: laid out like the q, k, v storages
        if not s["folded"]:
            acts["gscaled"] = probs   # gradient of the scaled scores, between the softmax and the scalar multiply
        bufs = dev.zeros_many([p[n] for n in PARAMS] + list(acts.values()), deferred=self.deferred_zeros)
        grads = dict(zip(PARAMS, bufs[:len(PARAMS)]))
        g = dict(zip(acts, bufs[len(PARAMS):]))
        try:
            dev.layer_norm_backward(s["h2"], p["g2"], g["gh2"], grads["g2"], grads["be2"], grad_out)
            dev.add_backward(g["gf2"], g["gn1"], g["gh2"])            # h2 = f2 + n1
            dev.linear_backward(r1, g["gr1"], p["w2"], grads["w2"], grads["b2"], g["gf2"])
            dev.relu_backward(f1, g["gf1"], g["gr1"])
            dev.linear_backward(n1, g["gn1"], p["w1"], grads["w1"], grads["b1"], g["gf1"])
            dev.layer_norm_backward(s["h1"], p["g1"], g["gh1"], grads["g1"], grads["be1"], g["gn1"])
            dev.add_backward(g["gattn"], g["gx"], g["gh1"])           # h1 = attn + x
            dev.linear_backward(tok, g["gtok"], p["wo"], grads["wo"], grads["bo"], g["gattn"])
            dev.reshape_backward(tokens.permute(0, 2, 1, 3), g["gtokens"], g["gtok"])
            dev.backward(probs, g["gp"], vv, g["gv"], g["gtokens"])
            if s["folded"]:
                dev.softmax_backward(probs, g["gscores"], g["gp"], s["scale"])
            else:
                dev.softmax_backward(probs, g["gscaled"], g["gp"], 1.0)
                dev.scalar_mul_backward(s["scale"], g["gscores"], g["gscaled"])
            dev.backward(qv, g["gq"], kv, g["gk"], g["gscores"])
            for w, b, gg in (("wq", "bq", "gq"), ("wk", "bk", "gk"), ("wv", "bv", "gv")):   # x feeds three Linears: one buffer
                dev.linear_backward(x, g["gx"], p[w], grads[w], grads[b], g[gg])
            dev.settle_zeros()   # nothing is left pending in this block; a gradient no op touched would be filled here
        except BaseException:
            # an op refused or raised in mid-pass: no declaration may outlive the pass unsettled, whoever still holds
            # a View of the arena (the caller sees the exception, not zeros it could rely on)
            if bufs[0].owner is not None:
                bufs[0].owner.forget()
            raise
        return grads, g["gx"]
