"""Host-side mirror of dfdx's ``TransformerEncoderBlock`` on the Rocm device: one call into the C ABI forward, one backward.

    TransformerEncoderBlock   dfdx/src/nn/layers/transformer.rs:24-48
        = ResidualAdd<MultiHeadAttention>, LayerNorm1D, ResidualAdd<(Linear, ReLU, Linear)>, LayerNorm1D
    MultiHeadAttention        dfdx/src/nn/layers/multi_head_attention.rs:105-146
    Linear / LayerNorm1D / ResidualAdd   linear.rs:82-89, layer_norm1d.rs:87-91, residual_add.rs:38-45

The library strings the block's ops together (``dfdx_rocm_encoder_forward`` / ``_backward``); here live the parameters, the
storage and the names of what the forward keeps.  The forward keeps what the backward needs; the other values of the
reference's tape (the attention probabilities where the fused attention runs, the pre-activation of the ReLU) are made
when somebody asks for them.  Gradients are stored, not added into zeros, so the step pays neither a fill nor the read of
the zeros.
"""
from __future__ import annotations

import ctypes
import math
from typing import Dict, Tuple

from .rocm import DTYPES, ITEMSIZE, Encoder, EncoderLayout, Rocm, View, _row_major

_POINTERS = ctypes.c_void_p * 16

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
        self.gapless = not any(self.pieces[1::2])
        self.grad_views = [(n, s, _row_major(s)) for n, s in self.shapes.items()] + [("x", (B, S, d), _row_major((B, S, d)))]


class _Saved(dict):
    """What the forward keeps, by name: ``x`` and ``out``, and Views into the one allocation ``arena`` made on first use."""

    def __init__(self, block: "EncoderBlock", plan: _Plan, x: View, arena):
        super().__init__(x=x)
        self.block, self.plan, self.arena = block, plan, arena

    def __missing__(self, name):
        value = self[name] = self._make(name)
        return value

    def _make(self, name):
        dev, dtype, l = self.block.dev, self.block.dtype, self.plan.layout
        B, S, d = self["x"].shape
        H, D, ff = self.block.h, d // self.block.h, self.block.ff

        def at(offset, shape, strides=None, kind=dtype):
            n = math.prod(shape) * ITEMSIZE[kind]
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
            return dev.linear_forward(self["n1"], self.block.p["w1"], self.block.p["b1"])
        if name == "scale":
            return 1.0 / math.sqrt(D)
        if l.fused_attention:
            if name == "lse":
                return at(l.lse, (B, H, S), kind="f32")
            if name == "probs":
                return dev.softmax_forward(dev.forward(self["qv"], self["kv"]), self["scale"])
            if name == "tokens":
                return at(l.tok, (B, H, S, D), heads)
        elif name in ("probs", "tokens"):
            return at(getattr(l, name), (B, H, S, S if name == "probs" else D))
        raise KeyError(name)


class EncoderBlock:
    """Parameters are device ``View``s: w* are (out, in) row-major Linear weights, b* biases, g*/be* the LayerNorm
    gamma / beta.  ``deferred_zeros`` is kept for callers that pass it: there are no gradient zeros to fill either way."""

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

    def _desc(self, plan: _Plan) -> Encoder:
        p, desc = self.p, Encoder.from_buffer_copy(plan.desc)
        ptrs = []
        for name, shape in plan.shapes.items():
            v = p[name]
            assert v.shape == shape and v.dtype == self.dtype and v.strides[-1] == 1 and (len(shape) == 1 or v.strides[0] == shape[1]), \
                f"{name}: left: {v.shape}\n right: {shape}"
            ptrs.append(v.ptr)
        desc.params[:] = ptrs
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
        arena = dev._bytes(l.saved_bytes)
        scratch = dev._bytes(l.forward_scratch_bytes) if l.forward_scratch_bytes else None
        dev._check(dev._f.encoder_forward(dev.ctx, ctypes.byref(self._desc(plan)), x.ptr, out.data_ptr(), arena.data_ptr(),
                                          scratch.data_ptr() if scratch is not None else None))
        return View(out, self.dtype, (B, S, d), strides), _Saved(self, plan, x, arena)

    def backward(self, saved: dict, grad_out: View) -> Tuple[Dict[str, View], View]:
        """grad_out: d(loss)/d(out), contiguous like the output.  Returns ({parameter: gradient}, d(loss)/d(x))."""
        dev = self.dev
        plan, x, dtype = saved.plan, saved["x"], self.dtype
        assert grad_out.shape == x.shape and grad_out.strides == x.strides and grad_out.dtype == dtype
        grads = dev._bytes(plan.grad_bytes)
        scratch = dev._bytes(plan.layout.backward_scratch_bytes)
        base, ptrs = grads.data_ptr(), []
        for n in range(0, len(plan.pieces), 2):
            ptrs.append(base)
            base += plan.pieces[n] + plan.pieces[n + 1]
        dev._check(dev._f.encoder_backward(dev.ctx, ctypes.byref(self._desc(plan)), x.ptr, saved.arena.data_ptr(), grad_out.ptr,
                                           _POINTERS(*ptrs[:-1]), ptrs[-1], scratch.data_ptr()))
        parts = grads.split(plan.pieces[::2]) if plan.gapless else grads.split(plan.pieces)[::2]
        views = {name: View(part, dtype, shape, strides) for part, (name, shape, strides) in zip(parts, plan.grad_views)}
        return views, views.pop("x")
