"""``Rocm``: the host-side mirror of a dfdx device for the matmul path.

Method names and argument meaning follow the reference's kernel traits
(dfdx-core/src/tensor_ops/matmul/mod.rs:116-131,197-212,234-249,273-288):
``forward(lhs, rhs) -> out`` allocates a fresh contiguous output, and
``backward(lhs, grad_lhs, rhs, grad_rhs, grad_out)`` accumulates into gradient
buffers that are laid out like the operands' physical storage.  A tensor is a
:class:`View`: device storage + shape + strides in elements, which is what a
dfdx ``Tensor`` hands its kernels (tensor_impls.rs:32-39).  Shape mismatches
raise ``AssertionError`` before any kernel runs, like the reference's
``assert_eq!`` (mod.rs:192,229,267-268,306-308).

PyTorch is used for device memory only (allocation, host<->device copies).
"""
from __future__ import annotations

import ctypes
import math
import os
import struct
from dataclasses import dataclass
from typing import Optional

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))

DTYPES = {"f32": 0, "f16": 1, "bf16": 2, "f64": 3}
ITEMSIZE = {"f32": 4, "f16": 2, "bf16": 2, "f64": 8}
NP_DTYPES = {"f32": np.float32, "f16": np.float16, "bf16": np.uint16, "f64": np.float64}

KERNEL_AUTO, KERNEL_GENERIC, KERNEL_MFMA, KERNEL_GEMV = 0, 1, 2, 3
ZERO_DEFERRED = 2   # dfdx_rocm_alloc: zero as far as the library can tell, fill only if needed
NOALLOC_SCRATCH_BYTES = 32 << 20   # DFDX_ROCM_NOALLOC_SCRATCH_BYTES
ERR_ALIASED_OUTPUT, ERR_SCRATCH_TOO_SMALL = -4, -5


class RocmError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"dfdx_rocm error {code}: {msg}")
        self.code = code


class GemmDesc(ctypes.Structure):
    """``dfdx_rocm_gemm_desc`` (include/dfdx_rocm.h)."""
    _fields_ = [
        ("dtype", ctypes.c_int32), ("accumulate", ctypes.c_int32),
        ("m", ctypes.c_int64), ("n", ctypes.c_int64), ("k", ctypes.c_int64),
        ("batch1", ctypes.c_int64), ("batch2", ctypes.c_int64),
        ("a", ctypes.c_void_p), ("a_rs", ctypes.c_int64), ("a_cs", ctypes.c_int64),
        ("a_b1", ctypes.c_int64), ("a_b2", ctypes.c_int64),
        ("b", ctypes.c_void_p), ("b_rs", ctypes.c_int64), ("b_cs", ctypes.c_int64),
        ("b_b1", ctypes.c_int64), ("b_b2", ctypes.c_int64),
        ("c", ctypes.c_void_p), ("c_rs", ctypes.c_int64), ("c_cs", ctypes.c_int64),
        ("c_b1", ctypes.c_int64), ("c_b2", ctypes.c_int64),
        ("bias", ctypes.c_void_p),
        ("reduce_batch", ctypes.c_int32), ("kernel", ctypes.c_int32),
        ("variant", ctypes.c_int32), ("flags", ctypes.c_int32),
    ]


class Conv2DOp(ctypes.Structure):
    """Mirrors ``dfdx_rocm_conv2d_op`` == the reference's ``Conv2DOp`` (conv2d/mod.rs:14-29)."""
    _fields_ = [(n, ctypes.c_size_t) for n in ("kernel", "stride", "padding", "dilation", "groups", "batch",
                                               "chan_in", "chan_out", "h_in", "h_out", "w_in", "w_out")]


ENCODER_PARAMS = 16   # DFDX_ROCM_ENCODER_PARAMS


class Encoder(ctypes.Structure):
    """``dfdx_rocm_encoder`` (include/dfdx_rocm.h)."""
    _fields_ = [("dtype", ctypes.c_int32), ("reserved", ctypes.c_int32), ("batch", ctypes.c_int64), ("seq", ctypes.c_int64),
                ("d_model", ctypes.c_int64), ("heads", ctypes.c_int64), ("d_ff", ctypes.c_int64),
                ("params", ctypes.c_void_p * ENCODER_PARAMS)]


class EncoderLayout(ctypes.Structure):
    """``dfdx_rocm_encoder_layout``."""
    _fields_ = [(n, ctypes.c_size_t) for n in ("saved_bytes", "forward_scratch_bytes", "backward_scratch_bytes", "q", "k", "v", "tok",
                                               "h1", "n1", "h2", "r1", "lse", "probs", "tokens")] + \
               [("fused_attention", ctypes.c_int32), ("reserved", ctypes.c_int32)]


def lib_path() -> str:
    return os.path.join(_HERE, "lib", "libdfdx_rocm.so")


_lib = None

# every symbol include/dfdx_rocm.h declares
EXPORTS = [
    "dfdx_rocm_create", "dfdx_rocm_destroy", "dfdx_rocm_strerror", "dfdx_rocm_device_info",
    "dfdx_rocm_alloc", "dfdx_rocm_free", "dfdx_rocm_memset_zero", "dfdx_rocm_copy_h2d", "dfdx_rocm_copy_d2h",
    "dfdx_rocm_copy_d2d", "dfdx_rocm_synchronize", "dfdx_rocm_zero_deferred", "dfdx_rocm_settle_zeros", "dfdx_rocm_forget_zeros",
    "dfdx_rocm_enable_cache", "dfdx_rocm_disable_cache",
    "dfdx_rocm_empty_cache", "dfdx_rocm_cache_stats", "dfdx_rocm_gemm", "dfdx_rocm_gemm_noalloc", "dfdx_rocm_gemm_plan",
    "dfdx_rocm_mfma_variant_count", "dfdx_rocm_gemm_time", "dfdx_rocm_gemm_time_rotating",
    "dfdx_rocm_matmat_forward", "dfdx_rocm_matmat_backward",
    "dfdx_rocm_matmat_br_forward", "dfdx_rocm_matmat_br_backward",
    "dfdx_rocm_matmat_batch3_forward", "dfdx_rocm_matmat_batch3_backward",
    "dfdx_rocm_matmat_batch4_forward", "dfdx_rocm_matmat_batch4_backward",
    "dfdx_rocm_linear_forward", "dfdx_rocm_linear_backward",
    "dfdx_rocm_bias_forward", "dfdx_rocm_bias_backward",
    "dfdx_rocm_scalar_mul_forward", "dfdx_rocm_scalar_mul_backward",
    "dfdx_rocm_softmax_forward", "dfdx_rocm_softmax_backward",
    "dfdx_rocm_reshape_forward", "dfdx_rocm_reshape_backward",
    "dfdx_rocm_attention_forward", "dfdx_rocm_attention_backward",
    "dfdx_rocm_layer_norm_forward", "dfdx_rocm_layer_norm_backward",
    "dfdx_rocm_relu_forward", "dfdx_rocm_relu_backward",
    "dfdx_rocm_add_forward", "dfdx_rocm_add_backward",
    "dfdx_rocm_encoder_plan", "dfdx_rocm_encoder_forward", "dfdx_rocm_encoder_backward",
    "dfdx_rocm_conv2d_forward", "dfdx_rocm_conv2d_backward",
]


def load_library() -> ctypes.CDLL:
    """Load the built HIP library; raises if it has not been built (no fallback)."""
    global _lib
    if _lib is None:
        path = lib_path()
        if not os.path.exists(path):
            raise FileNotFoundError(
                f"{path} is missing: build it with `make -C dfdx_amd/csrc` (or __graft_entry__.build())")
        lib = ctypes.CDLL(path)
        lib.dfdx_rocm_strerror.restype = ctypes.c_char_p
        lib.dfdx_rocm_strerror.argtypes = [ctypes.c_int]
        for name in EXPORTS:
            fn = getattr(lib, name)
            if name != "dfdx_rocm_strerror":
                fn.restype = ctypes.c_int
        _lib = lib
    return _lib


def _load_host():
    """The native half of this front-end (csrc/host.cpp): the entry points a training or inference step goes through, as functions
    that take addresses, Views and tuples of numbers as they are.  Needs torch's libraries, so torch is imported before."""
    try:
        from . import _host
    except ImportError as e:
        raise FileNotFoundError(f"the extension module _host in {_HERE} is missing or does not load ({e}): build it with `make -C dfdx_amd/csrc` "
                                "(or __graft_entry__.build()), with the interpreter and the torch that run this") from e
    return _host


def _i64s(v) -> bytes:
    """An int64_t array as an argument: the call reads it while the bytes object lives."""
    return struct.pack(f"{len(v)}q", *v)


def _axes(v):
    """One number per axis as an argument: a tuple as it is, unless it is longer than the native module takes (the library refuses such ranks)."""
    return tuple(v) if len(v) <= 8 else _i64s(v)


@dataclass
class View:
    """Device storage seen through a shape and element strides (a dfdx tensor's kernel-side face)."""
    storage: "object"           # torch.uint8 CUDA tensor owning the bytes
    dtype: str
    shape: tuple
    strides: tuple
    offset: int = 0             # in elements
    owner: "object" = None      # keeps an arena's declarations alive exactly as long as views of it exist (zeros_many)

    @property
    def ptr(self) -> int:
        return self.storage.data_ptr() + self.offset * ITEMSIZE[self.dtype] if self.offset else self.storage.data_ptr()

    def permute(self, *axes) -> "View":
        """Zero-copy permute (reference: tensor_ops/permute_to.rs:38-52)."""
        return View(self.storage, self.dtype, tuple(self.shape[a] for a in axes),
                    tuple(self.strides[a] for a in axes), self.offset, self.owner)

    def numel_storage(self) -> int:
        return self.storage.numel() // ITEMSIZE[self.dtype]


class _Arena:
    """One allocation that several Views are carved from.  When the last View of it goes, whatever zero declarations
    its pieces still carry are withdrawn (``dfdx_rocm_forget_zeros``) BEFORE torch gets the memory back, so that a later
    settle cannot write zeros into memory that has a new owner by then.  (At interpreter exit the context may go first; it
    takes its declarations with it.)"""
    __slots__ = ("dev", "raw")

    def __init__(self, dev: "Rocm", raw):
        self.dev, self.raw = dev, raw   # the views keep the device alive, which the declarations need anyway

    def forget(self):
        dev, raw = self.dev, self.raw
        if dev is not None and dev.ctx:
            dev._f.forget_zeros(dev._at, raw.data_ptr(), raw.numel())
        self.dev = None

    def __del__(self):
        try:
            self.forget()
        except Exception:   # at interpreter exit
            pass


def _row_major(shape):
    n = len(shape)
    if n == 1:
        return (1,)
    if n == 2:
        return (shape[1], 1)
    if n == 3:
        return (shape[1] * shape[2], shape[2], 1)
    s = [1] * n
    for i in range(n - 2, -1, -1):
        s[i] = s[i + 1] * shape[i + 1]
    return tuple(s)


class Rocm:
    """One GPU context.  ``Rocm(ordinal)`` ~ ``Cuda::try_build(ordinal, seed)`` (tensor/cuda/device.rs:72-90)."""

    def __init__(self, ordinal: int = 0):
        import torch

        self._torch = torch
        if not torch.cuda.is_available():
            raise RuntimeError("no GPU visible: the Rocm device needs an MI355X (there is no CPU fallback)")
        self.lib = load_library()
        self._f = _load_host()
        self.ordinal = ordinal
        self.device = torch.device("cuda", ordinal)
        torch.cuda.set_device(ordinal)
        stream = torch.cuda.current_stream(self.device).cuda_stream
        ctx = ctypes.c_void_p()
        self._check(self.lib.dfdx_rocm_create(ordinal, ctypes.c_void_p(stream), ctypes.byref(ctx)))
        self.ctx, self._at = ctx, ctx.value
        self._bytes = self._f.allocator(ordinal)   # uninitialised bytes on the device

    def close(self):
        if getattr(self, "ctx", None):
            self.lib.dfdx_rocm_destroy(self.ctx)
            self.ctx, self._at = None, 0

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # ------------------------------------------------------------------ misc --
    def _check(self, code: int):
        if code != 0:
            raise RocmError(code, self.lib.dfdx_rocm_strerror(code).decode())

    def synchronize(self):
        self._check(self.lib.dfdx_rocm_synchronize(self.ctx))

    def device_info(self):
        name = ctypes.create_string_buffer(128)
        cus, mhz = ctypes.c_int(), ctypes.c_int()
        self._check(self.lib.dfdx_rocm_device_info(self.ctx, name, 128, ctypes.byref(cus), ctypes.byref(mhz)))
        return {"name": name.value.decode(), "compute_units": cus.value, "clock_mhz": mhz.value}

    # ----------------------------------------------------------------- cache --
    def enable_cache(self):
        """``Cache::enable_cache`` (tensor/storage_traits.rs:41-77): freed buffers are kept for the next allocation of their size."""
        self._check(self.lib.dfdx_rocm_enable_cache(self.ctx))

    def disable_cache(self):
        self._check(self.lib.dfdx_rocm_disable_cache(self.ctx))

    def empty_cache(self):
        self._check(self.lib.dfdx_rocm_empty_cache(self.ctx))

    def cache_stats(self):
        n, b = ctypes.c_size_t(), ctypes.c_size_t()
        self._check(self.lib.dfdx_rocm_cache_stats(self.ctx, ctypes.byref(n), ctypes.byref(b)))
        return n.value, b.value

    def alloc(self, nbytes: int, zeroed=True) -> int:
        """``Storage::try_alloc_len`` / ``alloc_empty`` through the library's own allocator; returns the device address.
        ``zeroed`` = ``ZERO_DEFERRED``: zero as far as the library's calls can tell, the fill only runs if a call needs it."""
        p = ctypes.c_void_p()
        self._check(self.lib.dfdx_rocm_alloc(self.ctx, ctypes.c_size_t(nbytes), int(zeroed), ctypes.byref(p)))
        return p.value

    def free(self, ptr: int):
        self._check(self.lib.dfdx_rocm_free(self.ctx, ctypes.c_void_p(ptr)))

    def zero_deferred(self, ptr: int, nbytes: int):
        """Declares ``nbytes`` at ``ptr`` zero without filling them (``dfdx_rocm_zero_deferred``): the first call that
        accumulates into the whole buffer stores 0 + value, any other first use runs the fill."""
        self._check(self._f.zero_deferred(self._at, ptr, nbytes))

    def forget_zeros(self, ptr: int, nbytes: int):
        """Withdraws the zero declarations inside ``[ptr, ptr + nbytes)`` without filling (``dfdx_rocm_forget_zeros``):
        what the owner of declared storage calls before it releases that storage unsettled."""
        self._check(self.lib.dfdx_rocm_forget_zeros(self.ctx, ctypes.c_void_p(ptr), ctypes.c_size_t(nbytes)))

    def settle_zeros(self):
        """Runs every deferred fill still pending: needed before code outside the library reads such a buffer."""
        self._check(self._f.settle_zeros(self._at))

    # --------------------------------------------------------------- storage --
    def tensor(self, host: np.ndarray, dtype: str, shape=None, strides=None) -> View:
        """Upload ``host`` (storage order) and view it; bf16 storage is given as uint16 bit patterns."""
        torch = self._torch
        host = np.ascontiguousarray(host)
        if host.dtype != NP_DTYPES[dtype]:
            raise TypeError(f"{dtype} storage must be numpy {NP_DTYPES[dtype]}, got {host.dtype}")
        shape = tuple(host.shape) if shape is None else tuple(shape)
        strides = _row_major(shape) if strides is None else tuple(strides)
        raw = torch.from_numpy(host.reshape(-1).view(np.uint8).copy()).to(self.device)
        if raw.numel() == 0:
            raw = torch.zeros(16, dtype=torch.uint8, device=self.device)
        return View(raw, dtype, shape, strides)

    def zeros(self, dtype: str, shape, numel_storage: Optional[int] = None, strides=None) -> View:
        """Zero-filled storage (``Storage::try_alloc_len``, tensor/cuda/device.rs:259-266)."""
        torch = self._torch
        shape = tuple(shape)
        n = int(np.prod(shape, dtype=np.int64)) if numel_storage is None else numel_storage
        raw = self._zeroed_bytes(max(n * ITEMSIZE[dtype], 16))
        return View(raw, dtype, shape, _row_major(shape) if strides is None else tuple(strides))

    def zeros_many(self, likes, deferred: bool = False) -> list:
        """Zero-filled storages for several tensors at once: one allocation, ONE fill launch, each view on its own
        256 B-aligned piece.  ``likes`` are Views whose dtype / shape give the sizes (contiguous row-major results).
        What a pooling allocator behind ``try_alloc_grad`` would do for the gradient buffers of one backward pass:
        small fills are launch-bound (3.5 us for 2 MiB), one large fill runs at the HBM write rate.
        ``deferred``: no fill at all; every piece is declared zero (``zero_deferred``) and the first backward op that
        accumulates into the whole of it stores instead -- read the results through this object (``to_host``) or
        call ``settle_zeros`` first.  The declarations are withdrawn when the last of the returned Views (and of the
        Views derived from them) is dropped, so the arena never goes back to the allocator with a fill still promised."""
        return self._f.carve(self, View, _Arena, likes, deferred)

    def _zeroed_bytes(self, nbytes: int):
        """Device memory from torch's allocator, cleared by the library's own fill kernel (``dfdx_rocm_memset_zero``)."""
        raw = self._bytes(nbytes)
        self._check(self._f.memset_zero(self._at, raw.data_ptr(), nbytes))
        return raw

    def empty(self, dtype: str, shape) -> View:
        """Uninitialised storage for an output that a forward kernel overwrites (``alloc_empty``,
        tensor_ops/matmul/cuda_kernel.rs:253)."""
        return self._f.empty(View, self.ordinal, dtype, tuple(shape))

    def zeros_like_storage(self, v: View) -> View:
        """A gradient buffer for ``v``: zero-filled, same physical length, same strides (gradients.rs:53-58)."""
        raw = self._zeroed_bytes(v.storage.numel())
        return View(raw, v.dtype, v.shape, v.strides, v.offset)

    def to_host(self, v: View) -> np.ndarray:
        """The storage bytes as a flat numpy array of the storage dtype."""
        n = v.numel_storage()
        self.settle_zeros()   # the storage may still wait for a deferred zero fill
        return v.storage.cpu().numpy().view(NP_DTYPES[v.dtype])[:n].copy()

    # ------------------------------------------------------------------ gemm --
    def gemm_desc(self, dtype, m, k, n, a, a_strides, b, b_strides, c, c_strides, accumulate=False,
                  batch=(1, 1), a_batch=(0, 0), b_batch=(0, 0), c_batch=(0, 0), bias=None, reduce_batch=False,
                  kernel=KERNEL_AUTO, variant=0, no_split_k=False, split_k=0) -> GemmDesc:
        d = GemmDesc()
        d.dtype, d.accumulate = DTYPES[dtype], int(bool(accumulate))
        d.m, d.n, d.k = m, n, k
        d.batch1, d.batch2 = batch
        d.a, d.a_rs, d.a_cs, d.a_b1, d.a_b2 = a, a_strides[0], a_strides[1], a_batch[0], a_batch[1]
        d.b, d.b_rs, d.b_cs, d.b_b1, d.b_b2 = b, b_strides[0], b_strides[1], b_batch[0], b_batch[1]
        d.c, d.c_rs, d.c_cs, d.c_b1, d.c_b2 = c, c_strides[0], c_strides[1], c_batch[0], c_batch[1]
        d.bias = bias
        d.reduce_batch, d.kernel, d.variant = int(bool(reduce_batch)), kernel, variant
        d.flags = (1 if no_split_k else 0) | ((split_k & 0xff) << 8)
        return d

    def gemm(self, desc: GemmDesc):
        """``MatMulImpl::matmul`` / ``Cuda::gemm[_batch]`` (cpu_kernel.rs:38-50, cuda_kernel.rs:153-237)."""
        self._check(self.lib.dfdx_rocm_gemm(self.ctx, ctypes.byref(desc)))

    def gemm_noalloc(self, desc: GemmDesc):
        """The same product with the partial sums of a split reduction in the library's fixed scratch array: allocates
        nothing; ``RocmError`` (code -5) when the plan needs more than ``NOALLOC_SCRATCH_BYTES``."""
        self._check(self.lib.dfdx_rocm_gemm_noalloc(self.ctx, ctypes.byref(desc)))

    def gemm_plan(self, desc: GemmDesc):
        kernel, variant = ctypes.c_int(), ctypes.c_int()
        name = ctypes.create_string_buffer(96)
        self._check(self.lib.dfdx_rocm_gemm_plan(self.ctx, ctypes.byref(desc), ctypes.byref(kernel),
                                                 ctypes.byref(variant), name, 96))
        return kernel.value, variant.value, name.value.decode()

    def gemm_time(self, desc: GemmDesc, warmup: int, iters: int) -> float:
        ms = ctypes.c_float()
        self._check(self.lib.dfdx_rocm_gemm_time(self.ctx, ctypes.byref(desc), warmup, iters, ctypes.byref(ms)))
        return ms.value

    def gemm_time_rotating(self, descs, warmup: int, iters: int) -> float:
        """Average ms per launch with launch i running ``descs[i % len(descs)]`` (each on its own buffers)."""
        arr = (GemmDesc * len(descs))(*descs)
        ms = ctypes.c_float()
        self._check(self.lib.dfdx_rocm_gemm_time_rotating(self.ctx, arr, len(descs), warmup, iters, ctypes.byref(ms)))
        return ms.value

    def mfma_variant_count(self, dtype: str) -> int:
        return self.lib.dfdx_rocm_mfma_variant_count(DTYPES[dtype])

    # --------------------------------------------------------- kernel traits --
    def forward(self, lhs: View, rhs: View) -> View:
        """Dispatch on rank like ``TryMatMul`` (mod.rs:133-311); rank-1 operands are reshapes (mod.rs:139-174)."""
        dt, ls, rs, lt, rt = lhs.dtype, lhs.shape, rhs.shape, lhs.strides, rhs.strides
        assert dt == rhs.dtype
        L, R = len(ls), len(rs)
        if L <= 2 and R <= 2:
            if L == 2 and R == 2:
                assert ls[1] == rs[0], f"left: {ls[1]}\n right: {rs[0]}"
                (m, k), n = ls, rs[1]
                shape = (m, n)
            elif L == 1 and R == 1:      # outer product: (M,1) x (1,N)
                m, k, n = ls[0], 1, rs[0]
                shape, lt, rt = (m, n), (lt[0], 1), (n * rt[0], rt[0])
            elif L == 1:                 # (1,K) x (K,N) -> (N,)
                assert ls[0] == rs[0], f"left: {ls[0]}\n right: {rs[0]}"
                m, (k, n) = 1, rs
                shape, lt = (n,), (k * lt[0], lt[0])
            else:                        # (M,K) x (K,1) -> (M,)
                assert ls[1] == rs[0], f"left: {ls[1]}\n right: {rs[0]}"
                (m, k), n = ls, 1
                shape, rt = (m,), (rt[0], 1)
            fn, dims = self._f.matmat_forward, (m, k, n)
        elif L == 3 and R == 2:
            assert ls[2] == rs[0], f"left: {ls[2]}\n right: {rs[0]}"
            (b, m, k), n = ls, rs[1]
            fn, dims, shape = self._f.matmat_br_forward, (b, m, k, n), (b, m, n)
        elif L == 3 and R == 3:
            assert ls[0] == rs[0], f"left: {ls[0]}\n right: {rs[0]}"
            assert ls[2] == rs[1], f"left: {ls[2]}\n right: {rs[1]}"
            (b, m, k), n = ls, rs[2]
            fn, dims, shape = self._f.matmat_batch3_forward, (b, m, k, n), (b, m, n)
        elif L == 4 and R == 4:
            assert ls[0] == rs[0], f"left: {ls[0]}\n right: {rs[0]}"
            assert ls[1] == rs[1], f"left: {ls[1]}\n right: {rs[1]}"
            assert ls[3] == rs[2], f"left: {ls[3]}\n right: {rs[2]}"
            (b, s, m, k), n = ls, rs[3]
            fn, dims, shape = self._f.matmat_batch4_forward, (b, s, m, k, n), (b, s, m, n)
        else:
            raise TypeError(f"matmul of rank {L} by rank {R} is not defined (mod.rs:133-311)")
        out = self.empty(dt, shape)
        rc = fn(self._at, DTYPES[dt], *dims, lhs, lt, rhs, rt, out)
        if rc:
            self._check(rc)
        return out

    def backward(self, lhs: View, grad_lhs: View, rhs: View, grad_rhs: View, grad_out: View):
        """``D::backward(lhs, grad_lhs, rhs, grad_rhs, grad_out)``; grad_out contiguous; grads accumulate."""
        ls, rs, lt, rt = lhs.shape, rhs.shape, lhs.strides, rhs.strides
        L, R = len(ls), len(rs)
        if L <= 2 and R <= 2:
            if L == 2 and R == 2:
                dims = (*ls, rs[1])
            elif L == 1 and R == 1:
                n = rs[0]
                dims, lt, rt = (ls[0], 1, n), (lt[0], 1), (n * rt[0], rt[0])
            elif L == 1:
                k, n = rs
                dims, lt = (1, k, n), (k * lt[0], lt[0])
            else:
                dims, rt = (*ls, 1), (rt[0], 1)
            fn = self._f.matmat_backward
        elif L == 3 and R == 2:
            fn, dims = self._f.matmat_br_backward, (*ls, rs[1])
        elif L == 3 and R == 3:
            fn, dims = self._f.matmat_batch3_backward, (*ls, rs[2])
        elif L == 4 and R == 4:
            fn, dims = self._f.matmat_batch4_backward, (*ls, rs[3])
        else:
            raise TypeError(f"matmul of rank {L} by rank {R} is not defined")
        rc = fn(self._at, DTYPES[lhs.dtype], *dims, lhs, lt, grad_lhs, rhs, rt, grad_rhs, grad_out)
        if rc:
            self._check(rc)

    def linear_forward(self, x: View, weight: View, bias: Optional[View]) -> View:
        """``Linear::try_forward`` (dfdx/src/nn/layers/linear.rs:82-89); weight is the (O, I) storage."""
        o, i = weight.shape
        assert weight.strides == (i, 1), "Linear weight storage is (O, I) row-major"
        shape = x.shape
        assert shape[-1] == i, f"left: {shape[-1]}\n right: {i}"
        rows, xs = self._linear_rows(x, i)
        out = self.empty(x.dtype, (*shape[:-1], o))
        rc = self._f.linear_forward(self._at, DTYPES[x.dtype], rows, i, o, x, xs, weight, bias, out)
        if rc:
            self._check(rc)
        return out

    def _linear_rows(self, x: View, i: int):
        if len(x.shape) == 2:
            return x.shape[0], x.strides
        if len(x.shape) == 1:
            return 1, (i * x.strides[0], x.strides[0])
        assert x.strides == _row_major(x.shape), "batched Linear input must be contiguous to fold its rows"
        return math.prod(x.shape[:-1]), (i, 1)

    def linear_backward(self, x: View, grad_x: View, weight: View, grad_weight: View, grad_bias: Optional[View],
                        grad_out: View):
        """Backward of ``Linear``: grad_x += go.W, grad_weight += go^T.x, grad_bias += column sums of go."""
        o, i = weight.shape
        assert weight.strides == (i, 1), "Linear weight storage is (O, I) row-major"
        shape = x.shape
        assert shape[-1] == i, f"left: {shape[-1]}\n right: {i}"
        assert grad_out.shape == (*shape[:-1], o) and grad_out.strides == _row_major(grad_out.shape)
        rows, xs = self._linear_rows(x, i)
        rc = self._f.linear_backward(self._at, DTYPES[x.dtype], rows, i, o, x, xs, grad_x, weight, grad_weight, grad_bias, grad_out)
        if rc:
            self._check(rc)

    def bias_forward(self, x: View, bias: View) -> View:
        """``Bias1D::try_forward`` (dfdx/src/nn/layers/bias1d.rs:62-78) on a contiguous input."""
        cols = bias.shape[0]
        assert x.shape[-1] == cols, f"left: {x.shape[-1]}\n right: {cols}"
        assert x.strides == _row_major(x.shape) and bias.strides == (1,)
        out = self.empty(x.dtype, x.shape)
        self._check(self._f.bias_forward(self._at, DTYPES[x.dtype], math.prod(x.shape[:-1]), cols, x.ptr, bias.ptr, out.ptr))
        return out

    def bias_backward(self, grad_out: View, grad_bias: View):
        """grad_bias += column sums of grad_out (the broadcast operand's share of the add's backward)."""
        cols = grad_bias.shape[0]
        assert grad_out.shape[-1] == cols and grad_out.strides == _row_major(grad_out.shape)
        self._check(self._f.bias_backward(self._at, DTYPES[grad_out.dtype], math.prod(grad_out.shape[:-1]), cols, grad_out.ptr, grad_bias.ptr))

    # ------------------------------------------------- ops between attention's GEMMs --
    def _like(self, x: View) -> View:
        """Uninitialised storage of the same physical length, seen the same way."""
        return View(self._bytes(x.storage.nbytes), x.dtype, x.shape, x.strides, x.offset)

    def scalar_mul_forward(self, x: View, scalar: float) -> View:
        """``x * scalar`` over the physical storage (unary kernel, utilities/cpu_kernels.rs:46-79); same strides."""
        out = self._like(x)
        self._check(self._f.scalar_mul_forward(self._at, DTYPES[x.dtype], x.numel_storage(), x.storage.data_ptr(), scalar, out.storage.data_ptr()))
        return out

    def scalar_mul_backward(self, scalar: float, grad_inp: View, grad_out: View):
        assert grad_inp.numel_storage() == grad_out.numel_storage()
        self._check(self._f.scalar_mul_backward(self._at, DTYPES[grad_inp.dtype], grad_inp.numel_storage(), scalar,
                                                grad_inp.storage.data_ptr(), grad_out.storage.data_ptr()))

    def softmax_forward(self, x: View, scale: float = 1.0) -> View:
        """softmax(scale * x) over the last axis of a contiguous tensor (softmax.rs:70-83)."""
        assert x.strides == _row_major(x.shape), "softmax input must be contiguous"
        out = View(self._bytes(x.storage.nbytes), x.dtype, x.shape, x.strides)
        self._check(self._f.softmax_forward(self._at, DTYPES[x.dtype], math.prod(x.shape[:-1]), x.shape[-1], x.ptr, scale, out.ptr))
        return out

    def softmax_backward(self, out: View, grad_x: View, grad_out: View, scale: float = 1.0):
        assert out.strides == _row_major(out.shape) and grad_out.shape == out.shape and grad_x.shape == out.shape
        self._check(self._f.softmax_backward(self._at, DTYPES[out.dtype], math.prod(out.shape[:-1]), out.shape[-1], out.ptr, scale,
                                             grad_x.ptr, grad_out.ptr))

    def reshape_forward(self, x: View, new_shape) -> View:
        """``try_reshape_like`` (reshape_to/mod.rs:90-115): free for a contiguous tensor, a copy otherwise."""
        new_shape = tuple(int(d) for d in new_shape)
        assert math.prod(x.shape) == math.prod(new_shape), f"left: {math.prod(x.shape)}\n right: {math.prod(new_shape)}"
        if x.strides == _row_major(x.shape):
            return View(x.storage, x.dtype, new_shape, _row_major(new_shape), x.offset, x.owner)
        out = self.empty(x.dtype, new_shape)
        self._check(self._f.reshape_forward(self._at, DTYPES[x.dtype], len(x.shape), _axes(x.shape), _axes(x.strides), x, out))
        return out

    def reshape_backward(self, x: View, grad_inp: View, grad_out: View):
        """Backward of a copying reshape: grad_inp (laid out like x's storage) += grad_out through x's strides."""
        self._check(self._f.reshape_backward(self._at, DTYPES[x.dtype], len(x.shape), _axes(x.shape), _axes(x.strides), grad_inp, grad_out))

    def attention_supported(self, dtype: str, head_dim: int) -> bool:
        """Whether the fused attention takes this element type and head dimension (else: matmul, softmax, matmul)."""
        return dtype in ("f16", "bf16") and head_dim in (32, 64, 128)

    def attention_forward(self, q: View, k: View, v: View, scale: float, need_backward: bool = True):
        """softmax(scale * q.k^T).v for (B, H, S, D) views sharing their strides; returns the result in token layout
        (B, S, H * D) and the row statistics (f32) the backward takes (``None`` without ``need_backward``)."""
        B, H, S, D = q.shape
        assert k.shape == q.shape and v.shape == q.shape and k.strides == q.strides and v.strides == q.strides and q.strides[3] == 1
        out = self.empty(q.dtype, (B, S, H * D))
        lse = self.empty("f32", (B, H, S)) if need_backward else None
        self._check(self._f.attention_forward(self._at, DTYPES[q.dtype], B, H, S, D, q.ptr, k.ptr, v.ptr, tuple(q.strides[:3]), scale,
                                              out.ptr, (S * H * D, D, H * D), lse.ptr if lse is not None else None))
        return out, lse

    def attention_backward(self, q: View, grad_q: View, k: View, grad_k: View, v: View, grad_v: View, scale: float, out: View,
                           grad_out: View, lse: View):
        """Gradients of ``attention_forward``: added into grad_q, grad_k, grad_v, each laid out like the storage of q, k, v (one
        set of strides, no broadcast axis); out, lse: what the forward returned; grad_out: like out."""
        B, H, S, D = q.shape
        assert k.shape == q.shape and v.shape == q.shape and k.strides == q.strides and v.strides == q.strides and q.strides[3] == 1
        tokens = (B, S, H * D)
        assert out.shape == tokens and grad_out.shape == tokens and out.strides == grad_out.strides == _row_major(tokens), \
            f"left: {out.shape}, {grad_out.shape}\n right: {tokens}"
        assert lse.shape == (B, H, S) and lse.dtype == "f32" and all(t.dtype == q.dtype for t in (grad_q, k, grad_k, v, grad_v, out, grad_out))
        reach = 1 + sum((n - 1) * s for n, s in zip(q.shape, q.strides)) if B * H * S else 0
        assert all(t.numel_storage() - t.offset >= reach for t in (grad_q, grad_k, grad_v)), "gradients smaller than what their strides reach"
        self._check(self._f.attention_backward(self._at, DTYPES[q.dtype], B, H, S, D, q.ptr, k.ptr, v.ptr, tuple(q.strides[:3]), scale,
                                               out.ptr, grad_out.ptr, (S * H * D, D, H * D), lse.ptr, grad_q.ptr, grad_k.ptr, grad_v.ptr))

    # ------------------------------------------- ops between an encoder block's GEMMs --
    def layer_norm_forward(self, x: View, gamma: View, beta: View, epsilon: float = 1e-5) -> View:
        """``LayerNorm1D::try_forward`` over the last axis of a contiguous tensor (layer_norm1d.rs:87-91)."""
        assert x.strides == _row_major(x.shape), "layer norm input must be contiguous"
        cols = x.shape[-1]
        assert gamma.shape == (cols,) and beta.shape == (cols,), f"left: {gamma.shape}\n right: {(cols,)}"
        out = View(self._bytes(x.storage.nbytes), x.dtype, x.shape, x.strides)
        self._check(self._f.layer_norm_forward(self._at, DTYPES[x.dtype], math.prod(x.shape[:-1]), cols, x.ptr, gamma.ptr, beta.ptr, epsilon, out.ptr))
        return out

    def layer_norm_backward(self, x: View, gamma: View, grad_x: View, grad_gamma: View, grad_beta: View, grad_out: View,
                            epsilon: float = 1e-5):
        assert x.strides == _row_major(x.shape) and grad_out.shape == x.shape and grad_x.shape == x.shape
        self._check(self._f.layer_norm_backward(self._at, DTYPES[x.dtype], math.prod(x.shape[:-1]), x.shape[-1], x.ptr, gamma.ptr, epsilon,
                                                grad_x.ptr, grad_gamma.ptr, grad_beta.ptr, grad_out.ptr))

    def relu_forward(self, x: View) -> View:
        """``t.relu()`` over the physical storage (relu/cpu_kernel.rs:3-18); same strides."""
        out = self._like(x)
        self._check(self._f.relu_forward(self._at, DTYPES[x.dtype], x.numel_storage(), x.storage.data_ptr(), out.storage.data_ptr()))
        return out

    def relu_backward(self, x: View, grad_x: View, grad_out: View):
        assert grad_x.numel_storage() == grad_out.numel_storage() == x.numel_storage()
        self._check(self._f.relu_backward(self._at, DTYPES[x.dtype], x.numel_storage(), x.storage.data_ptr(), grad_x.storage.data_ptr(),
                                          grad_out.storage.data_ptr()))

    def add_forward(self, lhs: View, rhs: View) -> View:
        """``lhs + rhs`` for two tensors of one shape and layout (add/cpu_kernel.rs:4-26)."""
        assert lhs.shape == rhs.shape, f"left: {lhs.shape}\n right: {rhs.shape}"
        assert lhs.strides == rhs.strides and lhs.numel_storage() == rhs.numel_storage()
        out = self._like(lhs)
        self._check(self._f.add_forward(self._at, DTYPES[lhs.dtype], lhs.numel_storage(), lhs.storage.data_ptr(), rhs.storage.data_ptr(),
                                        out.storage.data_ptr()))
        return out

    def add_backward(self, grad_lhs: View, grad_rhs: View, grad_out: View):
        assert grad_lhs.numel_storage() == grad_rhs.numel_storage() == grad_out.numel_storage()
        self._check(self._f.add_backward(self._at, DTYPES[grad_out.dtype], grad_out.numel_storage(), grad_lhs.storage.data_ptr(),
                                         grad_rhs.storage.data_ptr(), grad_out.storage.data_ptr()))

    # ---------------------------------------------------------------- conv2d --
    def _conv2d_op(self, img: View, filters: View, stride, padding, dilation, groups) -> Conv2DOp:
        """Shape checks and output size of ``try_conv2d`` (conv2d/mod.rs:143-160, 279-308)."""
        shape = img.shape if len(img.shape) == 4 else (1,) + tuple(img.shape)
        batch, chan_in, h, w = shape
        chan_out, cg, kernel, k2 = filters.shape
        assert chan_in == cg * groups, f"left: {chan_in}\n right: {cg * groups}"
        assert kernel == k2, f"left: {kernel}\n right: {k2}"
        assert chan_out % groups == 0
        if img.strides != _row_major(img.shape) or filters.strides != _row_major(filters.shape):
            raise ValueError("Image & filter inputs to conv2d must be contiguous")
        size = lambda d: (d + 2 * padding - 1 - dilation * (kernel - 1)) // stride + 1
        assert h + 2 * padding - 1 >= dilation * (kernel - 1) and w + 2 * padding - 1 >= dilation * (kernel - 1)
        return Conv2DOp(kernel, stride, padding, dilation, groups, batch, chan_in, chan_out, h, size(h), w, size(w))

    def conv2d_forward(self, img: View, filters: View, stride=1, padding=0, dilation=1, groups=1) -> View:
        """``(img, filters).conv2d(stride, padding, dilation, groups)``; img (B, C, H, W) or (C, H, W)."""
        op = self._conv2d_op(img, filters, stride, padding, dilation, groups)
        lead = (op.batch,) if len(img.shape) == 4 else ()
        out = self.empty(img.dtype, lead + (op.chan_out, op.h_out, op.w_out))
        self._check(self._f.conv2d_forward(self._at, DTYPES[img.dtype], ctypes.addressof(op), img.ptr, filters.ptr, out.ptr))
        return out

    def conv2d_backward(self, img: View, grad_img: View, filters: View, grad_filters: View, grad_out: View,
                        stride=1, padding=0, dilation=1, groups=1):
        op = self._conv2d_op(img, filters, stride, padding, dilation, groups)
        self._check(self._f.conv2d_backward(self._at, DTYPES[img.dtype], ctypes.addressof(op), img.ptr, grad_img.ptr, filters.ptr,
                                            grad_filters.ptr, grad_out.ptr))
