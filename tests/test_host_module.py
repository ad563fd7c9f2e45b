"""The native half of the Python front-end (csrc/host.cpp): what its entry points take as arguments and refuse, without a GPU."""
import ctypes
import os
import subprocess
from types import SimpleNamespace

import pytest
import torch

from dfdx_amd import EncoderBlock, View
from dfdx_amd.rocm import Encoder, Rocm, RocmError, _load_host, load_library

INVALID = -1   # DFDX_ROCM_ERR_INVALID_ARG: what a null context gets


@pytest.mark.parametrize("ctx", [None, 0, ctypes.c_void_p()])
@pytest.mark.parametrize("strides", [(3, 1), [3, 1], ctypes.addressof((ctypes.c_int64 * 2)(3, 1)), bytes(16)])
def test_forms_of_arguments(ctx, strides):
    host, view = _load_host(), View(torch.zeros(64, dtype=torch.uint8), "f32", (2, 3), (3, 1), 1)
    assert host.matmat_forward(ctx, 0, 2, 3, 2, view, strides, view.ptr, strides, None) == INVALID


def test_what_is_refused():
    host = _load_host()
    with pytest.raises(TypeError):
        host.settle_zeros()
    with pytest.raises(TypeError):
        host.memset_zero(0, 0, "a size")
    with pytest.raises(AttributeError):
        host.memset_zero(0, object(), 0)
    with pytest.raises(ValueError):
        host.matmat_forward(0, 0, 1, 1, 1, 0, (1,) * 9, 0, (1, 1), 0)
    with pytest.raises(KeyError):
        host.memset_zero(0, View(torch.zeros(8, dtype=torch.uint8), "f8", (4,), (1,), 4), 0)
    with pytest.raises(KeyError):
        host.empty(View, 0, "f8", (4,))


def test_pieces_share_storage_and_count_of_changes():
    arena = torch.zeros(64, dtype=torch.uint8)
    views = _load_host().pieces(View, arena, "f32", (("a", 0, 16, (2, 2), (2, 1)), ("b", 32, 8, (2,), (1,))))
    assert list(views) == ["a", "b"] and views["b"] == View(views["b"].storage, "f32", (2,), (1,), 0, None)
    views["b"].storage.fill_(7)
    assert arena[32:40].eq(7).all() and arena.sum() == 56 and views["a"].storage.numel() == 16
    assert arena._version == views["a"].storage._version == 1
    assert views["a"].storage.view(torch.float32).shape == (4,) and views["b"].ptr == arena.data_ptr() + 32


def test_parameters():
    """Addresses of the sixteen parameters behind the description, or None where one is not what the block was made for."""
    host = _load_host()
    p = {f"p{i}": View(torch.zeros(64, dtype=torch.uint8), "f16", (4, 2), (2, 1), i % 2) for i in range(16)}
    specs = tuple((n, (4, 2), (2, 1)) for n in p)
    raw = bytes(Encoder(1, 0, 2, 3, 4, 5, 6))
    desc = Encoder.from_buffer_copy(host.parameters(raw, p, "f16", specs))
    assert list(desc.params) == [v.ptr for v in p.values()] and (desc.batch, desc.d_ff) == (2, 6)
    for wrong in (View(p["p3"].storage, "f16", (2, 4), (4, 1)), View(p["p3"].storage, "f16", (4, 2), (1, 4)), View(p["p3"].storage, "bf16", (4, 2), (2, 1))):
        assert host.parameters(raw, p | {"p3": wrong}, "f16", specs) is None
    with pytest.raises(KeyError):
        host.parameters(raw, {}, "f16", specs)


def test_parameters_with_strides_in_a_list():
    """A View's strides may be any sequence; what is refused stays refused."""
    host = _load_host()
    p = {f"p{i}": View(torch.zeros(64, dtype=torch.uint8), "f16", (4, 2), [2, 1] if i == 3 else (2, 1)) for i in range(16)}
    plan = SimpleNamespace(raw=bytes(Encoder(1, 0, 2, 3, 4, 5, 6)), params=tuple((n, (4, 2), (2, 1)) for n in p))
    block = SimpleNamespace(dev=SimpleNamespace(_f=host), p=p, dtype="f16")
    desc = Encoder.from_buffer_copy(EncoderBlock._desc(block, plan))
    assert list(desc.params) == [v.ptr for v in p.values()] and (desc.batch, desc.d_ff) == (2, 6)
    p["p3"].strides = [1, 4]
    with pytest.raises(AssertionError):
        EncoderBlock._desc(block, plan)


@pytest.mark.parametrize("rank", [8, 9, 12])
def test_reshapes_of_many_axes_are_refused_by_the_library(rank):
    """Nine axes are no error of the call's form: the library refuses them (here, without a context, eight as well)."""
    x = View(torch.zeros(64, dtype=torch.uint8), "f32", (1,) * (rank - 1) + (2,), (2,) * rank)
    check = SimpleNamespace(lib=load_library())
    dev = SimpleNamespace(_f=_load_host(), _at=0, empty=lambda dtype, shape: x, _check=lambda code: Rocm._check(check, code))
    for call in (lambda: Rocm.reshape_forward(dev, x, (2,)), lambda: Rocm.reshape_backward(dev, x, x, x)):
        with pytest.raises(RocmError) as err:
            call()
        assert err.value.code == INVALID


@pytest.mark.parametrize("shape", [(1 << 32, 1 << 32), (1 << 62,), (1 << 21, 1 << 21, 1 << 21), (3, 1 << 62)])
def test_sizes_beyond_64_bits(shape):
    """No allocation of what is left of the product: 2^64 elements are not none."""
    host, like = _load_host(), View(torch.zeros(16, dtype=torch.uint8), "f32", shape, (1,) * len(shape))
    with pytest.raises(OverflowError):
        host.empty(View, 0, "f32", shape)
    with pytest.raises(OverflowError):
        host.carve(SimpleNamespace(ordinal=0, _at=0), View, None, [like], True)
    with pytest.raises(OverflowError):   # (each of them fits)
        host.carve(SimpleNamespace(ordinal=0, _at=0), View, None, [View(like.storage, "f64", (1 << 59,), (1,))] * 2, True)


def test_the_library_builds_without_python():
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dfdx_amd", "csrc")
    plan = lambda *args: subprocess.run(["make", "-n", "-B", "-C", csrc, *args], capture_output=True, text=True)
    with_python, without = plan(), plan("PYTHON=/nonexistent")
    assert with_python.returncode == without.returncode == 0
    assert "host.cpp" in with_python.stdout and "host.cpp" not in without.stdout and "libdfdx_rocm.so" in without.stdout
