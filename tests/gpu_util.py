"""Helpers shared by the GPU parity tests (imported only by tests marked ``gpu``)."""
from __future__ import annotations

import sys

import numpy as np

import oracle
from helpers import logical, rng


_dev = None


def device():
    """One Rocm context per test process; fails loudly when the HIP library is missing."""
    global _dev
    if _dev is None:
        from dfdx_amd import Rocm

        _dev = Rocm(0)
    return _dev


def announce(*what):
    """Name the case on stdout before touching the GPU, so a fault can be attributed."""
    print("[gpu-case]", *what, flush=True)
    sys.stdout.flush()


def launches(prepare):
    """Launches of the call that ``prepare(dev)`` returns, on a context of its own: the nodes of the graph it is captured into, behind
    one run by itself (so that the workspaces have their sizes)."""
    import torch

    from dfdx_amd import Rocm
    from test_gpu_encoder_block import graph_nodes

    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        run = prepare(own)
        run()
        own.synchronize()
        n = graph_nodes(run, stream)
        own.synchronize()
    del run
    own.close()
    return n


def make_operand(g, rows, cols, transposed, dtype, pad=0, scale=1.0, dist="normal"):
    """Storage + strides of a (rows, cols) matrix view; `transposed` stores it as (cols, rows)."""
    r, c = (cols, rows) if transposed else (rows, cols)
    ld = c + pad
    vals = g.standard_normal((r, ld)) if dist == "normal" else g.uniform(-1.0, 1.0, (r, ld))
    st = oracle.to_storage((vals * scale).reshape(-1), dtype)
    strides = (1, ld) if transposed else (ld, 1)
    return st, strides


def values(st, dtype, shape, strides, offset=0):
    return logical(oracle.to_f64(st, dtype), shape, strides, offset)
