"""GPU checks of launches captured into a HIP graph from the context's stream.

Split products and split decode attention keep partial results in one array
per GPU, in the order of that stream.  A captured launch may be replayed on
another stream beside it, so it takes one workgroup per tile and no such array:
checked on the captured nodes' grids.  Replays run between eager calls of the
same products (split ones) and give the eager results up to a rounding.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rew_amd import _lib
from rew_amd import eager as E
from rew_amd import nn
from rew_amd.eager import DType


class Dim3(C.Structure):
    _fields_ = [("x", C.c_uint), ("y", C.c_uint), ("z", C.c_uint)]


class KernelNodeParams(C.Structure):
    _fields_ = [("block", Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", Dim3),
                ("params", C.c_void_p), ("shared", C.c_uint)]


def _ok(rc):
    assert rc == 0, f"HIP error {rc}"


def _capture(fn):
    """fn's launches as a graph: (replay, grid sizes, fn's results)."""
    hip = C.CDLL("libamdhip64.so")
    s = C.c_void_p()
    assert _lib.load().rew_mi355x_stream(E.context(), C.byref(s)) == 0
    E.sync()
    graph, ex, n = C.c_void_p(), C.c_void_p(), C.c_size_t()
    _ok(hip.hipStreamBeginCapture(s, 2))  # (relaxed: the allocator may allocate)
    try:
        out = fn()
        E.flush()
    finally:
        rc = hip.hipStreamEndCapture(s, C.byref(graph))
    _ok(rc)
    _ok(hip.hipGraphGetNodes(graph, None, C.byref(n)))
    nodes = (C.c_void_p * n.value)()
    _ok(hip.hipGraphGetNodes(graph, nodes, C.byref(n)))
    grids = []
    for node in nodes:
        p = KernelNodeParams()
        _ok(hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)))
        grids.append(p.grid.x)
    _ok(hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)))
    return lambda: _ok(hip.hipGraphLaunch(ex, s)), grids, out


def _bf16(r, shape, scale=1.0):
    return E.fromHost((r.standard_normal(shape) * scale).astype(np.float32), DType.BFLOAT16)


def _check(fn, split_label, grid):
    E.profileBegin()
    want = E.toHostF32(fn())
    names = [n for n, _, _ in E.profileEnd()]
    assert len(names) == 1 and split_label(names[0]), names
    keep = fn()  # (a block of the result's size returns to the allocator)
    E.sync()
    del keep
    replay, grids, out = _capture(fn)
    assert grids == [grid], grids
    first = None
    for _ in range(4):
        replay()
        eager = fn()
        np.testing.assert_array_equal(E.toHostF32(eager), want)
        got = E.toHostF32(out)
        assert np.linalg.norm(got - want) <= 4e-3 * np.linalg.norm(want)
        first = got if first is None else first
        np.testing.assert_array_equal(got, first)


def test_captured_products_are_not_split(gpu):
    r = np.random.default_rng(1)
    x, lin = _bf16(r, (8, 14336)), nn.Linear(_bf16(r, (14336, 256), 0.02), _bf16(r, (256,)))
    _check(lambda: lin.forward(x),
           lambda n: "_strip" in n and int(n.rsplit(" s", 1)[1]) > 1, 2)


def test_captured_decode_attention_is_not_split(gpu):
    r = np.random.default_rng(2)
    q, k, v = _bf16(r, (2, 4, 1, 128)), _bf16(r, (2, 4, 4000, 128)), _bf16(r, (2, 4, 4000, 128))
    _check(lambda: nn.scaledDotProductAttention(q, k, v), lambda n: n.startswith("flash_attn_dec"),
           8)
