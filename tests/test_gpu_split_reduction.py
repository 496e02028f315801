"""Reductions over axis sets whose positions are split over blocks: ragged runs, packed rows, chunks,
and the launch without a workspace, whose bits must be the split one's."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import unpopped_amd as u
from unpopped_amd import _lib, expr as X, forms as H, synth

pytestmark = pytest.mark.gpu

# (shape, reduced axes): the innermost run reduced (fewer elements than a vector, ragged, one and
# several reduced axes before it, few and many outputs), then kept (one column, packed rows, ragged
# strips, several reduced axes), with chunks and without.
CASES = [
    ((5, 7, 3), (0, 2)),
    ((9, 33, 49), (0, 2)),
    ((64, 3, 1027), (0, 2)),
    ((2, 5000, 17), (0, 2)),
    ((3, 2, 5, 4, 70), (0, 2, 4)),
    ((6, 1, 40, 1, 9), (0, 2, 4)),
    ((1000, 1), (0,)),
    ((3000, 3), (0,)),
    ((2111, 90), (0,)),
    ((700, 1030), (0,)),
    ((8, 300, 6, 258), (0, 2)),
    ((40000, 6), (0,)),
]


def data(shape, dtype):
    n = int(np.prod(shape))
    return synth.int16_i32(7, n).astype(dtype).reshape(shape)  # whole numbers: every order is exact


@pytest.mark.parametrize("shape,axes", CASES)
@pytest.mark.parametrize("dtype", ["F32", "F64", "I32", "I64"])
def test_sums_and_maxima_are_exact(hip_device, shape, axes, dtype):
    nt = {"F32": np.float32, "F64": np.float64, "I32": np.int32, "I64": np.int64}[dtype]
    x = data(shape, nt)
    H.say(f"[case] split reduction {shape} over {axes} {dtype}")
    want = x.astype(np.int64).sum(axis=axes).astype(nt)
    assert np.array_equal(H.reduce_axes(x, axes, "Sum"), want)
    assert np.array_equal(H.reduce_axes(x, axes, "Max"), x.max(axis=axes))


@pytest.mark.parametrize("shape,axes", CASES)
def test_two_inputs_a_body_and_a_post(hip_device, shape, axes):
    x, y = data(shape, np.float32), data(shape, np.float32)[::-1].copy()
    H.say(f"[case] split reduction with a body {shape} over {axes}")
    got = H.reduce_expr([x, y], axes, "Sum", X.input(0) * X.input(1), X.reduced(0) + X.konst(0.5))
    want = np.float32((x.astype(np.int64) * y.astype(np.int64)).sum(axis=axes)).astype(np.float64) + 0.5
    assert np.array_equal(got, want.astype(np.float32))


@pytest.mark.parametrize("shape,axes", [c for c in CASES if len(c[0]) > 2] + [((4000, 300), (0,))])
def test_without_a_workspace_the_bits_are_the_same(hip_device, shape, axes):
    """The no-allocation launch folds all chunks of an output in one block, and a second stream has a
    workspace of its own; on values whose sums round, only the same association gives the same bits."""
    x = synth.normal_f32(3, int(np.prod(shape))).reshape(shape)
    outs = int(np.prod([n for d, n in enumerate(shape) if d not in axes]))
    k = u.lift_reduction("r", "F32", len(shape), "Sum", axes=axes, launch=(256, 64), body=X.input(0) * X.konst(0.75),
                         post=X.reduced(0) * X.konst(3.0))
    ex = u.Executor(u.HipBackend().lower_kernel(k))
    din, a, b = u.DeviceBuffer.from_array(x), u.DeviceBuffer(outs * 4), u.DeviceBuffer(outs * 4)
    H.say(f"[case] split reduction without a workspace {shape} over {axes}")
    ex.launch(din, a, *shape)
    ex.launch_static(din, b, *shape)
    ex.check()
    want = a.download(np.uint32, outs)
    assert np.array_equal(b.download(np.uint32, outs), want)
    L, streams = _lib.lib(), []
    for _ in range(6):
        st = C.c_void_p()
        assert L.hipStreamCreate(C.byref(st)) == 0
        streams.append(st)
    got = [u.DeviceBuffer(outs * 4) for _ in streams]
    for st, o in zip(streams, got):
        ex.launch(din, o, *shape, stream=st.value)
    ex.check()
    for o in got:
        assert np.array_equal(o.download(np.uint32, outs), want)
    # Captured into a graph and replayed between eager launches.
    st, graph, exe = streams[0], C.c_void_p(), C.c_void_p()
    b.fill(0)
    assert L.hipStreamBeginCapture(st, 0) == 0
    ex.launch(din, b, *shape, stream=st.value)
    assert L.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert L.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        assert L.hipGraphLaunch(exe, st) == 0
        u.synchronize()
        assert np.array_equal(b.download(np.uint32, outs), want)
        b.fill(0)
        ex.launch(din, a, *shape, stream=st.value)
        ex.check()
    assert L.hipGraphExecDestroy(exe) == 0 and L.hipGraphDestroy(graph) == 0
    for st in streams:
        assert L.hipStreamDestroy(st) == 0


# (shape, reduced axes, the entry's tail): few positions under many outputs go a lane per output or vector
# of columns (fewer elements than a vector, ragged, one and several reduced axes, remainders of the eight
# in flight), strips of few rows a wave each.
SHORT = [
    ((100000, 3, 5), (1,), "mlv"), ((60000, 9, 3), (1,), "mls"), ((70000, 4, 6), (1,), "mlv"),
    ((3, 30000, 3, 7), (0, 2), "mlv"), ((13, 260001), (0,), "mlv"), ((70000, 1, 4), (1,), "mlv"),
    ((2, 100000, 2), (0, 2), "gls"), ((3, 60000, 5), (0, 2), "glv"), ((4, 100000, 8), (0, 2), "glv"),
    ((2, 300, 2, 300, 5), (0, 2, 4), "glv"), ((1, 90001, 9), (0, 2), None),
    ((1229, 59, 3), (1,), "mws"), ((1130, 47, 4), (1,), "mwv"), ((2000, 100, 7), (1,), "mwv"),
    ((4, 900, 10, 33), (0, 2), "mwv"), ((1000, 64, 17), (1,), "mwv"),
    ((1000, 1000, 4), (0, 2), "gwv"), ((2, 4096, 64), (0, 2), "gwv"),
]


@pytest.mark.parametrize("shape,axes,entry", SHORT)
@pytest.mark.parametrize("dtype", ["F32", "I64"])
def test_short_reductions_by_lanes_and_waves(hip_device, shape, axes, entry, dtype):
    nt = {"F32": np.float32, "I64": np.int64}[dtype]
    x = data(shape, nt)
    H.say(f"[case] short reduction {shape} over {axes} {dtype}")
    want = x.astype(np.int64).sum(axis=axes).astype(nt)
    assert np.array_equal(H.reduce_axes(x, axes, "Sum"), want)
    ran = H.executor(kind="reduction", dtype=dtype, rank=x.ndim, op="Sum", axes=axes, keepdim=False).last_launch()
    if dtype == "F32" and entry is not None:
        assert ran["entry"].rsplit("_", 1)[1] == entry
    got = H.reduce_expr([x, x], axes, "Sum", X.input(0) * X.input(1)) if dtype == "F32" else None
    if got is not None:
        assert np.array_equal(got, (x.astype(np.int64) ** 2).sum(axis=axes).astype(nt))
