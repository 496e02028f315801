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


class Streams(list):
    """n HIP streams, destroyed at the end."""

    def __init__(self, n):
        for _ in range(n):
            st = C.c_void_p()
            assert _lib.lib().hipStreamCreate(C.byref(st)) == 0
            self.append(st)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        u.synchronize()
        for st in self:
            assert _lib.lib().hipStreamDestroy(st) == 0


FORMS = [("column", (4000, 300), (0,)), ("channel", (16, 8, 40000), (0, 2)), ("rows", (3, 60001), (1,))]


def fresh(kind, shape, axes):
    """An executor no launch has been made with yet."""
    if kind == "rows":
        stages, epi = X.softmax()
        k = u.lift_row_reduce("fresh", "F32", 2, stages, epi, launch=H.CALLER_LAUNCH)
    else:
        k = u.lift_reduction("fresh", "F32", len(shape), "Sum", axes=axes, launch=H.CALLER_LAUNCH)
    outs = int(np.prod(shape)) if kind == "rows" else int(np.prod([n for d, n in enumerate(shape) if d not in axes]))
    return u.Executor(u.HipBackend().lower_kernel(k)), outs


@pytest.mark.parametrize("kind,shape,axes", FORMS)
def test_first_launches_on_new_streams_allocate_nothing(hip_device, kind, shape, axes):
    """Made while another stream captures in global mode, where an allocation or a synchronisation is an error
    and ends the capture; each has a workspace, on streams past the executor's own ones too."""
    x = synth.normal_f32(3, int(np.prod(shape))).reshape(shape)
    L = _lib.lib()
    ex, outs = fresh(kind, shape, axes)
    din, first = u.DeviceBuffer.from_array(x), u.DeviceBuffer(outs * 4)
    u.synchronize()
    H.say(f"[case] split launches during another stream's capture: {kind}")
    with Streams(7) as streams:
        got = [u.DeviceBuffer(outs * 4) for _ in streams]
        assert L.hipStreamBeginCapture(streams[0], 0) == 0
        shared = []
        try:
            for st, o in list(zip(streams, got))[1:]:
                ex.launch(din, o, *shape, stream=st.value)
                shared.append((ex.last_launch()["shared"], ex.last_launch()["chunks"] > 1))
        finally:
            graph = C.c_void_p()
            ended = L.hipStreamEndCapture(streams[0], C.byref(graph))
        assert ended == 0 and shared == [(True, True)] * 6
        L.hipGraphDestroy(graph)
        ex.launch(din, first, *shape)
        ex.check()
        want = first.download(np.uint32, outs)
        for o in got[1:]:
            assert np.array_equal(o.download(np.uint32, outs), want)


@pytest.mark.parametrize("kind,shape,axes", FORMS)
def test_overlapping_launches_on_many_streams(hip_device, kind, shape, axes):
    """Seven streams and the per-thread one, each with its own input, launched on in turn without a wait."""
    L = _lib.lib()
    n = int(np.prod(shape))
    ex, outs = fresh(kind, shape, axes)
    xs = [u.DeviceBuffer.from_array(synth.normal_f32(60 + i, n)) for i in range(8)]
    got = [u.DeviceBuffer(outs * 4) for _ in xs]
    want = []
    for x, o in zip(xs, got):
        ex.launch(x, o, *shape)
        ex.check()
        want.append(o.download(np.uint32, outs))
        o.fill(0)
    u.synchronize()
    H.say(f"[case] overlapping split launches: {kind}")
    with Streams(7) as streams:
        handles = [st.value for st in streams] + [2]  # hipStreamPerThread
        for _ in range(10):
            for x, o, st in zip(xs, got, handles):
                ex.launch(x, o, *shape, stream=st)
                assert ex.last_launch()["shared"]
        ex.check()
    for o, w in zip(got, want):
        assert np.array_equal(o.download(np.uint32, outs), w)


def test_a_stream_per_request_keeps_its_workspace(hip_device):
    shape, axes = (4000, 300), (0,)
    ex, outs = fresh("column", shape, axes)
    x = u.DeviceBuffer.from_array(synth.normal_f32(3, int(np.prod(shape))))
    o = u.DeviceBuffer(outs * 4)
    ex.launch(x, o, *shape)
    ex.check()
    want = o.download(np.uint32, outs)
    H.say("[case] a stream per launch")
    for _ in range(20):
        o.fill(0)
        u.synchronize()
        with Streams(1) as (st,):
            ex.launch(x, o, *shape, stream=st.value)
            assert ex.last_launch()["shared"]
        assert np.array_equal(o.download(np.uint32, outs), want)


@pytest.mark.parametrize("kind,shape,axes", FORMS + [("body", (4000, 300), (0,))])
def test_a_no_allocation_launch_splits_in_the_static_scratch(hip_device, kind, shape, axes):
    x = u.DeviceBuffer.from_array(synth.normal_f32(3, int(np.prod(shape))))
    if kind == "body":
        ex, outs = H.reduce_expr_executor("F32", 2, "Sum", axes, X.input(0) * X.konst(0.75)), shape[1]
    else:
        ex, outs = fresh(kind, shape, axes)
    a, b = u.DeviceBuffer(outs * 4), u.DeviceBuffer(outs * 4)
    H.say(f"[case] static split launch: {kind}")
    ex.launch(x, a, *shape)
    for _ in range(2):
        b.fill(0)
        ex.launch_static(x, b, *shape)
        last = ex.last_launch()
        ex.check()
        assert last["shared"] and last["chunks"] > 1
        assert np.array_equal(b.download(np.uint32, outs), a.download(np.uint32, outs))


# Every lane layout of the strips: one column, fewer lanes than a wave, ragged, whole strips, several reduced
# axes, kept axes before the reduced one.
CAPTURED = [((40000, 1), (0,)), ((40000, 3), (0,)), ((40000, 6), (0,)), ((12158, 90), (0,)), ((9001, 37), (0,)),
            ((6000, 2050), (0,)), ((3, 20000, 22), (1,)), ((30, 2, 700, 2, 70), (0, 2))]


@pytest.mark.parametrize("body", [False, True])
@pytest.mark.parametrize("shape,axes", CAPTURED)
def test_captured_column_reductions_replay_to_the_same_bits(hip_device, shape, axes, body):
    """Captured once and replayed between eager launches: a plain one over one run of axes splits in a workspace
    of its own, the others fold all chunks of their columns in one block."""
    x = u.DeviceBuffer.from_array(synth.normal_f32(3, int(np.prod(shape))))
    outs = int(np.prod([n for d, n in enumerate(shape) if d not in axes]))
    if body:
        ex = H.reduce_expr_executor("F32", len(shape), "Sum", axes, X.input(0) * X.konst(0.75))
    else:
        ex, _ = fresh("column", shape, axes)
    L, a, b, graph, exe = _lib.lib(), u.DeviceBuffer(outs * 4), u.DeviceBuffer(outs * 4), C.c_void_p(), C.c_void_p()
    H.say(f"[case] captured column reduction {shape} over {axes} body={body}")
    ex.launch(x, a, *shape)
    ex.check()
    assert ex.last_launch()["shared"] and ex.last_launch()["chunks"] > 1
    want = a.download(np.uint32, outs)
    with Streams(1) as (st,):
        assert L.hipStreamBeginCapture(st, 0) == 0
        ex.launch(x, b, *shape, stream=st.value)
        assert ex.last_launch()["shared"] == (not body and len(axes) == 1)
        assert L.hipStreamEndCapture(st, C.byref(graph)) == 0
        assert L.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
        for _ in range(4):
            b.fill(0)
            u.synchronize()
            assert L.hipGraphLaunch(exe, st) == 0
            ex.launch(x, a, *shape)
            ex.check()
            assert np.array_equal(b.download(np.uint32, outs), want)
            assert np.array_equal(a.download(np.uint32, outs), want)
        assert L.hipGraphExecDestroy(exe) == 0 and L.hipGraphDestroy(graph) == 0
