"""Scans along an axis with kept axes after it, whose rows stream through LDS tiles: strips of 64 columns
and their ragged last groups, tiles' last rows, several strips per block, unaligned buffers, in place."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
import unpopped_amd as u
from unpopped_amd import _lib, forms as H, synth

pytestmark = pytest.mark.gpu
NT = {"F32": np.float32, "F64": np.float64, "I32": np.int32, "I64": np.int64}


def values(dtype, n):
    return synth.normal_f32(5, n).astype(NT[dtype]) if dtype[0] == "F" else synth.int16_i32(5, n).astype(NT[dtype])


@pytest.mark.parametrize("a,s,b", [(1, 16, 32), (3, 33, 63), (2, 64, 64), (1, 65, 65), (2, 129, 130), (1, 600, 67),
                                   (5, 700, 256), (300, 20, 33), (7, 40, 8001), (1, 15, 64), (2, 50, 31)])
@pytest.mark.parametrize("dtype,op,exclusive,reverse", [("F32", "Sum", False, False), ("F32", "Sum", True, True),
                                                        ("F32", "Mean", False, True), ("F32", "Max", True, False),
                                                        ("F64", "Sum", False, True), ("I32", "Sum", True, False),
                                                        ("I64", "Min", False, False)])
def test_every_prefix_is_the_serial_ones(hip_device, a, s, b, dtype, op, exclusive, reverse):
    """Bit-exact against the serial scan, at aligned and unaligned addresses and in place."""
    if op == "Mean" and dtype[0] == "I":
        pytest.skip("an integer Mean")
    x = values(dtype, a * s * b).reshape(a, s, b)
    rows = np.ascontiguousarray(np.moveaxis(x, 1, -1)).reshape(-1, s)
    want = np.ascontiguousarray(np.moveaxis(oracle.scan_rows(rows, op, exclusive, reverse).reshape(a, b, s), -1, 1))
    ex = H.executor(kind="scan", dtype=dtype, rank=3, op=op, axis=1, exclusive=exclusive, reverse=reverse)
    H.say(f"[case] column scan {a}x{s}x{b} {dtype} {op} exclusive={exclusive} reverse={reverse}")
    for shift in (0, x.itemsize):
        buf = u.DeviceBuffer(x.nbytes + 64)
        dst = u.DeviceBuffer(x.nbytes + 64)
        dst.fill(0x5A)
        buf.at(shift).upload(x)
        ex.launch(buf.at(shift), dst.at(shift), a, s, b)
        u.synchronize()
        assert np.array_equal(dst.at(shift).download(NT[dtype], x.size).reshape(x.shape), want, equal_nan=True)
        edge = dst.at(shift + x.nbytes).download(np.uint8, 64 - shift)
        assert (edge == 0x5A).all()
        ex.launch(buf.at(shift), buf.at(shift), a, s, b)
        u.synchronize()
        assert np.array_equal(buf.at(shift).download(NT[dtype], x.size).reshape(x.shape), want, equal_nan=True)


@pytest.mark.parametrize("dtype,reverse", [("F32", False), ("I32", True), ("I64", False)])
def test_in_place_with_a_last_strip_of_less_than_a_vector(hip_device, dtype, reverse):
    """257 strips over 256 blocks: the last one, a single column wide, runs after its neighbour has stored."""
    a, s, b = 1, 600, 64 * 256 + 1
    x = values(dtype, a * s * b).reshape(s, b)
    want = oracle.scan_rows(np.ascontiguousarray(x.T), "Sum", False, reverse).T
    ex = H.executor(kind="scan", dtype=dtype, rank=3, op="Sum", axis=1, exclusive=False, reverse=reverse)
    H.say(f"[case] column scan in place {a}x{s}x{b} {dtype} reverse={reverse}")
    buf = u.DeviceBuffer(x.nbytes)
    buf.upload(x)
    ex.launch(buf, buf, a, s, b)
    u.synchronize()
    assert np.array_equal(buf.download(NT[dtype], x.size).reshape(x.shape), want)


@pytest.mark.parametrize("grid,strips", [(250, 249), (252, 251), (256, 249), (7, 6), (250, 600)])
def test_every_strip_is_scanned_at_any_grid(hip_device, grid, strips):
    """The entry launched by hand on grids that are and are not multiples of the eight XCDs."""
    s, b = 16, 64 * strips
    x = values("I32", s * b).reshape(s, b)
    g = u.HipBackend().lower_kernel(H.kernel_for(kind="scan", dtype="I32", rank=3, op="Sum", axis=1))
    symbol = g.name + "_c"
    L, m, f, err = _lib.lib(), C.c_void_p(), C.c_void_p(), _lib.Error()
    co = u.HipCompiler().compile(g.source, g.name)
    img = C.create_string_buffer(co, len(co))
    _lib.check(L.unp_hip_module_load(img, len(co), C.byref(m), C.byref(err)), err)

    class Args(C.Structure):
        _fields_ = [("src", C.c_uint64), ("dst", C.c_uint64), ("S", C.c_int64), ("B", C.c_int64),
                    ("nstrips", C.c_int64), ("ncb", C.c_int64), ("wide", C.c_int32)]

    try:
        _lib.check(L.unp_hip_get_function(m, symbol.encode(), C.byref(f), C.byref(err)), err)
        src, dst = u.DeviceBuffer.from_array(x), u.DeviceBuffer(x.nbytes)
        dst.fill(0x5A)
        a = Args(src.ptr, dst.ptr, s, b, strips, strips, 1)
        H.say(f"[case] column scan by hand, {strips} strips on {grid} blocks")
        _lib.check(L.unp_hip_launch(f, (C.c_uint32 * 3)(grid, 1, 1), (C.c_uint32 * 3)(576, 1, 1), 0, None, C.byref(a),
                                    C.sizeof(a), C.byref(err)), err)
        u.synchronize()
        assert np.array_equal(dst.download(np.int32, x.size).reshape(s, b), np.cumsum(x, axis=0, dtype=np.int32))
    finally:
        L.unp_hip_module_unload(m)


# A strip per CU at most, two over 200 rows, four over 512, each at its last strip and the next; rows of half a
# strip; a last strip of less than a vector in place.
@pytest.mark.parametrize("a,s,b,in_place,tail", [
    (1, 16, 64 * 256, False, "_c"), (1, 16, 64 * 256 + 1, False, "_q"), (1, 199, 64 * 300, False, "_q"),
    (1, 200, 64 * 300, False, "_c"), (1, 200, 64 * 512, False, "_c"), (1, 200, 64 * 513, False, "_q"),
    (2, 512, 64 * 400, False, "_c"), (1, 511, 64 * 600, False, "_q"), (1, 512, 64 * 1025, False, "_q"),
    (1, 15, 64, False, "_q"), (1, 16, 32, False, "_c"), (1, 16, 31, False, "_q"), (300, 20, 33, False, "_q"),
    (1, 100, 65, False, "_c"), (1, 100, 65, True, "_q"), (1, 100, 68, True, "_c"),
])
def test_the_entry_follows_the_strips(hip_device, a, s, b, in_place, tail):
    x = values("I32", a * s * b).reshape(a, s, b)
    ex = H.executor(kind="scan", dtype="I32", rank=3, op="Sum", axis=1, exclusive=False, reverse=False)
    H.say(f"[case] column scan entry {a}x{s}x{b} in_place={in_place}")
    src = u.DeviceBuffer.from_array(x)
    dst = src if in_place else u.DeviceBuffer(x.nbytes)
    ex.launch(src, dst, a, s, b)
    u.synchronize()
    assert ex.last_launch()["entry"] == ex.kernel.name + tail
    assert np.array_equal(dst.download(np.int32, x.size).reshape(x.shape), np.cumsum(x, axis=1, dtype=np.int32))
