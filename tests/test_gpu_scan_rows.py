"""Scans of short rows in a wave's or a block's registers, and of unaligned long rows in whole vectors."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import unpopped_amd as u
from unpopped_amd import forms as H, synth

pytestmark = pytest.mark.gpu
NT = {"F32": np.float32, "F64": np.float64, "I32": np.int32, "I64": np.int64}


@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 3), (3000, 5), (9, 63), (2, 257), (700, 511), (3, 513), (2, 1023),
                                       (2, 1025), (600, 2047), (3, 4097), (2, 8191), (2, 8193), (2, 16383), (1, 16385),
                                       (3, 20003), (2, 70001)])
@pytest.mark.parametrize("dtype", ["F32", "F64", "I32", "I64"])
@pytest.mark.parametrize("op,exclusive,reverse", [("Sum", False, False), ("Sum", True, True), ("Max", True, False)])
def test_rows_of_any_length(hip_device, rows, cols, dtype, op, exclusive, reverse):
    """Whole numbers (every order is exact) at aligned and unaligned addresses, and in place."""
    x = (synth.int16_i32(11, rows * cols) - 7).astype(NT[dtype]).reshape(rows, cols)
    want = oracle.scan_rows(x, op, exclusive, reverse)
    ex = H.executor(kind="scan", dtype=dtype, rank=2, op=op, exclusive=exclusive, reverse=reverse)
    H.say(f"[case] row scan {rows}x{cols} {dtype} {op} exclusive={exclusive} reverse={reverse}")
    for shift in (0, x.itemsize):
        src, dst = u.DeviceBuffer(x.nbytes + 64), u.DeviceBuffer(x.nbytes + 64)
        dst.fill(0x5A)
        src.at(shift).upload(x)
        ex.launch(src.at(shift), dst.at(shift), rows, cols)
        ex.check()
        assert np.array_equal(dst.at(shift).download(NT[dtype], x.size).reshape(x.shape), want)
        assert (dst.at(shift + x.nbytes).download(np.uint8, 64 - shift) == 0x5A).all()
        ex.launch(src.at(shift), src.at(shift), rows, cols)
        ex.check()
        assert np.array_equal(src.at(shift).download(NT[dtype], x.size).reshape(x.shape), want)


@pytest.mark.parametrize("rows,cols", [(40, 700), (9, 15001), (3, 30001)])
def test_normal_values_keep_their_bits_and_the_bound(hip_device, rows, cols):
    x = synth.normal_f32(12, rows * cols).reshape(rows, cols)
    ex = H.executor(kind="scan", dtype="F32", rank=2, op="Sum")
    din, dout = u.DeviceBuffer.from_array(x), u.DeviceBuffer(x.nbytes)
    H.say(f"[case] row scan of normal values {rows}x{cols}")
    runs = []
    for _ in range(3):
        ex.launch(din, dout, rows, cols)
        ex.check()
        runs.append(dout.download(np.float32, x.size).reshape(x.shape))
    assert all(r.tobytes() == runs[0].tobytes() for r in runs)
    # Both folds are f64 sums of the prefix: each within gamma_(n-1) sum|x| of it, then one rounding.
    k = np.arange(cols) * 2.0**-53
    bound = 2 * (k / (1 - k)) * np.cumsum(np.abs(x.astype(np.float64)), axis=1)
    want = oracle.scan_rows(x, "Sum").astype(np.float64)
    assert (np.abs(runs[0].astype(np.float64) - want) <= bound + np.spacing(np.abs(runs[0])).astype(np.float64)).all()


# A wave's and a block's registers, the staged tiles, and the register tiles at one per CU and past it.
@pytest.mark.parametrize("dtype,rows,cols,tail", [
    ("I32", 3, 1024, "_r1"), ("I32", 3, 1025, "_r8"), ("I32", 3, 16384, "_r8"), ("I32", 3, 16388, "_v"),
    ("I32", 1, 16385, "_1_s"), ("I32", 128, 16385, "_1_s"), ("I32", 129, 16385, "_s"), ("I32", 1, 256 * 16384 - 1, "_1_s"),
    ("I32", 1, 256 * 16384 + 1, "_s"), ("F32", 1, 16385, "_s"), ("I64", 3, 8192, "_r8"), ("I64", 3, 8193, "_s"),
    ("I64", 3, 8194, "_v")])
def test_the_entry_follows_the_row(hip_device, dtype, rows, cols, tail):
    x = synth.int16_i32(13, rows * cols).astype(NT[dtype]).reshape(rows, cols)
    op = "Max" if dtype == "F32" else "Sum"
    H.say(f"[case] row scan entry {rows}x{cols} {dtype}")
    for reverse, exclusive in ((False, False), (True, True)):
        ex = H.executor(kind="scan", dtype=dtype, rank=2, op=op, reverse=reverse,
                        exclusive=exclusive)
        din, dout = u.DeviceBuffer.from_array(x), u.DeviceBuffer(x.nbytes)
        ex.launch(din, dout, rows, cols)
        ex.check()
        assert ex.last_launch()["entry"] == ex.kernel.name + tail
        want = oracle.scan_rows(x, op, exclusive, reverse)
        assert np.array_equal(dout.download(NT[dtype], x.size).reshape(x.shape), want)
