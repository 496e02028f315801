"""Row folds over rows that are not whole aligned vectors, and over few long rows."""
from __future__ import annotations

import numpy as np
import pytest

import unpopped_amd as u
from unpopped_amd import forms as H, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(5, 1), (7, 2), (3, 3), (9, 5), (4000, 63), (600, 257), (3, 1027), (300, 4097),
                                       (256, 4096), (257, 4099), (2, 4095), (3, 8193), (1, 40001), (20, 32769)])
@pytest.mark.parametrize("dtype,nt", [("F32", np.float32), ("F64", np.float64), ("I32", np.int32), ("I64", np.int64)])
def test_sums_and_maxima_of_rows_of_any_length(hip_device, rows, cols, dtype, nt):
    x = (synth.int16_i32(9, rows * cols) - 9).astype(nt).reshape(rows, cols)  # whole numbers: exact in any order
    one = H.executor(kind="reduction", dtype=dtype, rank=2, op="Sum", reduced_from=1)
    two = H.executor(kind="row_reduce2", dtype=dtype, rank=2, op="Max", op1="Sum")
    want = x.astype(np.int64).sum(axis=1).astype(nt)
    H.say(f"[case] row fold {rows}x{cols} {dtype}")
    for shift in (0, x.itemsize):
        src = u.DeviceBuffer(x.nbytes + 64)
        src.at(shift).upload(x)
        s, m, t = (u.DeviceBuffer(rows * x.itemsize) for _ in range(3))
        one.launch(src.at(shift), s, rows, cols)
        two.launch(src.at(shift), m, t, rows, cols)
        u.synchronize()
        assert np.array_equal(s.download(nt, rows), want) and np.array_equal(t.download(nt, rows), want)
        assert np.array_equal(m.download(nt, rows), x.max(axis=1))


@pytest.mark.parametrize("rows,cols,shift,tail", [
    (7, 64, 0, "_wv"), (7, 64, 4, "_ws"), (7, 63, 0, "_ws"), (300, 4096, 0, "_wv"), (256, 4095, 0, "_ws"),
    (256, 4096, 0, "_bv"), (256, 4096, 4, "_bs"), (256, 4097, 0, "_bs"), (257, 4096, 0, "_wv"),
    (257, 32768, 0, "_wv"), (257, 32772, 0, "_bv"), (257, 32769, 0, "_bs")])
def test_the_entry_follows_the_rows(hip_device, rows, cols, shift, tail):
    x = (synth.int16_i32(9, rows * cols) - 9).astype(np.float32).reshape(rows, cols)
    ex = H.executor(kind="reduction", dtype="F32", rank=2, op="Sum", reduced_from=1)
    H.say(f"[case] row fold entry {rows}x{cols} +{shift}")
    src, dst = u.DeviceBuffer(x.nbytes + 64), u.DeviceBuffer(rows * 4)
    src.at(shift).upload(x)
    ex.launch(src.at(shift), dst, rows, cols)
    u.synchronize()
    assert ex.last_launch()["entry"] == ex.kernel.name + tail
    assert np.array_equal(dst.download(np.float32, rows), x.astype(np.int64).sum(axis=1).astype(np.float32))
