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
