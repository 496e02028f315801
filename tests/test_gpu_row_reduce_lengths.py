"""Row reductions over rows of every kind of length: ragged rows in registers, rows in chunks with a launch
per stage, rows of chunks in one block; unaligned buffers, in place, and the same bits without a
workspace."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import unpopped_amd as u
from tests.test_gpu_parity import f64_order_tolerance, ulps
from unpopped_amd import expr as X, forms as H

pytestmark = pytest.mark.gpu


def ran(ex):
    """The last launch's entry, without the kernel's name."""
    return ex.last_launch()["entry"][len(ex.kernel.name):]


@pytest.mark.parametrize("rows,cols", [(3, 1), (5, 3), (4, 4), (3, 5), (2, 1023), (2300, 37), (3, 4095), (3, 4097),
                                       (2, 8191), (2, 8193), (600, 8195), (2, 16383), (2, 16385), (1, 50001),
                                       (3, 20480), (1, 300001), (520, 16388)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("which", ["softmax", "rms_norm"])
def test_rows_of_any_length(hip_device, rows, cols, dtype, which):
    stages, epi = getattr(X, which)()
    x = np.random.default_rng(41).normal(size=(rows, cols)).astype(dtype)
    want = oracle.row_reduce([x], stages, epi)
    ex = H.row_reduce_executor("F32" if dtype == np.float32 else "F64", 2, stages, epi)
    H.say(f"[case] row_reduce length {which} {rows}x{cols} {np.dtype(dtype).name}")

    def near(got):
        # F32: 2 ulps.  F64: 4 ulps, or what another order of the row's sum allows: the serial fold and
        # this one are each within gamma_(n-1) * sum|x| of the exact sum.
        if dtype == np.float32:
            return ulps(got, want).max() <= 2
        far = ulps(got, want) > 4
        return (np.abs(got - want)[far] <= f64_order_tolerance(x, want, which)[far]).all()

    for shift in (0, x.itemsize):
        src, dst = u.DeviceBuffer(x.nbytes + 64), u.DeviceBuffer(x.nbytes + 64)
        dst.fill(0x5A)
        src.at(shift).upload(x)
        ex.launch(src.at(shift), dst.at(shift), rows, cols)
        u.synchronize()
        got = dst.at(shift).download(dtype, x.size).reshape(x.shape)
        assert near(got)
        assert (dst.at(shift + x.nbytes).download(np.uint8, 64 - shift) == 0x5A).all()
        ex.launch_static(src.at(shift), dst.at(shift), rows, cols)
        u.synchronize()
        assert dst.at(shift).download(dtype, x.size).tobytes() == got.tobytes()
        ex.launch(src.at(shift), src.at(shift), rows, cols)  # in place
        u.synchronize()
        assert src.at(shift).download(dtype, x.size).tobytes() == got.tobytes()


def test_two_inputs_nan_and_infinities_in_chunks(hip_device):
    """Max and Sum stages over two inputs, in chunks, with a NaN row, an infinite one and one of the lowest
    values: the oracle's values, the NaNs where it has them."""
    r = np.random.default_rng(42)
    a, b = r.integers(-8, 9, (4, 20001)).astype(np.float32), r.integers(-8, 9, (4, 20001)).astype(np.float32)
    a[1, 19999], a[2, 5], a[3, :] = np.nan, np.inf, np.finfo(np.float32).min
    b[3, :] = 0
    stages = [(X.input(0) * X.input(1), "Sum"), (X.input(0) - X.reduced(0), "Max")]
    epi = X.fma(X.input(0), X.reduced(1), X.input(1) - X.reduced(0))
    H.say("[case] row_reduce chunks, two inputs, special values")
    with np.errstate(all="ignore"):
        want = oracle.row_reduce([a, b], stages, epi)
    assert np.array_equal(H.row_reduce([a, b], stages, epi), want, equal_nan=True)
    last = H.row_reduce_executor("F32", 2, stages, epi, n_inputs=2).last_launch()
    assert last["entry"].endswith("_p_v") and last["chunks"] == 5 and last["shared"]


@pytest.mark.parametrize("cols,entry", [(257, "_s"), (1281, "_s"), (2305, "_c4_s"), (4353, "_c_s"), (8193, "_c512_s")])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_in_place_on_an_input_only_the_epilogue_reads(hip_device, cols, entry, dtype):
    """Ragged rows whose shifted last vector begins a wave: the elements it shares are another wave's, which
    may have stored them before this one loads them."""
    if dtype == np.float64:
        cols = cols // 2 + 1  # the same vector of 2
    r = np.random.default_rng(43)
    rows = 700
    a, b = (r.integers(-8, 9, (rows, cols)).astype(dtype) for _ in range(2))
    stages = [(X.input(0), "Sum")]
    epi = X.input(1) * X.konst(3.0) + X.reduced(0)
    ex = H.row_reduce_executor(H.NP_KIND[dtype], 2, stages, epi, n_inputs=2)
    H.say(f"[case] row_reduce in place on the epilogue's input {rows}x{cols} {np.dtype(dtype).name}")
    da, db = u.DeviceBuffer.from_array(a), u.DeviceBuffer.from_array(b)
    ex.launch(da, db, db, rows, cols)
    u.synchronize()
    assert ran(ex) == entry
    assert np.array_equal(db.download(dtype, b.size).reshape(b.shape), oracle.row_reduce([a, b], stages, epi))


# The entry at the ends of every range, for a chain that keeps a stage's values (softmax) and one that does not.
@pytest.mark.parametrize("which,rows,cols,shift,entry", [
    ("softmax", 9, 3, 0, "_s"), ("softmax", 9, 447, 0, "_s"), ("softmax", 9, 448, 0, "_c4"), ("softmax", 9, 448, 4, "_c4_s"),
    ("softmax", 9, 449, 0, "_c4_s"), ("softmax", 9, 4096, 0, "_c4"), ("softmax", 9, 4095, 0, "_c4_s"),
    ("softmax", 9, 4097, 0, "_c_s"), ("softmax", 9, 4100, 0, "_c"), ("softmax", 9, 8191, 0, "_c_s"),
    ("softmax", 9, 8192, 0, "_c"), ("softmax", 9, 8196, 0, "_c512_v"), ("softmax", 9, 8195, 0, "_c512_s"),
    ("softmax", 9, 16384, 0, "_c512_v"), ("softmax", 9, 16384, 4, "_c512_s"), ("softmax", 9, 16385, 0, "_p_v"),
    ("softmax", 447, 16388, 0, "_p_v"), ("softmax", 448, 16388, 0, "_a_v"), ("softmax", 449, 16389, 4, "_a_v"),
    ("rms_norm", 9, 2047, 0, "_s"), ("rms_norm", 9, 2049, 0, "_c4_s"), ("rms_norm", 9, 2048, 4, "_c4_s"),
    ("rms_norm", 9, 64, 0, "_c4"), ("rms_norm", 9, 64, 4, "_s"), ("rms_norm", 3, 70001, 4, "_p_v"),
])
def test_the_entry_follows_the_length_and_the_alignment(hip_device, which, rows, cols, shift, entry):
    stages, epi = getattr(X, which)()
    x = np.random.default_rng(44).normal(size=(rows, cols)).astype(np.float32)
    ex = H.row_reduce_executor("F32", 2, stages, epi)
    H.say(f"[case] row_reduce entry {which} {rows}x{cols} +{shift}")
    src, dst = u.DeviceBuffer(x.nbytes + 64), u.DeviceBuffer(x.nbytes + 64)
    src.at(shift).upload(x)
    ex.launch(src.at(shift), dst.at(shift), rows, cols)
    u.synchronize()
    assert ran(ex) == entry
    assert ex.last_launch()["shared"] == (entry == "_p_v")
    few = slice(0, 9)
    assert ulps(dst.at(shift).download(np.float32, x.size).reshape(x.shape)[few], oracle.row_reduce([x[few]], stages, epi)).max() <= 2
