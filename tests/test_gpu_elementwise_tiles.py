"""Elementwise ops over permuted inputs in tiles of two axes: ragged tiles, inputs turned along the same
axis and along different ones, further axes, every element size."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import unpopped_amd as u
from tests.test_gpu_elementwise import run
from unpopped_amd import forms as H

pytestmark = pytest.mark.gpu


def I(k):  # noqa: E743
    return {"Input": k}


@pytest.mark.parametrize("shape,perms", [
    ((16, 16), [[0, 1], [1, 0]]), ((17, 63), [[1, 0], [1, 0]]), ((65, 130), [[0, 1], [1, 0], [1, 0]]),
    ((300, 15), [[0, 1], [1, 0]]), ((15, 300), [[0, 1], [1, 0]]), ((1, 70), [[0, 1], [1, 0]]),
    ((3, 5, 40, 66), [[0, 1, 2, 3], [0, 2, 1, 3]]), ((4, 33, 20, 70), [[0, 1, 2, 3], [0, 1, 3, 2], [3, 1, 2, 0]]),
    ((30, 1, 50, 20), [[3, 2, 1, 0], [0, 1, 2, 3]]), ((40, 24, 18), [[2, 0, 1], [1, 2, 0]]),
])
@pytest.mark.parametrize("dtype,nt", [("F32", np.float32), ("F64", np.float64), ("I32", np.int32)])
def test_permuted_inputs_by_tiles(hip_device, shape, perms, dtype, nt):
    r = np.random.default_rng(31)
    ins = []
    for p in perms:
        other = [0] * len(shape)
        for d, a in enumerate(p):
            other[a] = shape[d]
        ins.append((r.normal(size=other) * 100).astype(nt))
    body = I(0)
    for k in range(1, len(ins)):
        body = {"Sub": [body, I(k)]}
    k = u.lift_elementwise("tiles", dtype, len(shape), body, n_inputs=len(ins), perms=perms, launch=(256, 16))
    H.say(f"[case] elementwise tiles {shape} {perms} {dtype}")
    got, _ = run(k, ins, shape, nt)
    assert got.tobytes() == oracle.elementwise(ins, body, dtype, perms=perms).tobytes()


@pytest.mark.parametrize("dtype,nt", [("U8", np.uint8), ("Bf16", np.uint16), ("U32", np.uint32), ("I64", np.int64),
                                      ("Complex128", np.complex128)])
def test_a_transposition_moves_bits(hip_device, dtype, nt):
    r = np.random.default_rng(32)
    for rows, cols in ((64, 64), (100, 257), (16, 1000)):
        x = np.frombuffer(r.bytes(rows * cols * np.dtype(nt).itemsize), nt).reshape(cols, rows)
        k = u.lift_elementwise("turn", dtype, 2, I(0), n_inputs=1, perms=[[1, 0]], launch=(64, 4))
        H.say(f"[case] transposition {rows}x{cols} {dtype}")
        got, entry = run(k, [x], (rows, cols), nt)
        assert entry.endswith("_t_e") and got.tobytes() == np.ascontiguousarray(x.T).tobytes()


# (output shape, the second input's permutation): tiles mostly inside the extents, with ragged edges on
# either axis, the second axis turned or not, next to the first or not; then tiles mostly outside, and
# planes of fewer tiles than CUs.
ENTRIES = [
    ((65, 130), [1, 0], "_t_e"), ((130, 65), [1, 0], "_t_e"), ((300, 40), [1, 0], "_t_e"), ((16, 1000), [1, 0], "_t_e"),
    ((16, 20, 60, 40), [0, 2, 1, 3], "_t_e"), ((60, 300, 33), [1, 0, 2], "_t_e"), ((64, 300, 17), [2, 1, 0], "_t_e"),
    ((40, 33, 20, 70), [3, 1, 2, 0], "_t_e"), ((300, 60, 65), [1, 0, 2], "_t_e"), ((64, 300, 28), [1, 0, 2], "_t_e"),
    ((66, 300, 17), [2, 1, 0], "_e"), ((64, 300, 24), [1, 0, 2], "_e"), ((3, 5000), [1, 0], "_e"),
    ((5000, 17), [1, 0], "_e"), ((5000, 2, 16), [1, 0, 2], "_e"), ((5000, 2, 16), [0, 2, 1], "_e"),
    ((300, 3, 3, 65), [0, 2, 1, 3], "_e"), ((64, 2, 64), [1, 0, 2], "_e"),
]


@pytest.mark.parametrize("shape,perm,entry", ENTRIES)
def test_the_entry_follows_the_tiles_share_inside(hip_device, shape, perm, entry):
    r = np.random.default_rng(33)
    other = [0] * len(shape)
    for d, a in enumerate(perm):
        other[a] = shape[d]
    ins = [r.normal(size=shape).astype(np.float32), r.normal(size=other).astype(np.float32)]
    body = {"Sub": [I(0), I(1)]}
    k = u.lift_elementwise("tiles", "F32", len(shape), body, n_inputs=2, perms=[list(range(len(shape))), perm],
                           launch=(256, 16))
    H.say(f"[case] elementwise entry {shape} {perm}")
    got, ran = run(k, ins, shape, np.float32)
    assert np.array_equal(got, ins[0] - ins[1].transpose(perm))
    assert ran == u.HipBackend().lower_kernel(k).name + entry
