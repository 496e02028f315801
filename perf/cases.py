"""The work that programs give this backend, as cases that can be timed and compared.

Every case lowers a KernelFn with ``Backend::lower_kernel``, keeps the executor, and launches it on
buffers that lie in HBM: ``prepare`` makes the buffers and the executor, ``run`` is one launch.  The
tensors are torch's; a launch takes their addresses.  A case is

* ``kind``: which form of the backend it is (the functions ``_fold`` .. ``_elementwise`` below);
* its extents and element type, and the options of that form.
"""
from __future__ import annotations

import math

import torch

import unpopped_amd as u
from unpopped_amd import expr as X
from unpopped_amd import forms as H

TORCH = {"F32": torch.float32, "F64": torch.float64, "I32": torch.int32, "I64": torch.int64}
SIZE = {"F32": 4, "F64": 8, "I32": 4, "I64": 8}
MOST = 1 << 25  # elements of the largest drawn input


class Held(u.DeviceBuffer):
    """A tensor's memory as a launch argument; the tensor owns it."""

    def __init__(self, t: torch.Tensor):
        self.nbytes, self.ptr, self._owner = t.numel() * t.element_size(), t.data_ptr(), t


_kept: dict = {}


def _executor(key, make) -> u.Executor:
    """A program lowers a kernel once and keeps its executor."""
    if key not in _kept:
        _kept[key] = u.Executor(H._backend.lower_kernel(make()))
    return _kept[key]


# ---------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # The fold pair ahead of a softmax over a small batch's logits: a small call, where the
        # launch itself counts.
        {"name": "row_fold_small", "kind": "fold2", "rows": 96, "cols": 1000},
        # Batch-norm statistics: the mean of each channel of an image batch, over three axes of four.
        {"name": "channel_mean", "kind": "channel", "n": 32, "c": 256, "hw": 784, "op": "Mean", "dtype": "F32"},
        # The 2-norm of each column of a weight matrix of odd extents: a pre-map and a fused post
        # around an outer-axis sum.
        {"name": "column_norm", "kind": "column", "rows": 6000, "cols": 2050, "op": "Sum", "norm": True, "dtype": "F32"},
        # RMS norm over the hidden size of a training batch.
        {"name": "rms_norm", "kind": "rms_norm", "rows": 8192, "cols": 4096},
        # Softmax over a vocabulary of odd size for a decode batch: few rows, long ones.
        {"name": "softmax_logits", "kind": "softmax", "rows": 64, "cols": 50001},
        # A large prefix sum of one sequence (sampling, stream compaction).
        {"name": "prefix_sum", "kind": "scan", "rows": 1, "cols": 1 << 26, "dtype": "F32", "exclusive": False,
         "reverse": False},
        # A running sum over time steps, every feature by itself: the scanned axis is the outer one.
        {"name": "running_sum_steps", "kind": "scan_axis", "a": 1, "s": 2048, "b": 3000, "dtype": "F32",
         "exclusive": False, "reverse": False},
        # An embedding lookup with skewed ids.
        {"name": "embedding", "kind": "gather", "table": 131072, "n": 16384, "d": 4096, "index": "I32"},
        # A whole int4 weight to bf16.
        {"name": "dequant_weight", "kind": "dequant", "rows": 8192, "cols": 28672, "group": 128},
        # The int4 weight times a decode batch's activations.
        {"name": "gemm_decode", "kind": "gemm", "r": 8192, "k": 28672, "c": 16, "group": 128, "x": "I8"},
        # The same weight times a prefill's.
        {"name": "gemm_prefill", "kind": "gemm", "r": 8192, "k": 28672, "c": 1024, "group": 128, "x": "I8"},
        # A matrix plus another's transpose: an elementwise op that reads one input through a permutation.
        {"name": "transposed_add", "kind": "elementwise", "shape": "4096,3000", "perm": "1,0", "dtype": "F32"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _pair(rng, lo0, hi0, lo1, hi1, most=MOST):
    while True:
        a, b = _log(rng, lo0, hi0), _log(rng, lo1, hi1)
        if a * b <= most:
            return a, b


def draw(rng) -> dict:
    """One more case: any form, over the range of sizes, types and options that the listed ones stand for."""
    kind = rng.choice(["fold", "fold2", "channel", "column", "rms_norm", "softmax", "scan", "scan_axis", "gather",
                       "dequant", "gemm", "elementwise"])
    whole = rng.random() < 0.5  # extents of whole 16-byte vectors, as weights and hidden sizes have

    def width(v: int, by: int = 64) -> int:
        return max(by, v // by * by) if whole else v

    if kind == "fold":
        rows, cols = _pair(rng, 1, 65536, 16, 262144)
        return {"kind": kind, "rows": rows, "cols": width(cols), "op": rng.choice(["Sum", "Max", "Mean"]),
                "dtype": rng.choice(["F32", "F32", "F64"])}
    if kind == "fold2":
        rows, cols = _pair(rng, 1, 16384, 64, 131072)
        return {"kind": kind, "rows": rows, "cols": width(cols)}
    if kind == "channel":
        while True:
            n, c, side = _log(rng, 1, 128), _log(rng, 3, 1024), rng.choice([7, 14, 20, 28, 56, 112])
            if n * c * side * side <= MOST:
                return {"kind": kind, "n": n, "c": c, "hw": side * side, "op": rng.choice(["Mean", "Sum", "Max"]),
                        "dtype": "F32"}
    if kind == "column":
        rows, cols = _pair(rng, 32, 65536, 32, 16384)
        norm = rng.random() < 0.5
        return {"kind": kind, "rows": rows, "cols": width(cols), "norm": norm,
                "op": "Sum" if norm else rng.choice(["Sum", "Max"]),
                "dtype": "F32" if norm else rng.choice(["F32", "I32"])}
    if kind == "rms_norm":
        rows, cols = _pair(rng, 1, 16384, 64, 16384)
        return {"kind": kind, "rows": rows, "cols": width(cols)}
    if kind == "softmax":
        rows, cols = _pair(rng, 1, 16384, 64, 131072)
        return {"kind": kind, "rows": rows, "cols": width(cols)}
    if kind == "scan":
        rows, cols = _pair(rng, 1, 4096, 256, MOST)
        return {"kind": kind, "rows": rows, "cols": width(cols), "dtype": rng.choice(["F32", "I32", "I64"]),
                "exclusive": rng.random() < 0.3, "reverse": rng.random() < 0.3}
    if kind == "scan_axis":
        while True:
            a, s, b = _log(rng, 1, 32), _log(rng, 16, 8192), _log(rng, 64, 8192)
            if a * s * b <= MOST:
                return {"kind": kind, "a": a, "s": s, "b": width(b), "dtype": rng.choice(["F32", "F32", "I32"]),
                        "exclusive": rng.random() < 0.3, "reverse": rng.random() < 0.3}
    if kind == "gather":
        n, d = _pair(rng, 64, 65536, 32, 8192, 1 << 26)
        return {"kind": kind, "table": _log(rng, 1024, 65536), "n": n, "d": width(d, 8),
                "index": rng.choice(["I32", "I64"])}
    if kind == "dequant":
        group = rng.choice([32, 64, 128])
        r, g = _pair(rng, 64, 8192, 4, 28672 // group, (1 << 27) // group)
        return {"kind": kind, "rows": r, "cols": g * group, "group": group}
    if kind == "gemm":
        group = rng.choice([64, 128, 128])
        while True:
            r, g, c = _log(rng, 512, 8192), _log(rng, 16, 28672 // group), _log(rng, 1, 1024)
            x = rng.choice(["I8", "I8", "I32"])
            if r * g * group * c * (4 if x == "I32" else 1) <= 1 << 37:
                return {"kind": kind, "r": r, "k": g * group, "c": c, "group": group, "x": x}
    # Elementwise: a sum of two inputs, the second as it lies, transposed, or with its heads moved.
    dtype = rng.choice(["F32", "I32"])
    how = rng.choice(["plain", "transposed", "heads"])
    if how == "heads":
        b, s, h, d = _log(rng, 1, 8), _log(rng, 16, 4096), _log(rng, 4, 64), rng.choice([64, 80, 128])
        while b * s * h * d > MOST:
            s = max(1, s // 2)
        return {"kind": "elementwise", "shape": f"{b},{h},{s},{d}", "perm": "0,2,1,3", "dtype": dtype}
    rows, cols = _pair(rng, 16, 16384, 16, 16384)
    return {"kind": "elementwise", "shape": f"{rows},{width(cols)}", "perm": "1,0" if how == "transposed" else "0,1",
            "dtype": dtype}


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, shape, dtype="F32") -> torch.Tensor:
    """Activations or weights: standard normal; whole numbers of a count's size for the integer types."""
    if dtype in ("I32", "I64"):
        return torch.randint(-1000, 1000, shape, generator=gen, device="cuda", dtype=TORCH[dtype])
    return torch.randn(shape, generator=gen, device="cuda", dtype=TORCH[dtype])


def _shape(case) -> tuple:
    return tuple(int(v) for v in case["shape"].split(","))


def _perm(case) -> tuple:
    return tuple(int(v) for v in case["perm"].split(","))


def _inputs(case: dict, seed: int) -> list:
    """The input tensors of a case, from the seed alone."""
    gen, kind = _gen(seed), case["kind"]
    if kind in ("fold", "column"):
        return [_normal(gen, (case["rows"], case["cols"]), case["dtype"])]
    if kind in ("fold2", "rms_norm", "softmax"):
        x = _normal(gen, (case["rows"], case["cols"]))
        return [x * 3.0 if kind == "softmax" else x]
    if kind == "channel":
        return [_normal(gen, (case["n"], case["c"], case["hw"]), case["dtype"])]
    if kind == "scan":
        shape = (case["rows"], case["cols"])
        if case["dtype"] == "F32":  # weights of a distribution
            return [torch.rand(shape, generator=gen, device="cuda").square_()]
        return [torch.randint(0, 16, shape, generator=gen, device="cuda", dtype=TORCH[case["dtype"]])]
    if kind == "scan_axis":
        return [_normal(gen, (case["a"], case["s"], case["b"]), case["dtype"])]
    if kind == "gather":
        table = torch.randn((case["table"], case["d"]), generator=gen, device="cuda", dtype=torch.bfloat16)
        # Ranks spread over their logarithm (few tokens make up most of a text), in shuffled order.
        rank = torch.rand(case["n"], generator=gen, device="cuda", dtype=torch.float64).mul_(math.log(case["table"])).exp_()
        order = torch.randperm(case["table"], generator=gen, device="cuda")
        ids = order[rank.long().clamp_(0, case["table"] - 1)]
        return [table, ids.to(TORCH[case["index"]])]
    if kind == "dequant":
        r, c, g = case["rows"], case["cols"], case["group"]
        q = torch.randint(0, 256, (r * c // 2,), generator=gen, device="cuda", dtype=torch.uint8)
        s = torch.rand(r * (c // g), generator=gen, device="cuda").mul_(0.019).add_(0.001).half()
        z = torch.randint(0, 256, ((r * (c // g) + 1) // 2,), generator=gen, device="cuda", dtype=torch.uint8)
        return [q, s, z]
    if kind == "gemm":
        r, k, c, ng = case["r"], case["k"], case["c"], case["k"] // case["group"]
        w = torch.randint(0, 256, (r * k // 2,), generator=gen, device="cuda", dtype=torch.uint8)
        zero = torch.randint(0, 16, (r, ng), generator=gen, device="cuda", dtype=torch.int32)
        scale = torch.randint(-800, 801, (r, ng), generator=gen, device="cuda", dtype=torch.int32)
        if case["x"] == "I8":
            x = torch.randint(-128, 128, (k, c), generator=gen, device="cuda", dtype=torch.int8)
        else:
            x = torch.randint(-30000, 30001, (k, c), generator=gen, device="cuda", dtype=torch.int32)
        return [w, zero, scale, x]
    shape, perm = _shape(case), _perm(case)
    other = [0] * len(shape)
    for d, p in enumerate(perm):
        other[p] = shape[d]
    return [_normal(gen, shape, case["dtype"]), _normal(gen, tuple(other), case["dtype"])]


def prepare(case: dict, seed: int) -> dict:
    """The inputs, the output buffers and the executor that a program holds before the call."""
    kind, ins = case["kind"], _inputs(case, seed)

    def empty(shape, like):
        return torch.empty(shape, device="cuda", dtype=like.dtype if isinstance(like, torch.Tensor) else like)

    if kind == "fold":
        ex = H.executor(kind="reduction", dtype=case["dtype"], rank=2, op=case["op"], reduced_from=1)
        outs, extents = [empty(case["rows"], ins[0])], (case["rows"], case["cols"])
    elif kind == "fold2":
        ex = H.executor(kind="row_reduce2", dtype="F32", rank=2, op="Sum", op1="Max", reduced_from=1)
        outs, extents = [empty(case["rows"], ins[0]), empty(case["rows"], ins[0])], (case["rows"], case["cols"])
    elif kind == "channel":
        # The image's two axes are walked as one: the same memory, the same sums.
        ex = H.executor(kind="reduction", dtype=case["dtype"], rank=3, op=case["op"], axes=(0, 2))
        outs, extents = [empty(case["c"], ins[0])], (case["n"], case["c"], case["hw"])
    elif kind == "column":
        if case["norm"]:
            ex = H.reduce_expr_executor(case["dtype"], 2, case["op"], (0,), X.input(0) * X.input(0),
                                        X.reduced(0).sqrt())
        else:
            ex = H.executor(kind="reduction", dtype=case["dtype"], rank=2, op=case["op"], axes=(0,))
        outs, extents = [empty(case["cols"], ins[0])], (case["rows"], case["cols"])
    elif kind in ("rms_norm", "softmax"):
        stages, epilogue = getattr(X, kind)()
        ex = H.row_reduce_executor("F32", 2, stages, epilogue)
        outs, extents = [empty(ins[0].shape, ins[0])], (case["rows"], case["cols"])
    elif kind == "scan":
        ex = H.executor(kind="scan", dtype=case["dtype"], rank=2, op="Sum", exclusive=case["exclusive"],
                        reverse=case["reverse"])
        outs, extents = [empty(ins[0].shape, ins[0])], (case["rows"], case["cols"])
    elif kind == "scan_axis":
        ex = H.executor(kind="scan", dtype=case["dtype"], rank=3, op="Sum", axis=1, exclusive=case["exclusive"],
                        reverse=case["reverse"])
        outs, extents = [empty(ins[0].shape, ins[0])], (case["a"], case["s"], case["b"])
    elif kind == "gather":
        ex = H.executor(kind="gather", dtype="Bf16", rank=2, index_dtype=case["index"], oob="ZeroFill")
        outs, extents = [empty((case["n"], case["d"]), ins[0])], (case["n"], case["d"], case["table"])
    elif kind == "dequant":
        ex = H.executor(kind="dequant4", q_kind="U4", z_kind="U4", group=case["group"], out_kind="Bf16")
        outs, extents = [empty((case["rows"], case["cols"]), torch.bfloat16)], (case["rows"], case["cols"])
    elif kind == "gemm":
        ex = H.executor(kind="dequant_gemm", q_kind="U4", dtype=case["x"], group=case["group"])
        outs, extents = [empty((case["r"], case["c"]), torch.int32)], (case["r"], case["k"], case["c"])
    else:
        shape, perm = _shape(case), _perm(case)
        ident = list(range(len(shape)))
        ex = _executor(("elementwise", case["dtype"], perm), lambda: u.lift_elementwise(
            "add", case["dtype"], len(shape), X.input(0) + X.input(1), n_inputs=2, perms=[ident, list(perm)],
            launch=H.CALLER_LAUNCH))
        outs, extents = [empty(shape, ins[0])], shape
    return {"ex": ex, "args": [Held(t) for t in ins + outs] + [int(v) for v in extents], "outs": outs}


def run(state: dict):
    """One launch; the outputs are the program's own buffers."""
    state["ex"].launch(*state["args"])
    outs = state["outs"]
    return outs[0] if len(outs) == 1 else outs


def _elements(case: dict) -> int:
    kind = case["kind"]
    if kind == "channel":
        return case["n"] * case["c"] * case["hw"]
    if kind == "scan_axis":
        return case["a"] * case["s"] * case["b"]
    if kind == "elementwise":
        return math.prod(_shape(case))
    return case["rows"] * case["cols"]


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "gather":
        # Every output row is written once, and the rows that the ids name are read once each: at most
        # one per id, and no more than the table has.
        row = case["d"] * 2
        return {"bytes": case["n"] * (row + SIZE[case["index"]]) + min(case["n"], case["table"]) * row, "flops": 0}
    if kind == "dequant":
        n, groups = case["rows"] * case["cols"], case["rows"] * (case["cols"] // case["group"])
        return {"bytes": n // 2 + groups * 2 + (groups + 1) // 2 + n * 2, "flops": 2 * n}
    if kind == "gemm":
        r, k, c = case["r"], case["k"], case["c"]
        xb = 1 if case["x"] == "I8" else 4
        return {"bytes": r * k // 2 + r * (k // case["group"]) * 8 + k * c * xb + r * c * 4, "flops": 2 * r * k * c}
    n, size = _elements(case), SIZE[case.get("dtype", "F32")]
    if kind in ("fold", "fold2"):
        return {"bytes": n * size + case["rows"] * size * (2 if kind == "fold2" else 1), "flops": n}
    if kind == "channel":
        return {"bytes": (n + case["c"]) * size, "flops": n}
    if kind == "column":
        return {"bytes": (n + case["cols"]) * size, "flops": 2 * n if case["norm"] else n}
    if kind == "elementwise":
        return {"bytes": 3 * n * size, "flops": n}
    # scans and row norms: read once, written once
    return {"bytes": 2 * n * size, "flops": 4 * n if kind in ("rms_norm", "softmax") else n}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("gather", "dequant", "gemm") or case.get("dtype") in ("I32", "I64") or case.get("op") == "Max":
        return "exact"
    if case.get("dtype") == "F64":
        # Sums of 64-bit values in another order (the values have both signs, so a sum is small
        # beside what went into it).
        return {"rel": 1e-13, "max": 1e-12}
    if kind in ("rms_norm", "softmax"):
        # A fold rounded once to 32 bits and an output rounded once over it.
        return {"rel": 2.5e-7, "max": 1e-6}
    if kind == "elementwise":
        return {"rel": 1e-8, "max": 1e-7}  # one rounding: the same everywhere
    # Sums in 64 bits, rounded once to 32.
    return {"rel": 1.2e-7, "max": 2.4e-7}


def exact(case: dict, seed: int):
    """What `run` returns, from plain torch in 64 bits; None where the outputs are whole numbers or moved bytes."""
    kind = case["kind"]
    if kind in ("gather", "dequant", "gemm") or case.get("dtype") in ("I32", "I64"):
        return None
    ins = [t.double() for t in _inputs(case, seed)]
    x = ins[0]
    if kind == "fold":
        return {"Sum": x.sum, "Mean": x.mean, "Max": x.amax}[case["op"]](1)
    if kind == "fold2":
        return [x.sum(1), x.amax(1)]
    if kind == "channel":
        y = x.transpose(0, 1).reshape(case["c"], -1)
        return {"Sum": y.sum, "Mean": y.mean, "Max": y.amax}[case["op"]](1)
    if kind == "column":
        if case["norm"]:
            return (x * x).sum(0).sqrt()
        return x.sum(0) if case["op"] == "Sum" else x.amax(0)
    if kind == "rms_norm":
        return x / ((x * x).mean(1, keepdim=True) + 1.0e-3).sqrt()
    if kind == "softmax":
        return torch.softmax(x, 1)
    if kind in ("scan", "scan_axis"):
        y = x.flip(1) if case["reverse"] else x
        got = torch.cumsum(y, 1)
        if case["exclusive"]:
            got = torch.cat([torch.zeros_like(got[:, :1]), got[:, :-1]], 1)
        return got.flip(1) if case["reverse"] else got
    return x + ins[1].permute(_perm(case))
