"""What a program on this library spends its time in, as measurable cases.

Ten kinds of array program, each over a range of sizes, element types and
options: small host-resident calls, fused and single elementwise operations,
reductions, per-column statistics, prefix sums, a fused expression with a row
sum, matrix products, sorting with the indexing that goes with it, and a
least-squares fit.  ``listed`` names twelve of them, ``draw`` gives others of
the same ranges.

Inputs are made from the seed alone and handed over as a program would hold
them: NumPy arrays where the call starts on the host, device arrays
elsewhere.  Device results are returned as torch views of the library's own
memory, so that returning them copies nothing.
"""
from __future__ import annotations

import numpy as np
import torch

import macmetalpy_amd as cp

_TORCH = {"float16": torch.float16, "float32": torch.float32, "float64": torch.float64,
          "int32": torch.int32}
_ITEM = {"float16": 2, "float32": 4, "float64": 8, "int32": 4}


# ------------------------------------------------------------------ cases
def listed():
    return [
        # A script's many little calls: arrays of a thousand values that come
        # from the host, three results that go back there.
        {"name": "small_host_1k", "kind": "small_host", "n": 1000},
        # The fused expression at an everyday size, where the launch counts.
        {"name": "fused_1m", "kind": "fused", "n": 1 << 20, "dtype": "float32"},
        # Streaming operations one by one, far larger than any cache, with a
        # length that no vector width divides.
        {"name": "binary_100m", "kind": "binary", "n": 99_999_999},
        # Reductions of a big matrix in every direction, rows of odd length.
        {"name": "reduce_10k", "kind": "reduce", "rows": 10_000, "cols": 10_001,
         "dtype": "float32"},
        # A table of samples: mean and deviation of every column, then the
        # standardised table.  Few columns, many rows.
        {"name": "columns_2m_x_50", "kind": "columns", "rows": 2_000_000, "cols": 50,
         "dtype": "float32"},
        # Prefix sums: of everything, down the columns and along the rows.
        {"name": "scan_50m", "kind": "scan", "rows": 10_000, "cols": 5000},
        # Eight operations and a row sum with a broadcast row vector.
        {"name": "chain_8k", "kind": "chain", "rows": 8192, "cols": 8192},
        # A dense product of sizes that no tile divides.
        {"name": "matmul_f32_ragged", "kind": "matmul", "batch": 1, "m": 3000, "n": 2500,
         "k": 2001, "dtype": "float32"},
        # The largest product, in half precision.
        {"name": "matmul_f16_8k", "kind": "matmul", "batch": 1, "m": 8192, "n": 8192,
         "k": 8192, "dtype": "float16"},
        # Many small products.
        {"name": "matmul_batched_500", "kind": "matmul", "batch": 500, "m": 120, "n": 100,
         "k": 90, "dtype": "float32"},
        # Ordering a table by a key and filtering it.
        {"name": "sort_16m", "kind": "sort", "n": 16_000_000, "dtype": "float32"},
        # Linear regression by the normal equations, in double precision.
        {"name": "least_squares_500", "kind": "lsq", "rows": 100_000, "cols": 500,
         "dtype": "float64"},
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("small_host", "fused", "binary", "reduce", "columns", "scan", "chain",
                       "matmul", "matmul", "sort", "lsq"))
    if kind == "small_host":
        return {"kind": kind, "n": _log(rng, 16, 50_000)}
    if kind == "fused":
        return {"kind": kind, "n": _log(rng, 70_000, 100_000_000),
                "dtype": rng.choice(("float32", "float32", "float64", "float16"))}
    if kind == "binary":
        return {"kind": kind, "n": _log(rng, 70_000, 99_000_000)}
    if kind == "reduce":
        rows = _log(rng, 100, 300_000)
        return {"kind": kind, "rows": rows, "cols": _log(rng, 100, 100_000_000 // rows),
                "dtype": rng.choice(("float32", "float32", "float16", "int32"))}
    if kind == "columns":
        cols = _log(rng, 8, 1000)
        return {"kind": kind, "rows": _log(rng, 30_000, 100_000_000 // cols), "cols": cols,
                "dtype": rng.choice(("float32", "float32", "float64"))}
    if kind == "scan":
        rows = _log(rng, 100, 100_000)
        return {"kind": kind, "rows": rows, "cols": _log(rng, 700, 50_000_000 // min(rows, 50_000))}
    if kind == "chain":
        rows = _log(rng, 100, 100_000)
        return {"kind": kind, "rows": rows, "cols": _log(rng, 700, 60_000_000 // rows)}
    if kind == "matmul":
        shape = rng.choice(("dense", "dense", "batched", "vector"))
        dtype = rng.choice(("float32", "float32", "float16", "float64"))
        if shape == "batched":
            c = {"batch": _log(rng, 8, 2000), "m": _log(rng, 8, 300), "n": _log(rng, 8, 300),
                 "k": _log(rng, 8, 300)}
        elif shape == "vector":
            c = {"batch": 1, "m": _log(rng, 300, 20_000), "n": 1, "k": _log(rng, 300, 20_000)}
        else:
            c = {"batch": 1, "m": _log(rng, 64, 5000), "n": _log(rng, 64, 5000),
                 "k": _log(rng, 64, 5000)}
        return {"kind": kind, **c, "dtype": dtype}
    if kind == "sort":
        return {"kind": kind, "n": _log(rng, 70_000, 16_000_000),
                "dtype": rng.choice(("float32", "float32", "int32", "float64"))}
    cols = _log(rng, 4, 500)
    return {"kind": "lsq", "rows": _log(rng, max(2000, 4 * cols), 50_000_000 // cols), "cols": cols,
            "dtype": rng.choice(("float64", "float32"))}


# ----------------------------------------------------------------- inputs
def _inputs(case, seed):
    """The case's inputs by name, as torch tensors on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, dtype="float32"):
        f = torch.float64 if dtype == "float64" else torch.float32
        return torch.randn(*shape, generator=g, device="cuda", dtype=f).to(_TORCH[dtype])

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32)

    kind = case["kind"]
    if kind == "small_host":
        return {"x": normal(case["n"]), "y": normal(case["n"])}
    if kind == "fused":
        return {"x": normal(case["n"], dtype=case["dtype"])}
    if kind == "binary":
        n = case["n"]
        return {"a": normal(n), "b": normal(n), "i": ints(-2 ** 30, 2 ** 30, n),
                "j": ints(1, 1001, n) * (2 * ints(0, 2, n) - 1)}
    if kind == "reduce":
        shape = (case["rows"], case["cols"])
        return {"x": ints(-1000, 1000, *shape) if case["dtype"] == "int32"
                else normal(*shape, dtype=case["dtype"])}
    if kind == "columns":
        d = case["cols"]
        scale = torch.linspace(0.5, 20.0, d, device="cuda")
        x = normal(case["rows"], d, dtype=case["dtype"])
        return {"x": (x * scale + 3.0 * scale).to(_TORCH[case["dtype"]])}
    if kind == "scan":
        shape = (case["rows"], case["cols"])
        return {"x": torch.rand(*shape, generator=g, device="cuda"), "i": ints(-100, 101, *shape)}
    if kind == "chain":
        return {"x": normal(case["rows"], case["cols"]),
                "r": torch.rand(1, case["cols"], generator=g, device="cuda") * 1.5 + 0.5}
    if kind == "matmul":
        b, m, n, k = (case[q] for q in ("batch", "m", "n", "k"))
        lead = (b,) if b > 1 else ()
        s = k ** -0.5

        def mat(*shape):
            f = torch.float64 if case["dtype"] == "float64" else torch.float32
            return (torch.randn(*shape, generator=g, device="cuda", dtype=f) * s).to(
                _TORCH[case["dtype"]])

        return {"a": mat(*lead, m, k), "b": mat(*lead, k) if n == 1 else mat(*lead, k, n)}
    if kind == "sort":
        n = case["n"]
        key = (ints(-2 ** 31, 2 ** 31 - 1, n) if case["dtype"] == "int32"
               else normal(n, dtype=case["dtype"]))
        keep = torch.zeros(n, device="cuda", dtype=torch.bool)  # half of the rows
        keep[torch.randperm(n, generator=g, device="cuda")[:n // 2]] = True
        return {"key": key, "value": normal(n), "keep": keep}
    n, d = case["rows"], case["cols"]
    x = normal(n, d, dtype=case["dtype"])
    w = normal(d, dtype=case["dtype"])
    return {"x": x, "y": x @ w + normal(n, dtype=case["dtype"])}


def prepare(case, seed):
    state = {"kind": case["kind"]}
    for name, t in _inputs(case, seed).items():
        h = t.cpu().numpy()
        if case["kind"] == "small_host":
            state[name] = h
        else:
            state[name] = cp.array(h)
            state[name].ravel()  # on the device from here on
    cp.synchronize()
    return state


# ------------------------------------------------------------------ a pass
class _View:
    """A device array as torch.as_tensor reads one; it keeps the array alive."""

    __slots__ = ("array", "__cuda_array_interface__")

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str, "strides": None,
                                         "data": (a._ptr, False), "version": 2}


def _out(a):
    a = a._ensure_contiguous()
    return torch.as_tensor(_View(a), device="cuda")


def run(state):
    kind = state["kind"]
    if kind == "small_host":
        x, y = cp.array(state["x"]), cp.array(state["y"])
        return {"fused": (cp.sqrt(cp.abs(x)) + cp.exp(-x ** 2)).get(), "add": (x + y).get(),
                "sum": float(cp.sum(x))}
    if kind == "fused":
        x = state["x"]
        return _out(cp.sqrt(cp.abs(x)) + cp.exp(-x ** 2))
    if kind == "binary":
        a, b, i, j = state["a"], state["b"], state["i"], state["j"]
        return {"add": _out(a + b), "sin": _out(cp.sin(a)),
                "floor_divide": _out(cp.floor_divide(i, j)), "mod": _out(cp.mod(i, j))}
    if kind == "reduce":
        x = state["x"]
        return {"sum_rows": _out(cp.sum(x, axis=1)), "max_rows": _out(cp.max(x, axis=1)),
                "argmax_rows": _out(cp.argmax(x, axis=1)), "sum_columns": _out(cp.sum(x, axis=0)),
                "argmax_columns": _out(cp.argmax(x, axis=0)), "mean": _out(cp.mean(x))}
    if kind == "columns":
        x = state["x"]
        mean, dev = cp.mean(x, axis=0), cp.std(x, axis=0)
        return {"mean": _out(mean), "std": _out(dev), "standard": _out((x - mean) / dev)}
    if kind == "scan":
        x, i = state["x"], state["i"]
        return {"all": _out(cp.cumsum(x)), "all_int": _out(cp.cumsum(i)),
                "down": _out(cp.cumsum(x, axis=0)), "along": _out(cp.cumsum(x, axis=1))}
    if kind == "chain":
        x, r = state["x"], state["r"]
        return _out(cp.sum(cp.tanh(x * r + 1.0) * cp.exp(-cp.abs(x)) - cp.log1p(x * x), axis=1))
    if kind == "matmul":
        return _out(cp.matmul(state["a"], state["b"]))
    if kind == "sort":
        key, value, keep = state["key"], state["value"], state["keep"]
        order = cp.argsort(key)
        return {"sorted": _out(cp.sort(key)), "order": _out(order), "table": _out(value[order]),
                "kept": _out(value[keep])}
    x, y = state["x"], state["y"]
    xt = x.T
    gram, moment = cp.matmul(xt, x), cp.matmul(xt, y)
    w = cp.linalg.solve(gram, moment)
    return {"gram": _out(gram), "weights": _out(w), "rest": _out(y - cp.matmul(x, w))}


# -------------------------------------------------------- what a pass needs
def work(case):
    kind = case["kind"]
    if kind == "small_host":
        # two uploads, three reads, two results and a number
        return {"bytes": 4.0 * 4 * case["n"] + 4, "flops": 0.0}
    if kind == "fused":
        return {"bytes": 2.0 * _ITEM[case["dtype"]] * case["n"], "flops": 0.0}
    if kind == "binary":
        return {"bytes": 4.0 * (4 + 4) * case["n"], "flops": 0.0}
    if kind == "reduce":
        r, c, s = case["rows"], case["cols"], _ITEM[case["dtype"]]
        return {"bytes": 1.0 * s * r * c + r * (2 * s + 8) + c * (s + 8) + s, "flops": 0.0}
    if kind == "columns":
        s = _ITEM[case["dtype"]]
        return {"bytes": 2.0 * s * case["rows"] * case["cols"] + 2 * s * case["cols"], "flops": 0.0}
    if kind == "scan":
        # two inputs read, three float32 and one int64 result written
        return {"bytes": 28.0 * case["rows"] * case["cols"], "flops": 0.0}
    if kind == "chain":
        return {"bytes": 4.0 * (case["rows"] * case["cols"] + case["rows"] + case["cols"]),
                "flops": 0.0}
    if kind == "matmul":
        b, m, n, k = (float(case[q]) for q in ("batch", "m", "n", "k"))
        return {"bytes": _ITEM[case["dtype"]] * b * (m * k + k * n + m * n),
                "flops": 2.0 * b * m * n * k}
    if kind == "sort":
        # keys, values and mask read; sorted keys, int64 order, the gathered
        # table and half the values written
        s = _ITEM[case["dtype"]]
        return {"bytes": (2.0 * s + 4 + 1 + 8 + 4 + 2) * case["n"], "flops": 0.0}
    n, d, s = float(case["rows"]), float(case["cols"]), _ITEM[case["dtype"]]
    return {"bytes": s * (n * d + 2 * n + d * d + d), "flops": 2 * n * d * d + 4 * n * d + 2 / 3 * d ** 3}


def tolerance(case):
    """About four times the error against 64 bits, measured over the ranges."""
    kind, dtype = case["kind"], case.get("dtype", "float32")
    if kind in ("small_host", "fused", "binary"):
        # a few roundings a value; the sum is one number, good to an ulp or two
        return {"float16": {"rel": 1.2e-3, "max": 3e-3}, "float32": {"rel": 2.5e-7, "max": 6e-7},
                "float64": {"rel": 1e-15, "max": 4e-15}}[dtype]
    if kind == "reduce":
        # sums in 64 bits, rounded once: the mean of all is one number, and
        # two such may be an ulp apart
        return {"rel": {"int32": 1e-15, "float16": 2e-3, "float32": 2.5e-7}[dtype]}
    if kind == "columns":
        return {"rel": 8e-15 if dtype == "float64" else 4e-7}
    if kind in ("scan", "chain"):
        return {"rel": 2e-7}
    if kind == "matmul":
        # sums in the accumulator's precision, over up to 20,000 terms
        return {"rel": {"float16": 1e-3, "float32": 1e-5, "float64": 2e-14}[dtype]}
    if kind == "sort":
        return {"rel": 0.0}  # the same values and the same stable order
    # The products sum up to 10^7 terms in the type itself (1.7e-5 of the
    # Gram matrix in float32); the residual is a difference of values
    # sqrt(columns) times its size, so it shows that error many times over.
    return {"rel": 1e-12 if dtype == "float64" else 2e-3}


def exact(case, seed):
    """The same values in 64 bits, by torch alone."""
    kind, v = case["kind"], _inputs(case, seed)
    v = {q: t.double() if t.is_floating_point() else t if t.dtype == torch.bool else t.long()
         for q, t in v.items()}
    if kind in ("small_host", "fused"):
        x = v["x"]
        fused = x.abs().sqrt() + (-x * x).exp()
        if kind == "fused":
            return fused
        return {"fused": fused.cpu().numpy(), "add": (x + v["y"]).cpu().numpy(),
                "sum": float(x.sum())}
    if kind == "binary":
        return {"add": v["a"] + v["b"], "sin": v["a"].sin(),
                "floor_divide": torch.div(v["i"], v["j"], rounding_mode="floor"),
                "mod": torch.remainder(v["i"], v["j"])}
    if kind == "reduce":
        x = v["x"]
        return {"sum_rows": x.sum(1), "max_rows": x.amax(1), "argmax_rows": None,
                "sum_columns": x.sum(0), "argmax_columns": None, "mean": x.double().mean()}
    if kind == "columns":
        x = v["x"]
        mean, dev = x.mean(0), x.std(0, unbiased=False)
        return {"mean": mean, "std": dev, "standard": (x - mean) / dev}
    if kind == "scan":
        x = v["x"]
        return {"all": x.reshape(-1).cumsum(0), "all_int": v["i"].reshape(-1).cumsum(0),
                "down": x.cumsum(0), "along": x.cumsum(1)}
    if kind == "chain":
        x, r = v["x"], v["r"]
        return ((x * r + 1.0).tanh() * (-x.abs()).exp() - (x * x).log1p()).sum(1)
    if kind == "matmul":
        return torch.matmul(v["a"], v["b"])
    if kind == "sort":
        key, order = torch.sort(v["key"], stable=True)
        return {"sorted": key, "order": order, "table": v["value"][order],
                "kept": v["value"][v["keep"]]}
    x, y = v["x"], v["y"]
    gram, moment = x.T.contiguous() @ x, x.T.contiguous() @ y
    w = torch.linalg.solve(gram, moment)
    return {"gram": gram, "weights": w, "rest": y - x @ w}
