"""The work that is timed: single public calls of ``musapy_amd`` and short chains of them.

Each kind of case stands for one thing that a program using this backend does with device arrays, over
the sizes, ragged shapes, dtypes and layouts that such a program has.  Inputs are PyTorch tensors on the
GPU, adopted without a copy through DLPack; results go to preallocated tensors through ``out=`` where the
call takes one, and come back through DLPack where it does not.
"""
import math

import torch

import musapy_amd as ms

_DT = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64, "i8": torch.int8, "u8": torch.uint8,
       "i16": torch.int16, "i32": torch.int32, "i64": torch.int64, "bf16": torch.bfloat16, "f16": torch.float16}
_SIZE = {"f32": 4, "f64": 8, "c64": 8, "i8": 1, "u8": 1, "i16": 2, "i32": 4, "i64": 8, "bf16": 2, "f16": 2}


def listed():
    return [
        # Launch-bound: the calls of one small step on a (256, 256) array, the size of the reference's
        # own 2-D table (elementwise, both axis sums, argmax, a row scan).
        {"name": "small_step", "kind": "small", "rows": 256, "cols": 256, "dtype": "f32"},
        # The headline: contiguous f32 arrays of 64M elements, elementwise add, whole-array sum and argmax.
        {"name": "flat_64m", "kind": "flat", "n": 1 << 26, "op": "add", "dtype": "f32"},
        # Centring the columns of a table with odd sides: x - mean, the mean broadcast over the rows.
        {"name": "center_columns", "kind": "binary", "layout": "row", "rows": 20011, "cols": 3001, "op": "sub",
         "dtype": "f32"},
        # A matrix plus the transposed view of another (symmetrising, (x, y) against (y, x) grids).
        {"name": "add_transposed", "kind": "binary", "layout": "transposed", "rows": 6000, "cols": 5000, "op": "add",
         "dtype": "f32"},
        # Type promotion and casts: i64 + f64, clamp to [-1, 1], to f32, to bf16.
        {"name": "promote_cast", "kind": "promote", "n": 2048 * 2048 * 4, "ints": "i64", "half": "bf16"},
        # A transposed view through an elementwise op, and its materialisation.
        {"name": "transposed_view", "kind": "view", "rows": 8192, "cols": 4096, "dtype": "f32"},
        # Statistics of each row of a table with odd sides: mean, max and argmax along the last axis.
        {"name": "row_stats", "kind": "rows", "rows": 12007, "cols": 4099, "dtype": "f32"},
        # Statistics of the few columns of a long table (records x features): mean and max down axis 0.
        {"name": "column_stats", "kind": "columns", "rows": 1000003, "cols": 37, "dtype": "f32"},
        # Pooling over the middle axis of (batch, steps, channels), and over batch and steps together.
        {"name": "middle_axis", "kind": "middle", "outer": 64, "mid": 2048, "inner": 384, "dtype": "f32"},
        # Integer data: per-row totals and argmax, per-column means.
        {"name": "integer_stats", "kind": "ints", "rows": 4096, "cols": 8192, "dtype": "i32"},
        # Running sums along the rows, f64.
        {"name": "cumsum_rows", "kind": "scan", "axis": 1, "rows": 1024, "cols": 65536, "dtype": "f64"},
        # Running sums down the columns (a time series per column).
        {"name": "cumsum_columns", "kind": "scan", "axis": 0, "rows": 8192, "cols": 4096, "dtype": "f32"},
    ]


_MOST = 600e6  # bytes that a drawn case moves, at most


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["small", "flat", "binary", "binary", "promote", "view", "rows", "columns", "middle", "ints",
                       "scan", "scan"])
    while True:
        if kind == "small":
            c = {"rows": _log(rng, 2, 700), "cols": _log(rng, 2, 700), "dtype": rng.choice(["f32", "f64"])}
        elif kind == "flat":
            c = {"n": _log(rng, 1 << 18, 1 << 26), "op": rng.choice(["add", "sub", "mul", "div"]),
                 "dtype": rng.choice(["f32", "f32", "f64"])}
        elif kind == "binary":
            layout = rng.choice(["same", "row", "column", "transposed", "shifted", "stepped"])
            c = {"layout": layout, "rows": _log(rng, 16, 60000), "cols": _log(rng, 16, 60000),
                 "op": rng.choice(["add", "sub", "mul", "div"]), "dtype": rng.choice(["f32", "f32", "f64", "c64"])}
        elif kind == "promote":
            c = {"n": _log(rng, 1 << 14, 1 << 24), "ints": rng.choice(["i32", "i64"]),
                 "half": rng.choice(["bf16", "f16"])}
        elif kind == "view":
            c = {"rows": _log(rng, 16, 60000), "cols": _log(rng, 16, 60000), "dtype": rng.choice(["f32", "f32", "f64"])}
        elif kind == "rows":
            c = {"rows": _log(rng, 8, 1000000), "cols": _log(rng, 8, 1000000), "dtype": rng.choice(["f32", "f32", "f64"])}
        elif kind == "columns":
            c = {"rows": _log(rng, 64, 2000000), "cols": _log(rng, 2, 20000), "dtype": rng.choice(["f32", "f32", "f64"])}
        elif kind == "middle":
            c = {"outer": _log(rng, 2, 512), "mid": _log(rng, 16, 8192), "inner": _log(rng, 4, 2048),
                 "dtype": rng.choice(["f32", "f64", "c64"])}
        elif kind == "ints":
            c = {"rows": _log(rng, 64, 100000), "cols": _log(rng, 64, 100000),
                 "dtype": rng.choice(["i8", "u8", "i16", "i32", "i64"])}
        elif rng.random() < 0.5:  # rows: from many short ones to one long one
            c = {"axis": 1, "rows": _log(rng, 1, 200000), "cols": _log(rng, 16, 4000000),
                 "dtype": rng.choice(["f32", "f64"])}
        else:
            c = {"axis": 0, "rows": _log(rng, 64, 50000), "cols": _log(rng, 32, 20000),
                 "dtype": rng.choice(["f32", "f64"])}
        c["kind"] = kind
        b = work(c)["bytes"]
        if b <= _MOST and (kind == "small" or b >= 1e5):
            return c


# ---- inputs -------------------------------------------------------------------------------------
def _inputs(c, seed):
    """The case's input tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = c["kind"]
    dt = _DT[c["dtype"]] if "dtype" in c else None

    def uniform(shape, lo, hi):
        return torch.empty(shape, dtype=dt, device="cuda").uniform_(lo, hi, generator=g)

    def normal(shape, mean=0.0):
        x = torch.randn(shape, dtype=dt, device="cuda", generator=g)
        return x.add_(mean) if mean else x

    def ints(shape, d):
        lo, hi = {"i8": (-100, 101), "u8": (0, 256)}.get(d, (-1000, 1001))
        return torch.randint(lo, hi, shape, dtype=_DT[d], device="cuda", generator=g)

    if kind == "small":
        s = (c["rows"], c["cols"])
        return {"a": uniform(s, 0.0, 1.0), "b": uniform(s, 0.0, 1.0)}
    if kind == "flat":
        return {"a": uniform((c["n"],), 0.0, 1.0), "b": uniform((c["n"],), 0.5, 1.5)}
    if kind == "binary":
        r, k, layout = c["rows"], c["cols"], c["layout"]
        second = {"same": (r, k), "row": (k,), "column": (r, 1), "transposed": (k, r)}.get(layout)
        a = normal((r, k))
        return {"a": a, "b": normal(second)} if second else {"a": a}
    if kind == "promote":
        return {"i": ints((c["n"],), c["ints"]),
                "f": torch.randn((c["n"],), dtype=torch.float64, device="cuda", generator=g)}
    if kind == "view":
        return {"x": uniform((c["rows"], c["cols"]), -4.0, 4.0)}
    if kind == "rows":
        return {"x": normal((c["rows"], c["cols"]), 1.0)}
    if kind == "columns":
        return {"x": normal((c["rows"], c["cols"]), 1.0)}
    if kind == "middle":
        return {"x": normal((c["outer"], c["mid"], c["inner"]), 1.0)}
    if kind == "ints":
        return {"x": ints((c["rows"], c["cols"]), c["dtype"])}
    return {"x": uniform((c["rows"], c["cols"]), 0.0, 1.0)}


def _operands(c, t, slicer, transposer):
    """The two operands of a "binary" case, as views of its inputs."""
    a, layout = t["a"], c["layout"]
    r, k = c["rows"], c["cols"]
    if layout == "transposed":
        return a, transposer(t["b"])
    if layout == "shifted":  # neighbouring differences along the rows
        return slicer(a, [(0, r, 1), (1, k, 1)]), slicer(a, [(0, r, 1), (0, k - 1, 1)])
    if layout == "stepped":  # the even against the odd columns
        h = k // 2
        return slicer(a, [(0, r, 1), (0, 2 * h, 2)]), slicer(a, [(0, r, 1), (1, 2 * h, 2)])
    return a, t["b"]


def _binary_cols(c):
    return {"shifted": c["cols"] - 1, "stepped": c["cols"] // 2}.get(c["layout"], c["cols"])


def prepare(case, seed):
    c = case
    t = _inputs(c, seed)
    m = {k: ms.from_dlpack(v) for k, v in t.items()}
    kind = c["kind"]
    dt = _DT[c["dtype"]] if "dtype" in c else None
    i64, f64 = torch.int64, torch.float64
    if kind == "small":
        r, k = c["rows"], c["cols"]
        outs = [((r, k), dt), ((r, k), dt), ((k,), dt), ((r,), dt), ((r,), i64), ((r, k), dt)]
    elif kind == "flat":
        outs = [((c["n"],), dt), ((), dt), ((), i64)]
    elif kind == "binary":
        outs = [((c["rows"], _binary_cols(c)), dt)]
    elif kind == "promote":
        n = (c["n"],)
        outs = [(n, f64), (n, f64), (n, torch.float32), (n, _DT[c["half"]])]
    elif kind == "view":
        outs = [((c["cols"], c["rows"]), dt)]
    elif kind == "rows":
        outs = [((c["rows"],), dt), ((c["rows"],), dt), ((c["rows"],), i64)]
    elif kind == "columns":
        outs = [((c["cols"],), dt), ((c["cols"],), dt)]
    elif kind == "middle":
        outs = [((c["outer"], c["inner"]), dt)]
    elif kind == "ints":
        outs = [((c["rows"],), i64), ((c["rows"],), i64), ((c["cols"],), f64)]
    else:
        outs = [((c["rows"], c["cols"]), dt)]
    out_t = [torch.empty(s, dtype=d, device="cuda") for s, d in outs]
    return {"case": c, "in": m, "out_t": out_t, "out": [ms.from_dlpack(o) for o in out_t]}


def run(state):
    c, m, o, out = state["case"], state["in"], state["out"], state["out_t"]
    kind = c["kind"]
    if kind == "small":
        ms.add(m["a"], m["b"], out=o[0])
        ms.exp(m["a"], out=o[1])
        ms.sum(m["a"], axis=0, out=o[2])
        ms.sum(m["b"], axis=1, out=o[3])
        ms.argmax(m["a"], axis=1, out=o[4])
        ms.cumsum(m["b"], axis=1, out=o[5])
        return out
    if kind == "flat":
        getattr(ms, c["op"])(m["a"], m["b"], out=o[0])
        ms.sum(m["a"], out=o[1])
        ms.argmax(m["b"], out=o[2])
        return out
    if kind == "binary":
        a, b = _operands(c, m, ms.slice, ms.transpose)
        getattr(ms, c["op"])(a, b, out=o[0])
        return out
    if kind == "promote":
        ms.add(m["i"], m["f"], out=o[0])
        ms.clamp(o[0], -1.0, 1.0, out=o[1])
        ms.astype(o[1], "f32", out=o[2])
        ms.astype(o[2], c["half"], out=o[3])
        return out
    if kind == "view":
        ms.exp(m["x"].T, out=o[0])
        return [out[0], torch.from_dlpack(ms.contiguous(m["x"].T))]
    if kind == "rows":
        ms.mean(m["x"], axis=-1, out=o[0])
        ms.max(m["x"], axis=-1, out=o[1])
        ms.argmax(m["x"], axis=-1, out=o[2])
        return out
    if kind == "columns":
        ms.mean(m["x"], axis=0, out=o[0])
        ms.max(m["x"], axis=0, out=o[1])
        return out
    if kind == "middle":
        ms.sum(m["x"], axis=1, out=o[0])
        return [out[0], torch.from_dlpack(ms.mean(m["x"], axis=(0, 1)))]
    if kind == "ints":
        ms.sum(m["x"], axis=1, out=o[0])
        ms.argmax(m["x"], axis=1, out=o[1])
        ms.mean(m["x"], axis=0, out=o[2])
        return out
    ms.cumsum(m["x"], axis=c["axis"], out=o[0])
    return out


def work(case):
    """Each call's inputs read once and its result written once; one operation per element it computes on."""
    c, kind = case, case["kind"]
    es = _SIZE[c["dtype"]] if "dtype" in c else 0
    if kind == "small":
        r, k = c["rows"], c["cols"]
        n = r * k
        return {"bytes": n * es * (3 + 2 + 1 + 1 + 1 + 2) + (k + r) * es + 8 * r, "flops": 6 * n}
    if kind == "flat":
        return {"bytes": c["n"] * es * 5, "flops": 3 * c["n"]}
    if kind == "binary":
        r, k = c["rows"], _binary_cols(c)
        second = {"same": r * k, "row": k, "column": r, "transposed": r * k, "shifted": r, "stepped": r * k}[c["layout"]]
        return {"bytes": es * (2 * r * k + second), "flops": r * k}
    if kind == "promote":
        return {"bytes": c["n"] * (_SIZE[c["ints"]] + 16 + 16 + 12 + 6), "flops": 2 * c["n"]}
    if kind == "view":
        return {"bytes": 4 * es * c["rows"] * c["cols"], "flops": c["rows"] * c["cols"]}
    if kind == "rows":
        n = c["rows"] * c["cols"]
        return {"bytes": 3 * n * es + c["rows"] * (2 * es + 8), "flops": 3 * n}
    if kind == "columns":
        n = c["rows"] * c["cols"]
        return {"bytes": 2 * es * (n + c["cols"]), "flops": 2 * n}
    if kind == "middle":
        n = c["outer"] * c["mid"] * c["inner"]
        return {"bytes": es * (2 * n + c["outer"] * c["inner"] + c["inner"]), "flops": 2 * n}
    if kind == "ints":
        n = c["rows"] * c["cols"]
        return {"bytes": 3 * n * es + 16 * c["rows"] + 8 * c["cols"], "flops": 3 * n}
    return {"bytes": 2 * es * c["rows"] * c["cols"], "flops": c["rows"] * c["cols"]}


def tolerance(case):
    """IEEE elementwise results, casts, extremes, indices and integer results are bit-exact.  exp is within
    2 ulp (3e-8 norm-wise measured for f32).  Sums and scans differ by their association: f32 sums by up to
    2.2e-7 norm-wise against 64 bits, f64 ones by about 5e-16.  A running sum in order is further off the
    longer it is: 1.1e-6 (f32) and 2.0e-15 (f64) over 8192 values, 2.9e-6 and 4.8e-15 over 50000."""
    kind = case["kind"]
    if kind in ("binary", "promote", "ints"):
        return {"rel": 1e-14} if kind == "ints" else "exact"
    if kind == "view":
        return {"rel": 3e-7} if case["dtype"] == "f32" else {"rel": 6e-16}
    if kind == "scan":
        return {"rel": 2e-14} if case["dtype"] == "f64" else {"rel": 1.2e-5}
    return {"rel": 1e-14} if case["dtype"] == "f64" else {"rel": 1e-6}


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    kind = c["kind"]

    def wide(x):
        return x.to(torch.complex128 if x.is_complex() else torch.float64)

    ops = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div}
    if kind == "small":
        a, b = wide(t["a"]), wide(t["b"])
        return [a + b, a.exp(), a.sum(0), b.sum(1), None, b.cumsum(1)]
    if kind == "flat":
        a, b = wide(t["a"]), wide(t["b"])
        return [ops[c["op"]](a, b), a.sum(), None]
    if kind == "binary":
        def cut(x, ranges):
            return x[tuple(slice(*r) for r in ranges)]
        a, b = _operands(c, t, cut, lambda x: x.T)
        return [ops[c["op"]](wide(a), wide(b))]
    if kind == "promote":
        s = t["i"].to(torch.float64) + t["f"]
        u = s.clamp(-1.0, 1.0)
        return [s, u, u, u]
    if kind == "view":
        x = wide(t["x"]).T
        return [x.exp(), x.contiguous()]
    if kind == "rows":
        x = wide(t["x"])
        return [x.mean(1), x.amax(1), None]
    if kind == "columns":
        x = wide(t["x"])
        return [x.mean(0), x.amax(0)]
    if kind == "middle":
        x = wide(t["x"])
        return [x.sum(1), x.mean((0, 1))]
    if kind == "ints":
        return [None, None, t["x"].to(torch.float64).mean(0)]
    return [wide(t["x"]).cumsum(c["axis"])]
