"""Calls of the library that its performance is measured by, each through the ctypes binding as a program makes it.

A program that uses these primitives holds its device buffers and the temporary storage of every call from the
start (the storage contract is the caller's), and then calls.  `prepare` makes those buffers, `run` makes the call.

The listed cases go from a reduction of a few thousand items, where launches and latency are all there is, over
arrays of about a million items (a frame's particles, a batch of events), to the sizes that the benchmark
quotes: 2^28 four-byte items and 2^27 eight-byte keys with their values.  `draw` spreads over the same families,
with more item types, options, value distributions and odd sizes.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("luisacompute-parallelprimitive_amd"))
import lcpp_hip as hip  # noqa: E402

DTYPE = {"i32": torch.int32, "u32": torch.int32, "f32": torch.float32,
         "i64": torch.int64, "u64": torch.int64, "f64": torch.float64}
BYTES = hip.ELEM_BYTES


def listed():
    return [
        # A loss or a residual norm over one small array: two launches and their latency.
        {"name": "reduce_sum_f32_5k", "op": "reduce", "fold": "sum", "type": "f32", "n": 5003},
        # The benchmark's smaller reduction: 64 MiB, partly resident in the memory-side cache.
        {"name": "reduce_sum_i32_2p24", "op": "reduce", "fold": "sum", "type": "i32", "n": 1 << 24},
        # Cumulative weights of about a million samples (resampling, inverse-CDF tables).
        {"name": "inclusive_sum_f32_1m", "op": "scan", "type": "f32", "inclusive": True, "n": 1_000_003},
        # The benchmark's scan: offsets of 2^28 variable-length records.
        {"name": "exclusive_sum_u32_2p28", "op": "scan", "type": "u32", "inclusive": False, "n": 1 << 28},
        # Back-to-front order of a small scene: float depths with the index of each object.
        {"name": "sort_pairs_f32_20k_descending", "op": "sort", "key": "f32", "value_bytes": 4, "n": 20_011,
         "keys": "normal", "descending": True, "bits": 32},
        # Spatial (Morton) codes of about a million particles with their indices; codes have 30 bits.
        {"name": "sort_pairs_u32_1m_30bit", "op": "sort", "key": "u32", "value_bytes": 4, "n": 1_000_003,
         "keys": "uniform", "descending": False, "bits": 30},
        # The benchmark's headline.
        {"name": "sort_keys_u32_2p28", "op": "sort", "key": "u32", "value_bytes": 0, "n": 1 << 28,
         "keys": "uniform", "descending": False, "bits": 32},
        # The benchmark's largest sort: eight passes over 12-byte pairs.
        {"name": "sort_pairs_u64_2p27", "op": "sort", "key": "u64", "value_bytes": 4, "n": 1 << 27,
         "keys": "uniform", "descending": False, "bits": 64},
        # Stream compaction of ten million items, a third of them kept (live rays, active cells).
        {"name": "select_if_u32_10m", "op": "select", "type": "u32", "form": "if", "n": 10_000_019, "kept": 0.33},
        # Sums of float contributions per sorted key (a histogram or gradient gathered by index).
        {"name": "reduce_by_key_f32_4m", "op": "by_key", "form": "reduce", "key": "i32", "type": "f32",
         "n": 4_000_037, "mean_run": 20},
        # Per-list order of ragged lists (screen tiles, neighbour lists): lengths spread over two decades.
        {"name": "segmented_sort_pairs_u32_4m", "op": "segmented_sort", "key": "u32", "value_bytes": 4,
         "n": 4_000_037, "mean_length": 300},
        # The benchmark's sparse product: Zipf(1.5) row lengths up to 4096, columns anywhere.
        {"name": "spmv_f32_zipf_2p20", "op": "spmv", "type": "f32", "rows": 1 << 20, "cols": 1 << 20,
         "nnz": 49 << 20, "matrix": "zipf"},
    ]


def _size(rng, low, high):
    """A size between the two, spread over its logarithm; every third one a multiple of 256."""
    n = int(math.exp(rng.uniform(math.log(low), math.log(high))))
    return max(low, n // 256 * 256) if rng.randrange(3) == 0 else n


def draw(rng):
    op = rng.choice(["reduce", "scan", "sort", "sort", "sort", "select", "runs", "by_key", "segmented", "segmented_sort",
                     "spmv"])
    if op == "reduce":
        t = rng.choice(["i32", "u32", "f32", "f32", "i64", "f64"])
        fold = rng.choice(["sum", "sum", "min", "max"])
        return {"op": op, "fold": fold, "type": t, "n": _size(rng, 1 << 10, (1 << 30) // BYTES[t])}
    if op == "scan":
        t = rng.choice(["i32", "u32", "u32", "f32", "u64", "f64"])
        return {"op": op, "type": t, "inclusive": rng.random() < 0.5, "n": _size(rng, 1 << 10, (1 << 30) // BYTES[t])}
    if op == "sort":
        k = rng.choice(["u32", "u32", "i32", "f32", "u64"])
        v = rng.choice([0, 4, 4, 8])
        keys = rng.choice(["normal", "normal", "uniform"]) if k == "f32" else rng.choice(["uniform", "uniform", "and3"])
        bits = rng.choice([32, 32, 24, 16]) if k == "u32" else 8 * BYTES[k]
        return {"op": op, "key": k, "value_bytes": v, "n": _size(rng, 1 << 10, (1 << 30) // (BYTES[k] + v)),
                "keys": keys, "descending": rng.random() < 0.25, "bits": bits}
    if op == "select":
        t = rng.choice(["u32", "u32", "f32", "u64"])
        return {"op": op, "type": t, "form": rng.choice(["if", "if", "flagged", "partition"]),
                "n": _size(rng, 1 << 10, (1 << 30) // BYTES[t]), "kept": round(rng.uniform(0.05, 0.95), 3)}
    if op == "runs":
        t = rng.choice(["u32", "u32", "u64"])
        return {"op": op, "type": t, "form": rng.choice(["encode", "unique"]),
                "n": _size(rng, 1 << 10, (1 << 30) // BYTES[t]), "mean_run": rng.choice([2, 8, 64, 1000])}
    if op == "by_key":
        t = rng.choice(["u32", "f32", "f32", "f64"])
        return {"op": op, "form": rng.choice(["reduce", "scan"]), "key": rng.choice(["i32", "i32", "i64"]), "type": t,
                "n": _size(rng, 1 << 10, (1 << 29) // BYTES[t]), "mean_run": rng.choice([4, 20, 64, 1000])}
    if op == "segmented":
        t = rng.choice(["i32", "f32", "f32", "f64"])
        return {"op": op, "form": rng.choice(["sum", "max", "scan"]), "type": t,
                "n": _size(rng, 1 << 12, (1 << 29) // BYTES[t]), "mean_length": rng.choice([16, 100, 700, 4096])}
    if op == "segmented_sort":
        k = rng.choice(["u32", "u32", "f32", "u64"])
        return {"op": op, "key": k, "value_bytes": rng.choice([0, 4, 4, 8]),
                "n": _size(rng, 1 << 12, (1 << 28) // BYTES[k]), "mean_length": rng.choice([16, 100, 300, 1500])}
    rows = _size(rng, 1 << 10, 1 << 20)
    matrix = rng.choice(["zipf", "zipf", "band"])
    per_row = 49 if matrix == "zipf" else rng.choice([5, 7, 27])
    return {"op": "spmv", "type": rng.choice(["f32", "f32", "f64"]), "rows": rows, "cols": rows, "nnz": per_row * rows,
            "matrix": matrix}


# ---- inputs ----------------------------------------------------------------------------------------
def _items(t, n, g, low=-1000, high=1000):
    """Items to be summed: small integers, or floats in [0, 1)."""
    if t in ("f32", "f64"):
        return torch.rand(n, dtype=DTYPE[t], device="cuda", generator=g)
    return torch.randint(0 if t[0] == "u" else low, high + 1, (n,), dtype=DTYPE[t], device="cuda", generator=g)


def _words(t, n, g):
    """Uniform over every bit of the type."""
    bits = 8 * BYTES[t]
    if bits == 32:
        return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device="cuda", generator=g)
    high = torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int64, device="cuda", generator=g)
    high <<= 32
    return high.bitwise_or_(torch.randint(0, 1 << 32, (n,), dtype=torch.int64, device="cuda", generator=g))


def _keys(case, n, g):
    t = case["key"]
    kind = case.get("keys", "uniform")
    if t == "f32":
        if kind == "normal":
            return torch.randn(n, device="cuda", generator=g)
        return torch.rand(n, device="cuda", generator=g)
    k = _words(t, n, g)
    if kind == "and3":
        k &= _words(t, n, g)
        k &= _words(t, n, g)
    if case.get("bits", 64) < 32:
        k &= (1 << case["bits"]) - 1
    return k


def _runs(t, n, mean, g):
    """Sorted keys in runs of geometric length."""
    start = torch.rand(n, device="cuda", generator=g) < 1.0 / mean
    return torch.cumsum(start, 0, dtype=torch.int64).to(DTYPE[t])


def _offsets(n, segments, g):
    """Segment bounds: log-normal lengths (a few empty, a few ten times the mean) that add up to n."""
    w = torch.randn(segments, dtype=torch.float64, device="cuda", generator=g).exp_().cumsum(0)
    bounds = torch.zeros(segments + 1, dtype=torch.int32, device="cuda")
    bounds[1:] = (w / w[-1] * n).to(torch.int32)
    bounds[-1] = n
    return bounds


def _matrix(case, g):
    """CSR structure: row offsets and sorted columns."""
    rows, cols, nnz = case["rows"], case["cols"], case["nnz"]
    if case["matrix"] == "zipf":
        law = torch.arange(1, 4097, dtype=torch.float64, device="cuda").pow(-1.5).cumsum(0)
        u = torch.rand(rows, dtype=torch.float64, device="cuda", generator=g) * law[-1]
        length = (torch.searchsorted(law, u) + 1).to(torch.float64).cumsum(0)
        offsets = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
        offsets[1:] = (length / length[-1] * nnz).round().to(torch.int64)
        offsets[-1] = nnz
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"), offsets.diff(), output_size=nnz)
        column = torch.randint(0, cols, (nnz,), dtype=torch.int64, device="cuda", generator=g)
    else:
        per = nnz // rows
        offsets = torch.arange(rows + 1, device="cuda") * per
        row = torch.arange(rows, device="cuda").repeat_interleave(per)
        side = max(2, int(rows ** 0.5))
        reach = torch.tensor([0, -1, 1, -side, side], device="cuda")
        column = row + reach[torch.arange(nnz, device="cuda") % per % 5] * (1 + torch.arange(nnz, device="cuda") % per // 5)
        column.clamp_(0, cols - 1)
    key = torch.sort(row * cols + column).values
    return offsets.to(torch.int32), (key % cols).to(torch.int32)


def _threshold(case):
    """The bound below which uniform items are kept, in the item type."""
    bits = 8 * BYTES[case["type"]]
    return case["kept"] if case["type"] == "f32" else min(int(case["kept"] * (1 << 32)) << (bits - 32), (1 << bits) - 1)


def _temp(nbytes):
    return torch.empty(max(1, hip.bytes_to_uint_count(nbytes)), dtype=torch.int32, device="cuda")


def _out(t, n):
    return torch.zeros(n, dtype=DTYPE[t], device="cuda")


def _inputs(case, seed):
    """What a case's call reads, by name."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    op = case["op"]
    if op in ("reduce", "scan"):
        high = 15 if op == "scan" else 1000
        return {"x": _items(case["type"], case["n"], g, high=high)}
    if op in ("sort", "segmented_sort"):
        n = case["n"]
        d = {"k": _keys(case, n, g)}
        if case["value_bytes"]:
            d["v"] = torch.arange(n, dtype=torch.int32 if case["value_bytes"] == 4 else torch.int64, device="cuda")
        if op == "segmented_sort":
            d["b"] = _offsets(n, max(1, n // case["mean_length"]), g)
        return d
    if op == "select":
        t, n = case["type"], case["n"]
        d = {"x": torch.rand(n, device="cuda", generator=g) if t == "f32" else _words(t, n, g)}
        if case["form"] == "flagged":
            d["flags"] = (torch.rand(n, device="cuda", generator=g) < case["kept"]).to(torch.uint8)
        return d
    if op == "runs":
        return {"x": _runs(case["type"], case["n"], case["mean_run"], g)}
    if op == "by_key":
        return {"k": _runs(case["key"], case["n"], case["mean_run"], g), "x": _items(case["type"], case["n"], g)}
    if op == "segmented":
        return {"x": _items(case["type"], case["n"], g), "b": _offsets(case["n"], max(1, case["n"] // case["mean_length"]), g)}
    offsets, columns = _matrix(case, g)
    signed = lambda m: torch.rand(m, dtype=DTYPE[case["type"]], device="cuda", generator=g).mul_(2).sub_(1)
    return {"offsets": offsets, "columns": columns, "values": signed(case["nnz"]), "x": signed(case["cols"])}


# ---- calls -----------------------------------------------------------------------------------------
def prepare(case, seed):
    """The call with its buffers (`call`), and the buffers that it fills (`out`)."""
    d = _inputs(case, seed)
    op, n = case["op"], case.get("n", 0)
    if op == "reduce":
        t, out, temp = case["type"], _out(case["type"], 1), _temp(hip.reduce_temp_bytes(n, BYTES[case["type"]]))
        if case["fold"] == "sum":
            return {"call": lambda: hip.reduce_sum(t, d["x"], out, n, temp=temp), "out": out}
        return {"call": lambda: hip.reduce_minmax(case["fold"], t, d["x"], out, n, temp=temp), "out": out}
    if op == "scan":
        t, out, temp = case["type"], _out(case["type"], n), _temp(hip.scan_temp_bytes(n, BYTES[case["type"]]))
        inclusive = case["inclusive"]
        return {"call": lambda: hip.scan_sum(t, d["x"], out, n, inclusive=inclusive, temp=temp), "out": out}
    if op == "sort":
        k, vb, bits, desc = case["key"], case["value_bytes"], case["bits"], case["descending"]
        ko = _out(k, n)
        if not vb:
            temp = _temp(hip.sort_keys_temp_bytes(n, BYTES[k]))
            return {"call": lambda: hip.sort_keys(k, d["k"], ko, n, end_bit=bits, descending=desc, temp=temp), "out": ko}
        vo, temp = torch.zeros_like(d["v"]), _temp(hip.sort_pairs_temp_bytes(n, BYTES[k], vb))
        return {"call": lambda: hip.sort_pairs(k, vb, d["k"], ko, d["v"], vo, n, end_bit=bits, descending=desc, temp=temp),
                "out": [ko, vo]}
    if op == "select":
        t, out, num = case["type"], _out(case["type"], n), _out("u32", 1)
        temp = _temp(hip.select_temp_bytes(n))
        if case["form"] == "flagged":
            return {"call": lambda: hip.select_flagged(t, "b8", d["x"], d["flags"], out, num, n, temp=temp), "out": [out, num]}
        below = hip.predicate(t, (hip.PRED_LT, _threshold(case)))
        call = hip.select_if if case["form"] == "if" else hip.partition_if
        return {"call": lambda: call(t, d["x"], out, num, n, below, temp=temp), "out": [out, num]}
    if op == "runs":
        t, out, num = case["type"], _out(case["type"], n), _out("u32", 1)
        if case["form"] == "unique":
            temp = _temp(hip.select_temp_bytes(n))
            return {"call": lambda: hip.select_unique(t, d["x"], out, num, n, temp=temp), "out": [out, num]}
        counts, temp = _out("u32", n), _temp(hip.run_length_encode_temp_bytes(n))
        return {"call": lambda: hip.run_length_encode(t, d["x"], out, counts, num, n, temp=temp), "out": [out, counts, num]}
    if op == "by_key":
        k, t, out = case["key"], case["type"], _out(case["type"], n)
        if case["form"] == "scan":
            temp = _temp(hip.scan_by_key_temp_bytes(n, BYTES[k], BYTES[t]))
            return {"call": lambda: hip.scan_by_key(k, t, d["k"], d["x"], out, n, temp=temp), "out": out}
        unique, num, temp = _out(k, n), _out("u32", 1), _temp(hip.reduce_by_key_temp_bytes(n, BYTES[k], BYTES[t]))
        return {"call": lambda: hip.reduce_by_key(k, t, d["k"], d["x"], unique, out, num, n, temp=temp),
                "out": [out, unique, num]}
    if op == "segmented":
        t, segments = case["type"], d["b"].numel() - 1
        begins, ends = d["b"][:-1].clone(), d["b"][1:].clone()
        if case["form"] == "scan":
            out = _out(t, n)
            return {"call": lambda: hip.segmented_scan(t, d["x"], out, begins, ends, segments, inclusive=True), "out": out}
        out = _out(t, segments)
        return {"call": lambda: hip.segment_reduce(case["form"], t, d["x"], out, segments, begins=begins, ends=ends), "out": out}
    if op == "segmented_sort":
        k, vb, segments, ko = case["key"], case["value_bytes"], d["b"].numel() - 1, _out(case["key"], n)
        begins, ends = d["b"][:-1].clone(), d["b"][1:].clone()
        if not vb:
            temp = _temp(hip.segmented_sort_keys_temp_bytes(n, BYTES[k]))
            return {"call": lambda: hip.segmented_sort(k, d["k"], ko, n, segments, begins, ends, temp=temp), "out": ko}
        vo, temp = torch.zeros_like(d["v"]), _temp(hip.segmented_sort_pairs_temp_bytes(n, BYTES[k], vb))
        return {"call": lambda: hip.segmented_sort(k, d["k"], ko, n, segments, begins, ends, values_in=d["v"], values_out=vo,
                                                   temp=temp), "out": [ko, vo]}
    t, rows, cols, nnz, y = case["type"], case["rows"], case["cols"], case["nnz"], _out(case["type"], case["rows"])
    return {"call": lambda: hip.spmv_csr(t, "i32", d["values"], d["offsets"], d["columns"], d["x"], y, rows, cols, nnz),
            "out": y}


def run(state):
    state["call"]()
    return state["out"]


def work(case):
    op, n = case["op"], case.get("n", 0)
    if op == "reduce":
        return {"bytes": n * BYTES[case["type"]], "flops": n}
    if op == "scan":
        return {"bytes": 2 * n * BYTES[case["type"]], "flops": n}
    if op == "sort":
        return {"bytes": 2 * n * (BYTES[case["key"]] + case["value_bytes"]), "flops": 0}
    if op == "select":
        b = BYTES[case["type"]]
        kept = n if case["form"] == "partition" else int(case["kept"] * n)
        return {"bytes": b * (n + kept) + (n if case["form"] == "flagged" else 0), "flops": 0}
    if op == "runs":
        b = BYTES[case["type"]]
        return {"bytes": b * n + (b + (4 if case["form"] == "encode" else 0)) * (n // case["mean_run"]), "flops": 0}
    if op == "by_key":
        k, b = BYTES[case["key"]], BYTES[case["type"]]
        out = n * b if case["form"] == "scan" else (k + b) * (n // case["mean_run"])
        return {"bytes": n * (k + b) + out, "flops": n}
    if op == "segmented":
        b, segments = BYTES[case["type"]], max(1, n // case["mean_length"])
        return {"bytes": b * n + 8 * segments + b * (n if case["form"] == "scan" else segments), "flops": n}
    if op == "segmented_sort":
        return {"bytes": 2 * n * (BYTES[case["key"]] + case["value_bytes"]) + 8 * (n // case["mean_length"]), "flops": 0}
    b = BYTES[case["type"]]
    return {"bytes": (b + 4) * case["nnz"] + 4 * (case["rows"] + 1) + b * (case["rows"] + case["cols"]),
            "flops": 2 * case["nnz"]}


def tolerance(case):
    """Order and whole numbers are exact; sums of floats may be added up in another order.  The bounds are four times
    the largest distance from `exact` over the ranges: 3.2e-7 (a scan of 2^27 items) and 1.2e-7 (SpMV) for f32, 1.2e-15
    (a scan) for f64."""
    t, op = case.get("type", ""), case["op"]
    summed = op in ("scan", "spmv", "by_key") or (op == "reduce" and case["fold"] == "sum") or \
        (op == "segmented" and case["form"] in ("sum", "scan"))
    if not summed or t not in ("f32", "f64"):
        return "exact"
    return {"rel": 4e-15 if t == "f64" else 1.3e-6 if op == "scan" else 5e-7}


# ---- the same results by plain torch in 64 bits ------------------------------------------------------
def _ordered(k, t):
    """Integer keys whose signed order is the order of the type."""
    if t == "u32":
        return k.to(torch.int64) & 0xFFFFFFFF
    return k ^ (-1 << 63) if t == "u64" else k


def exact(case, seed):
    if case.get("type") == "f64" and case["op"] in ("by_key", "segmented", "spmv"):
        return None  # torch adds in 64 bits too, one item after the other: further off than the results themselves
    d = _inputs(case, seed)
    op, n = case["op"], case.get("n", 0)
    if op == "reduce":
        x = d["x"]
        if case["fold"] == "sum":
            return x.double().sum().reshape(1) if x.is_floating_point() else x.sum(dtype=torch.int64).to(x.dtype).reshape(1)
        return getattr(x, case["fold"])().reshape(1)
    if op == "scan":
        x = d["x"]
        if x.is_floating_point():
            s = torch.cumsum(x, 0, dtype=torch.float64)
            return s if case["inclusive"] else s - x
        s = torch.cumsum(x, 0, dtype=torch.int64)
        return (s if case["inclusive"] else s.sub_(x)).to(x.dtype)
    if op == "sort":
        k, order = torch.sort(_ordered(d["k"], case["key"]), stable=True, descending=case["descending"])
        if case["key"] in ("u32", "u64"):
            k = (k.to(torch.int32) if case["key"] == "u32" else k ^ (-1 << 63))
        return [k, order.to(d["v"].dtype)] if case["value_bytes"] else k
    if op == "select":
        x = d["x"]
        if case["form"] == "flagged":
            keep = d["flags"] != 0
        else:
            keep = _ordered(x, case["type"]) < _ordered(torch.tensor(_threshold(case) if case["type"] == "f32" else (
                _threshold(case) if case["type"] == "u32" else _threshold(case) - (1 << 64) * (_threshold(case) >> 63)),
                device="cuda"), case["type"])
        num = keep.sum().to(torch.int32).reshape(1)
        rest = x[~keep].flip(0) if case["form"] == "partition" else x.new_zeros(n - int(num))
        return [torch.cat([x[keep], rest]), num]
    if op == "runs":
        u, c = torch.unique_consecutive(d["x"], return_counts=True)
        num = torch.tensor([u.numel()], dtype=torch.int32, device="cuda")
        out = torch.cat([u, u.new_zeros(n - u.numel())])
        if case["form"] == "unique":
            return [out, num]
        return [out, torch.cat([c.to(torch.int32), torch.zeros(n - u.numel(), dtype=torch.int32, device="cuda")]), num]
    if op in ("by_key", "segmented"):
        x = d["x"]
        wide = x.double() if x.is_floating_point() else x.to(torch.int64)
        if op == "by_key":
            u, c = torch.unique_consecutive(d["k"], return_counts=True)
        else:
            c = d["b"].diff().to(torch.int64)
        segments = c.numel()
        which = torch.repeat_interleave(torch.arange(segments, device="cuda"), c, output_size=n)
        if case["form"] == "max":
            low = float("-inf") if x.is_floating_point() else -(1 << 63)
            best = torch.full((segments,), low, dtype=wide.dtype, device="cuda").scatter_reduce(0, which, wide, "amax")
            # An empty segment has the type's lowest value.
            lowest = torch.finfo(x.dtype).min if x.is_floating_point() else torch.iinfo(x.dtype).min
            return best.clamp(min=lowest).to(x.dtype)
        if case["form"] == "scan":
            s = torch.cumsum(wide, 0)
            before = torch.cat([s.new_zeros(1), s])[(c.cumsum(0) - c)]
            s = s - before[which]
            s = s if op == "segmented" else s - wide
            return s if x.is_floating_point() else s.to(x.dtype)
        total = torch.zeros(segments, dtype=wide.dtype, device="cuda").index_add_(0, which, wide)
        total = total if x.is_floating_point() else total.to(x.dtype)
        if op == "segmented":
            return total
        fill = lambda a: torch.cat([a, a.new_zeros(n - segments)])
        return [fill(total), fill(u), torch.tensor([segments], dtype=torch.int32, device="cuda")]
    if op == "segmented_sort":
        c = d["b"].diff().to(torch.int64)
        which = torch.repeat_interleave(torch.arange(c.numel(), device="cuda"), c, output_size=n)
        order = torch.sort(_ordered(d["k"], case["key"]), stable=True).indices
        order = order[torch.sort(which[order], stable=True).indices]
        return [d["k"][order], d["v"][order]] if case["value_bytes"] else d["k"][order]
    row = torch.repeat_interleave(torch.arange(case["rows"], device="cuda"), d["offsets"].diff().to(torch.int64),
                                  output_size=case["nnz"])
    y = torch.zeros(case["rows"], dtype=torch.float64, device="cuda")
    return y.index_add_(0, row, d["values"].double() * d["x"].double()[d["columns"].to(torch.int64)])
