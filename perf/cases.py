"""Performance cases of the execution library's public Python entry points.

Each case is one call (or the few calls that belong together) as a program
makes it on resident data: span reductions, scans and sorts from a thousand
elements to 2^28, the batched (segmented) entry points over many uneven
ranges, and the request server on a mixed stream.  Inputs come from torch
generators, so the 64-bit references below use none of this package's code.

Kinds and the ranges their drawn cases cover:
  reduce     span reductions (sum, min, max, minloc, maxloc and the fused
             sum/min/max/minloc), n in [2^10, 2^28]
  scan       inclusive and exclusive scans, in place or not, n in [2^10, 2^28]
  sort       stable sorts of keys or (key, value) pairs, either direction,
             full-range or heavily duplicated keys, n in [2^10, 2^28]
  seg        one plan of uneven segments: a sum and an exclusive scan over it
  seg_sort   one plan of uneven segments: a sort of every segment
  serve      a batched server running a list of mixed requests that all wait
"""
import math

import numpy as np
import torch

import raja_amd as R

DEV = "cuda:0"
DTYPES = {"i32": torch.int32, "u32": torch.uint32, "f32": torch.float32,
          "i64": torch.int64, "u64": torch.uint64, "f64": torch.float64}
SIZE = {"i32": 4, "u32": 4, "f32": 4, "i64": 8, "u64": 8, "f64": 8}
OPS = {"sum": R.operators.plus, "min": R.operators.minimum, "max": R.operators.maximum}


def listed():
    return [
        # A reduction inside an iteration over a small range: launch latency.
        {"name": "reduce_sum_f64_1k", "kind": "reduce", "dtype": "f64", "op": "sum", "n": 1000},
        # A residual or dot-product style sum over a field of about 2^24 cells (the
        # benchmark's forall size).
        {"name": "reduce_sum_f64_16m", "kind": "reduce", "dtype": "f64", "op": "sum", "n": (1 << 24) + 3},
        # Four reducers of one loop over 2^28 FP64 (the benchmark's multi-reduction).
        {"name": "multi_reduce_f64_268m", "kind": "reduce", "dtype": "f64", "op": "multi", "n": 1 << 28},
        # Offsets of a short list (stream compaction, CSR rows of a small block).
        {"name": "exclusive_scan_i32_10k", "kind": "scan", "dtype": "i32", "op": "sum",
         "exclusive": True, "inplace": False, "n": 10007},
        # Offsets of a mesh-sized list.
        {"name": "exclusive_scan_i32_2m", "kind": "scan", "dtype": "i32", "op": "sum",
         "exclusive": True, "inplace": False, "n": (1 << 21) + 5},
        # The benchmark's 64-bit scan.
        {"name": "inclusive_scan_i64_268m", "kind": "scan", "dtype": "i64", "op": "sum",
         "exclusive": False, "inplace": False, "n": 1 << 28},
        # Sorting a small work list by key.
        {"name": "sort_pairs_u32_5k", "kind": "sort", "dtype": "u32", "val_bytes": 4,
         "descending": False, "bits": 32, "n": 5000},
        # Sorting a particle- or cell-list of a million entries.
        {"name": "sort_pairs_u32_1m", "kind": "sort", "dtype": "u32", "val_bytes": 4,
         "descending": False, "bits": 32, "n": 1000003},
        # The benchmark's headline sort.
        {"name": "sort_pairs_u32_268m", "kind": "sort", "dtype": "u32", "val_bytes": 4,
         "descending": False, "bits": 32, "n": 1 << 28},
        # The benchmark's batched work: sum and scan over 20,000 segments of
        # log-uniform length in [1, 2^16].
        {"name": "segmented_sum_scan_20000", "kind": "seg", "nseg": 20000, "max_log2": 16},
        # The same segments, each sorted by key.
        {"name": "segmented_sort_pairs_20000", "kind": "seg_sort", "dtype": "u32", "val_bytes": 4,
         "nseg": 20000, "max_log2": 16},
        # The benchmark's request mix (40 % sums, 30 % scans, 30 % sorts, sizes
        # log-uniform in [2^10, 2^24]), all requests waiting.
        {"name": "serve_mix_400", "kind": "serve", "nreq": 400, "lo_log2": 10, "span_log2": 14},
    ]


def _log_uniform(rng, lo, hi):
    return int(min(hi, max(lo, math.floor(2.0 ** rng.uniform(math.log2(lo), math.log2(hi))))))


def draw(rng):
    kind = rng.choice(["reduce", "reduce", "scan", "scan", "sort", "sort", "seg", "seg_sort", "serve"])
    if kind == "reduce":
        op = rng.choice(["sum", "sum", "min", "max", "minloc", "maxloc", "multi"])
        dtype = "f64" if op == "multi" else rng.choice(["f64", "f64", "f32", "i32", "i64"])
        return {"kind": kind, "dtype": dtype, "op": op, "n": _log_uniform(rng, 1 << 10, 1 << 28)}
    if kind == "scan":
        dtype = rng.choice(["i32", "i32", "i64", "u32", "f32", "f64"])
        op = rng.choice(["sum", "sum", "sum", "min", "max"])
        # an exclusive floating min or max starts with the type's largest
        # value, beside which no other output would count: inclusive there
        exclusive = rng.random() < 0.5 and not (op != "sum" and dtype[0] == "f")
        return {"kind": kind, "dtype": dtype, "op": op, "exclusive": exclusive,
                "inplace": rng.random() < 0.25, "n": _log_uniform(rng, 1 << 10, 1 << 28)}
    if kind == "sort":
        dtype = rng.choice(["u32", "u32", "i32", "f32", "u64", "i64", "f64"])
        vb = rng.choice([0, 4, 4, 8])
        # passes x bytes per pair of the largest listed sort bound the length
        cap = (1 << 28) * 32 // (max(SIZE[dtype] + vb, 8) * SIZE[dtype])
        return {"kind": kind, "dtype": dtype, "val_bytes": vb, "descending": rng.random() < 0.3,
                "bits": 12 if dtype in ("u32", "i32") and rng.random() < 0.25 else 8 * SIZE[dtype],
                "n": _log_uniform(rng, 1 << 10, cap)}
    if kind in ("seg", "seg_sort"):
        c = {"kind": kind, "nseg": _log_uniform(rng, 200, 30000), "max_log2": rng.randint(7, 16)}
        if kind == "seg_sort":
            c.update(dtype=rng.choice(["u32", "i32", "f32"]), val_bytes=rng.choice([0, 4, 4]))
        return c
    small = rng.random() < 0.5  # the benchmark's small-request stream or its full mix
    return {"kind": kind, "nreq": _log_uniform(rng, 40, 2000 if small else 400), "lo_log2": 10,
            "span_log2": 6 if small else 14}


# ---- inputs ------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _values(dtype, n, g, positive=False):
    """Values to reduce or scan: FP64 ~ N(0, 1), FP32 in [0, 1) (well
    conditioned sums), small non-negative integers (counts) for scans, signed
    ones for reductions."""
    if dtype == "f64":
        return torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    if dtype == "f32":
        return torch.rand(n, generator=g, device=DEV, dtype=torch.float32)
    lo, hi = (0, 16) if positive else (-1000000, 1000000)
    x = torch.randint(lo, hi, (n,), generator=g, device=DEV,
                      dtype=torch.int32 if SIZE[dtype] == 4 else torch.int64)
    return x.view(DTYPES[dtype])


def _keys(dtype, bits, n, g):
    if dtype == "f64":
        return torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    if dtype == "f32":
        return torch.randn(n, generator=g, device=DEV, dtype=torch.float32)
    if SIZE[dtype] == 4:
        lo, hi = (0, 1 << bits) if bits < 32 else (-(1 << 31), 1 << 31)
        return torch.randint(lo, hi, (n,), generator=g, device=DEV, dtype=torch.int32).view(DTYPES[dtype])
    hi32 = torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device=DEV, dtype=torch.int64)
    lo32 = torch.randint(0, 1 << 32, (n,), generator=g, device=DEV, dtype=torch.int64)
    return ((hi32 << 32) | lo32).view(DTYPES[dtype])


def _raw(t):
    """The same bits as a signed integer tensor (torch copies and compares those on every device)."""
    if t.dtype == torch.uint32:
        return t.view(torch.int32)
    return t.view(torch.int64) if t.dtype == torch.uint64 else t


def _offsets(case):
    """Segment lengths of a case: its layout is fixed, the seed makes the data."""
    u = np.random.default_rng([case["nseg"], case["max_log2"]]).random(case["nseg"])
    top = case["max_log2"]
    lens = np.clip(np.floor(2.0 ** (top * u)), 1, 1 << top).astype(np.int64)
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)


def _requests(case):
    """(kind, n, source element) of every request: fixed by the case, the seed makes the data."""
    rng = np.random.default_rng([case["nreq"], case["span_log2"]])
    u = rng.random(case["nreq"])
    kinds = np.where(u < 0.4, 0, np.where(u < 0.7, 1, 2))
    sizes = np.floor(2.0 ** (case["lo_log2"] + case["span_log2"] * rng.random(case["nreq"]))).astype(np.int64)
    top = 1 << (case["lo_log2"] + case["span_log2"])
    src = (rng.random(case["nreq"]) * ((top - sizes) // 64 + 1)).astype(np.int64) * 64
    return kinds, sizes, src, top


def _request_sources(top, g):
    x = torch.randn(top, generator=g, device=DEV, dtype=torch.float64)
    xi = torch.randint(0, 16, (top,), generator=g, device=DEV, dtype=torch.int32)
    xk = torch.randint(-(1 << 31), 1 << 31, (top,), generator=g, device=DEV, dtype=torch.int32)
    xv = torch.arange(top, dtype=torch.int32, device=DEV)
    return x, xi, xk, xv


def prepare(case, seed):
    g = _gen(seed)
    kind, n = case["kind"], case.get("n")
    if kind == "reduce":
        return {"case": case, "x": _values(case["dtype"], n, g)}
    if kind == "scan":
        x = _values(case["dtype"], n, g, positive=True)
        return {"case": case, "x": x, "out": torch.empty_like(x)}
    if kind == "sort":
        keys0 = _keys(case["dtype"], case["bits"], n, g)
        s = {"case": case, "keys0": keys0, "keys": torch.empty_like(keys0), "vals0": None, "vals": None}
        if case["val_bytes"]:
            s["vals0"] = torch.arange(n, device=DEV, dtype=torch.int32 if case["val_bytes"] == 4 else torch.int64)
            s["vals"] = torch.empty_like(s["vals0"])
        return s
    if kind in ("seg", "seg_sort"):
        off = _offsets(case)
        total = int(off[-1])
        s = {"case": case, "plan": R.Segments(off)}
        if kind == "seg":
            s["x"] = _values("f64", total, g)
            s["xi"] = _values("i32", total, g, positive=True)
            s["out"] = torch.empty_like(s["xi"])
            s["sums"] = torch.empty(case["nseg"], dtype=torch.float64, device=DEV)
        else:
            s["keys0"] = _keys(case["dtype"], 32, total, g)
            s["keys"] = torch.empty_like(s["keys0"])
            s["vals0"] = torch.arange(total, dtype=torch.int32, device=DEV) if case["val_bytes"] else None
            s["vals"] = torch.empty_like(s["vals0"]) if case["val_bytes"] else None
        return s
    kinds, sizes, src, top = _requests(case)
    x, xi, xk, xv = _request_sources(top, g)
    room = lambda k: int(((sizes[kinds == k] + 63) // 64 * 64).sum())  # noqa: E731
    sums = torch.zeros(case["nreq"], dtype=torch.float64, device=DEV)
    so = torch.zeros(max(room(1), 64), dtype=torch.int32, device=DEV)
    ok = torch.zeros(max(room(2), 64), dtype=torch.int32, device=DEV)
    ov = torch.zeros_like(ok)
    reqs = (R.Request * case["nreq"])()
    at = [0, 0, 0]
    for i in range(case["nreq"]):
        k, m, b = int(kinds[i]), int(sizes[i]), int(src[i])
        o = at[k]
        at[k] += (m + 63) // 64 * 64
        if k == 0:
            reqs[i] = R.request(R.REQ_SUM_F64, m, x.data_ptr() + 8 * b, sums.data_ptr() + 8 * i)
        elif k == 1:
            reqs[i] = R.request(R.REQ_EXCLUSIVE_SCAN_I32, m, xi.data_ptr() + 4 * b, so.data_ptr() + 4 * o)
        else:
            reqs[i] = R.request(R.REQ_SORT_PAIRS_U32_I32, m, xk.data_ptr() + 4 * b, ok.data_ptr() + 4 * o,
                                xv.data_ptr() + 4 * b, ov.data_ptr() + 4 * o)
    server = R.Server(R.SERVE_BATCHED, streams=16, max_inflight=64, max_batch=512, batch_limit=1 << 24,
                      arena_bytes=8 << 30)
    return {"case": case, "server": server, "reqs": reqs, "in": (x, xi, xk, xv), "out": (sums, so, ok, ov)}


# ---- one pass ------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "reduce":
        x, op = state["x"], case["op"]
        if op == "sum":
            return R.reduce_sum(x)
        if op == "min":
            return R.reduce_min(x)
        if op == "max":
            return R.reduce_max(x)
        if op == "minloc":
            return R.reduce_minloc(x)
        if op == "maxloc":
            return R.reduce_maxloc(x)
        out = R.multi_reduce_f64(x)  # sum, min, max, minloc value, minloc index (int64 bits)
        return out[:4], out[4:5].view(torch.int64)
    if kind == "scan":
        x, out, op = state["x"], state["out"], OPS[case["op"]]
        if case["inplace"]:
            out.copy_(x)  # the program keeps its unscanned values
            fn = R.exclusive_scan_inplace if case["exclusive"] else R.inclusive_scan_inplace
            return _raw(fn(out, op))
        fn = R.exclusive_scan if case["exclusive"] else R.inclusive_scan
        return _raw(fn(x, out, op))
    if kind == "sort":
        keys, vals = state["keys"], state["vals"]
        keys.copy_(state["keys0"])  # sorts are in place: the program keeps its unsorted list
        if vals is not None:
            vals.copy_(state["vals0"])
        R.sort_pairs(keys, vals, R.operators.greater if case["descending"] else R.operators.less)
        return _raw(keys), vals
    if kind == "seg":
        R.segmented_reduce(state["plan"], state["x"], R.operators.plus, 0.0, state["sums"])
        R.segmented_exclusive_scan(state["plan"], state["xi"], state["out"], R.operators.plus, 0)
        return state["sums"], state["out"]
    if kind == "seg_sort":
        keys, vals = state["keys"], state["vals"]
        keys.copy_(state["keys0"])
        if vals is not None:
            vals.copy_(state["vals0"])
        R.segmented_sort_pairs(state["plan"], keys, vals)
        return _raw(keys), vals
    results, _ = state["server"].run(state["reqs"])
    return list(state["out"])


# ---- what a pass cannot do without -----------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "reduce":
        per = 4 if case["op"] == "multi" else 1
        return {"bytes": case["n"] * SIZE[case["dtype"]], "flops": per * case["n"]}
    if kind == "scan":
        return {"bytes": 2 * case["n"] * SIZE[case["dtype"]], "flops": case["n"]}
    if kind == "sort":
        return {"bytes": 2 * case["n"] * (SIZE[case["dtype"]] + case["val_bytes"]), "flops": 0}
    if kind in ("seg", "seg_sort"):
        # the mean of floor(2^(m u)), u uniform, is close to (2^m - 1) / (m ln 2) - 1/2
        mean = ((1 << case["max_log2"]) - 1) / (case["max_log2"] * math.log(2)) - 0.5
        total = int(case["nseg"] * mean)
        if kind == "seg":
            return {"bytes": 16 * total + 16 * case["nseg"], "flops": 2 * total}
        return {"bytes": 2 * total * (4 + case["val_bytes"]), "flops": 0}
    lo, span = case["lo_log2"], case["span_log2"]
    mean = (2.0 ** (lo + span) - 2.0 ** lo) / (span * math.log(2))
    per = 0.4 * 8 + 0.3 * 8 + 0.3 * 16
    return {"bytes": int(case["nreq"] * mean * per), "flops": int(0.7 * case["nreq"] * mean)}


# ---- the same in 64 bits, by torch ------------------------------------------------------

def exact(case, seed):
    g = _gen(seed)
    kind, n = case["kind"], case.get("n")
    if kind == "reduce":
        x = _values(case["dtype"], n, g)
        if not x.is_floating_point():
            return None
        d, op = x.double(), case["op"]
        if op == "sum":
            return d.sum().reshape(1)
        if op in ("min", "minloc"):
            v = d.min().reshape(1)
        elif op in ("max", "maxloc"):
            v = d.max().reshape(1)
        else:
            return torch.stack([d.sum(), d.min(), d.max(), d.min()]), None
        return (v, None) if op.endswith("loc") else v
    if kind == "scan":
        x = _values(case["dtype"], n, g, positive=True)
        if not x.is_floating_point():
            return None
        d = x.double()
        op = case["op"]
        y = {"sum": lambda: torch.cumsum(d, 0), "min": lambda: torch.cummin(d, 0).values,
             "max": lambda: torch.cummax(d, 0).values}[op]()
        if not case["exclusive"]:
            return y
        return torch.cat([torch.zeros(1, dtype=torch.float64, device=DEV), y[:-1]])
    if kind == "sort":
        keys = _keys(case["dtype"], case["bits"], n, g)
        if not keys.is_floating_point():
            return None
        return torch.sort(keys.double(), descending=case["descending"]).values, None
    if kind in ("seg", "seg_sort"):
        off = _offsets(case)
        total = int(off[-1])
        at = torch.from_numpy(off).to(DEV)
        if kind == "seg":
            x = _values("f64", total, g)
            return torch.segment_reduce(x, "sum", offsets=at), None
        keys = _keys(case["dtype"], 32, total, g)
        if not keys.is_floating_point():
            return None
        seg = torch.repeat_interleave(torch.arange(case["nseg"], device=DEV), at[1:] - at[:-1])
        k, order = torch.sort(keys.double())
        return k[torch.sort(seg[order], stable=True).indices], None
    kinds, sizes, src, top = _requests(case)
    x = _request_sources(top, g)[0]
    sums = torch.zeros(case["nreq"], dtype=torch.float64, device=DEV)
    for i in range(case["nreq"]):
        if kinds[i] == 0:
            sums[i] = x[int(src[i]):int(src[i] + sizes[i])].sum()
    return [sums, None, None, None]
