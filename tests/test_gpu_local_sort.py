"""Ranges sorted by one block or wave (local_sort.hip): every length class at
its edges, alone (a span) and as segments of one plan, with keys that take
the bin placement (spread out) and the LSD passes (few distinct keys, a spike,
infinities), against numpy's stable argsort.  Exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EDGES = [1, 2, 63, 64, 65, 127, 128, 129, 255, 511, 512, 513, 1025, 2047, 2048, 2049, 5000, 5119, 5120, 5121, 8191, 8192]
TYPES = {"u32": np.uint32, "i32": np.int32, "f32": np.float32,
         "u64": np.uint64, "i64": np.int64, "f64": np.float64}
TORCH = {"u32": torch.uint32, "u64": torch.uint64}


def keys_of(name, how, n, rng):
    t = TYPES[name]
    if how == "equal":
        return np.full(n, 7, dtype=t)
    if how == "few":
        return rng.integers(0, 5, n).astype(t)
    if how == "small":
        return rng.integers(0, 4096, n).astype(t)
    if name[0] == "f":
        x = rng.standard_normal(n).astype(t)
        x[rng.random(n) < 0.02] = 0.0
        x[rng.random(n) < 0.02] = -0.0
        if how == "spike":
            x[:] = np.where(rng.random(n) < 0.9, t(1) + x * t(1e-6), x * t(1e30))
        if how == "ends":
            x[rng.random(n) < 0.1] = np.inf
            x[rng.random(n) < 0.1] = -np.inf
        return x
    info = np.iinfo(t)
    x = rng.integers(info.min, info.max, n, dtype=t, endpoint=True)
    if how == "spike":
        x = np.where(rng.random(n) < 0.9, x % t(50), x)
    if how == "ends":
        x[rng.random(n) < 0.1] = info.max
        x[rng.random(n) < 0.1] = info.min
    return x.astype(t)


def order_of(k, desc):
    if not desc:
        return np.argsort(k, kind="stable")
    if k.dtype.kind == "f":
        return np.argsort(-k, kind="stable")
    return np.argsort(~k, kind="stable")


def dev(a):
    if a.dtype.kind == "u":
        t = {4: (np.int32, torch.uint32), 8: (np.int64, torch.uint64)}[a.itemsize]
        return torch.from_numpy(a.view(t[0])).to(DEV).view(t[1])
    return torch.from_numpy(a).to(DEV)


def host(t, like):
    if like.dtype.kind == "u":
        return t.view({4: torch.int32, 8: torch.int64}[like.itemsize]).cpu().numpy().view(like.dtype)
    return t.cpu().numpy()


def same_bits(a, b):
    return np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("vb", [0, 4, 8])
@pytest.mark.parametrize("name", list(TYPES))
def test_span_and_segment_sorts_of_short_ranges(raja, name, vb):
    rng = np.random.default_rng([ord(c) for c in name] + [vb])
    for how in ("spread", "equal", "few", "small", "spike", "ends"):
        desc = how in ("spread", "few", "spike") and vb != 8
        comp = raja.operators.greater if desc else raja.operators.less
        parts = [keys_of(name, how, n, rng) for n in EDGES + [0, 3]]
        vt = np.int64 if vb == 8 else np.int32
        vals = [np.arange(len(p)).astype(vt)[::-1].copy() for p in parts]
        want = [order_of(p, desc) for p in parts]
        # as spans
        for p, v, o in zip(parts, vals, want):
            if len(p) == 0:
                continue
            k, w = dev(p), (dev(v) if vb else None)
            raja.sort_pairs(k, w, comp)
            assert same_bits(host(k, p), p[o]), (how, desc, len(p))
            if vb:
                assert np.array_equal(w.cpu().numpy(), v[o]), (how, desc, len(p))
        # as segments: few (one launch for all) and over 512 (a launch per length class)
        for reps in (1, 24):
            off = np.concatenate([[0], np.cumsum([len(p) for p in parts] * reps)])
            plan = raja.Segments(off)
            k, w = dev(np.concatenate(parts * reps)), (dev(np.concatenate(vals * reps)) if vb else None)
            raja.segmented_sort_pairs(plan, k, w, comp)
            assert same_bits(host(k, parts[0]), np.concatenate([p[o] for p, o in zip(parts, want)] * reps)), (how, reps)
            if vb:
                assert np.array_equal(w.cpu().numpy(), np.concatenate([v[o] for v, o in zip(vals, want)] * reps)), (how, reps)
            plan.close()
