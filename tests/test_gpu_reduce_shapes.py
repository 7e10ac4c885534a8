"""Span and segmented reductions at the edges of their units (wave tile, quad,
tile, and the span lengths where the launch shape changes).  The FP data are
integer-valued, so every order of summation is exact; values repeat, so the
first-index rule of MinLoc / MaxLoc is seen."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# wave tile, quad and tile of 8-byte elements; 4-byte ones have twice as many
W, Q, T = 2048, 8192, 32768
EDGES = [1, 3, 64, W - 1, W, W + 1, Q - 1, Q, Q + 1, 2 * Q, 2 * Q + 1, T - 1, T, T + 1, 4 * T + Q + 5,
         128 * T - 1, 128 * T, 128 * T + 1, 1024 * T, 1024 * T + 1, 1040 * T + 77]


def data(n, dtype, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randint(-9999, 10000, (n,), generator=g, device=DEV, dtype=torch.int32).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.int32, torch.float32])
@pytest.mark.parametrize("shift", [0, 1])
def test_span_reductions_at_unit_edges(raja, dtype, shift):
    per = 2 if dtype in (torch.int32, torch.float32) else 1
    for n in EDGES:
        if per * n > (1 << 26):
            n = (1 << 26) // per + 13
        m = per * n if n % 2 else per * n + per - 1
        buf = data(m + 1, dtype, m)
        x = buf[shift:m + shift]  # shift 1: not 16-byte aligned
        h = x.cpu().numpy()
        tot = int(h.astype(np.int64).sum())
        if dtype == torch.float32:  # exact while partial sums stay below 2^24
            x = torch.sign(x)
            h = x.cpu().numpy()
            tot = int(h.astype(np.int64).sum())
        assert int(raja.reduce_sum(x).item()) == (tot if dtype != torch.int32 else np.int64(tot).astype(np.int32)), m
        assert raja.reduce_min(x).item() == h.min() and raja.reduce_max(x).item() == h.max(), m
        v, i = raja.reduce_minloc(x)
        assert (v.item(), i.item()) == (h.min(), int(h.argmin())), m
        v, i = raja.reduce_maxloc(x)
        assert (v.item(), i.item()) == (h.max(), int(h.argmax())), m
        if dtype == torch.float64:
            r = raja.unpack_multi(raja.multi_reduce_f64(x))
            assert r == {"sum": tot, "min": h.min(), "max": h.max(), "minloc_val": h.min(),
                         "minloc_loc": int(h.argmin())}, m


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64, torch.int32])
def test_segmented_reductions_at_unit_edges(raja, dtype):
    per = 2 if dtype == torch.int32 else 1
    lens = [0, 1, 0] + [per * n + d for n in EDGES[:15] for d in (0, 1)] + [0]
    off = np.concatenate([[0], np.cumsum(lens)])
    x = data(int(off[-1]), dtype, 3)
    h = x.cpu().numpy()
    plan = raja.Segments(off)
    for op, f, ident in ((raja.operators.plus, np.sum, 7), (raja.operators.minimum, np.min, 20000),
                         (raja.operators.maximum, np.max, -20000)):
        got = raja.segmented_reduce(plan, x, op, ident).cpu().numpy()
        for s in range(plan.nseg):
            seg = h[off[s]:off[s + 1]]
            want = ident if len(seg) == 0 else f([ident, f(seg)])
            assert got[s] == want, (s, lens[s], op)
    # FP data with rounding: a segment's bits alone and in the batch
    if dtype == torch.float64:
        y = torch.randn(int(off[-1]), device=DEV, dtype=torch.float64)
        got = raja.segmented_reduce(plan, y, raja.operators.plus, 0.0).cpu().numpy()
        for s in range(plan.nseg):
            assert raja.reduce_sum(y[off[s]:off[s + 1]], 0.0).item() == got[s], (s, lens[s])
    plan.close()
