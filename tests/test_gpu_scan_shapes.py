"""Span scans at the edges of every tile shape (one-tile spans, the lengths
where the shape changes, partial tiles and vectors), from element-aligned
slices and in place, against numpy.  Exact: integers, and min/max of floats."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EDGES4 = [1, 2, 3, 5, 255, 256, 257, 1023, 1024, 1025, 8191, 8192, 8193, 16383, 16384, 16385, 32767,
          32768, 32769, 70001, 512 * 8192, 512 * 8192 + 1]
EDGES8 = [1, 2, 3, 127, 128, 129, 383, 384, 385, 3071, 3072, 3073, 6143, 6144, 6145, 12287, 12288, 12289,
          64 * 3072, 64 * 3072 + 1, 192 * 6144, 192 * 6144 + 1]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64, torch.float32, torch.float64])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_span_scans_at_shape_edges(raja, dtype, shift):
    small = dtype in (torch.int32, torch.float32)
    g = torch.Generator(device=DEV)
    g.manual_seed(shift)
    for n in EDGES4 if small else EDGES8:
        base = torch.randint(-99, 100, (n + shift,), generator=g, device=DEV, dtype=torch.int32).to(dtype)
        x = base[shift:]
        h = x.cpu().numpy()
        room = torch.full((n + shift + 8,), 55, dtype=dtype, device=DEV)
        out = room[shift:n + shift]
        if not dtype.is_floating_point:
            raja.exclusive_scan(x, out, raja.operators.plus, 7)
            want = np.concatenate([[7], 7 + np.cumsum(h, dtype=h.dtype)[:-1]]).astype(h.dtype)
            assert np.array_equal(out.cpu().numpy(), want), n
            y = x.clone()
            raja.inclusive_scan_inplace(y)
            assert np.array_equal(y.cpu().numpy(), np.cumsum(h, dtype=h.dtype)), n
        raja.inclusive_scan(x, out, raja.operators.minimum)
        assert np.array_equal(out.cpu().numpy(), np.minimum.accumulate(h)), n
        raja.inclusive_scan(x, out, raja.operators.maximum)
        assert np.array_equal(out.cpu().numpy(), np.maximum.accumulate(h)), n
        edge = room.cpu().numpy()  # nothing written outside the span
        assert np.all(edge[:shift] == 55) and np.all(edge[n + shift:] == 55), n
    raja.device_status()
