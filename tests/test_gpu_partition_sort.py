"""Long spans sorted by partition (partition_sort.hip) against torch's stable
sort of the keys' ordered bits: the lengths where the number of scatters
changes, key sets that the partition takes, that its sample rejects and that
only the exact counts reject (they then take the LSD passes), both directions,
all key and value widths.  Exact, values included."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
INT = {4: torch.int32, 8: torch.int64}
U = {"u32": torch.uint32, "u64": torch.uint64}
ONE = 256 * 4700  # longest one-level span
BUCKET = 256 * 2201  # from here on a group needs the larger block


def bits_of(raw, name):
    """Signed 64-bit integers in the order of the keys (raw: the keys' bits as a signed integer)."""
    x = raw.to(torch.int64)
    if name == "u32":
        return x & 0xFFFFFFFF
    if name == "u64":
        return x ^ (-2 ** 63)
    if name[0] == "f":
        top = -2 ** 31 if name == "f32" else -2 ** 63
        x = torch.where(x == top, torch.zeros_like(x), x)  # -0.0 == +0.0
        return torch.where(x < 0, (~x) ^ top, x) if name == "f64" else torch.where(x < 0, -(x & 0x7FFFFFFF) - 1, x)
    return x


def keys_of(name, how, n, g):
    size = 4 if name[1:] == "32" else 8
    if name[0] == "f":
        dt = torch.float32 if size == 4 else torch.float64
        x = torch.rand(n, generator=g, device=DEV, dtype=dt) if how == "uniform" else \
            torch.randn(n, generator=g, device=DEV, dtype=dt)
        if how == "zeros":
            x = torch.round(x * 2000) / 2000  # ties, -0.0 among them
        if how == "ends":
            x[:: n // 50] = float("inf")
            x[1:: n // 60] = -float("inf")
        if how == "few":
            x = torch.round(x)
        return x.view(INT[size]), x
    if how == "few":
        raw = torch.randint(0, 7, (n,), generator=g, device=DEV, dtype=INT[size])
    elif how == "zeros":  # 2^12 distinct keys
        raw = torch.randint(0, 1 << 12, (n,), generator=g, device=DEV, dtype=INT[size])
    elif how == "ends":  # uniform in a narrow range with outliers far away
        raw = torch.randint(1000, 50_000_000, (n,), generator=g, device=DEV, dtype=INT[size])
        raw[:: n // 30] = torch.iinfo(INT[size]).max
        raw[1:: n // 40] = torch.iinfo(INT[size]).min
    elif how == "normal":
        raw = (torch.randn(n, generator=g, device=DEV, dtype=torch.float64) * 2 ** 27).to(INT[size])
    elif how == "spike":  # one bucket too full, too thin for the sample to see: one level has
        # buckets of up to 4700 on average and room for 5120, two levels far smaller ones
        raw = torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g, device=DEV, dtype=INT[size])
        raw[n // 2: n // 2 + (1200 if n <= ONE else 9000)] = 12345
    else:
        raw = torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g, device=DEV, dtype=torch.int64)
        if size == 8:
            raw = (raw << 32) | torch.randint(0, 2 ** 32, (n,), generator=g, device=DEV, dtype=torch.int64)
        raw = raw.to(INT[size])
    return raw, raw.view(U[name]) if name in U else raw


def routed(raja, sort):
    """Launches of the sort's phases: sample, counts, scatters, block sorts, digit passes."""
    raja.timing_enable(True)
    try:
        raja.timing_reset()
        sort()
        return tuple(raja.timing_query(p)["count"] for p in (
            "partition_sample", "partition_hist", "partition_scatter", "partition_local", "onesweep_pass"))
    finally:
        raja.timing_enable(False)


def check(raja, name, vb, desc, how, n, shift=0):
    """Sorts and compares; returns the sort's route."""
    g = torch.Generator(device=DEV)
    g.manual_seed(n + vb)
    raw, keys = keys_of(name, how, n, g)
    want = bits_of(raw, name)
    order = torch.sort(~want if desc else want, stable=True).indices
    size = raw.element_size()
    room = torch.empty(n + shift, dtype=keys.dtype, device=DEV)
    k = room[shift:]
    k.view(INT[size]).copy_(raw) if shift == 0 else room.view(INT[size])[shift:].copy_(raw)
    v = torch.arange(n, device=DEV, dtype=INT[vb]) if vb else None
    route = routed(raja, lambda: raja.sort_pairs(k, v, raja.operators.greater if desc else raja.operators.less))
    assert torch.equal(room.view(INT[size])[shift:], raw[order]), (name, vb, desc, how, n)
    if vb:
        assert torch.equal(v.to(torch.int64), order), (name, vb, desc, how, n)
    raja.device_status()
    return route


def levels(name, vb, n):
    """Levels the partition has for a span of this length (0: digit passes)."""
    if n < 1 << 18 or n > 65536 * 4700:
        return 0
    if n <= ONE:
        return 1
    if name[1:] == "64":
        return 2 if n >= 1 << 22 else 0
    return 2 if vb and n >= 1 << 25 else 0


ACCEPTED = {0: (0, 0, 0, 0), 1: (1, 1, 1, 1), 2: (1, 1, 2, 1)}


@pytest.mark.parametrize("name", ["u32", "i32", "f32", "u64", "i64", "f64"])
@pytest.mark.parametrize("how", ["uniform", "normal", "zeros", "few", "ends"])
def test_key_sets(raja, name, how):
    for n, vb, desc in ((400_003, 4, False), (1 << 22, 8, True), ((1 << 22) + 54321, 0, False), (600_000, 0, True)):
        check(raja, name, vb, desc, how, n)


@pytest.mark.parametrize("name,vb,n", [
    ("u32", 4, (1 << 18) - 1), ("u32", 4, 1 << 18), ("u32", 4, (1 << 18) + 1), ("u32", 4, ONE), ("u32", 4, ONE + 1),
    ("u32", 4, (1 << 22) - 1), ("i32", 0, ONE), ("f32", 8, BUCKET - 1), ("f32", 8, BUCKET), ("u64", 4, BUCKET),
    ("i64", 8, ONE - 1), ("u32", 4, (1 << 25) + 7), ("u32", 8, (1 << 25) - 1), ("u32", 4, 9 * (1 << 24) + 11), ("u64", 0, 1 << 22),
    ("u64", 4, (1 << 24) + 3), ("i64", 8, 330 * 65536), ("i64", 0, 1200 * 65536), ("f64", 4, (1 << 23) + 1)])
def test_lengths(raja, name, vb, n):
    want = ACCEPTED[levels(name, vb, n)]
    assert check(raja, name, vb, False, "uniform", n)[:4] == want
    assert check(raja, name, vb, True, "uniform", n, shift=1)[:4] == want


@pytest.mark.parametrize("name,n", [("i32", ONE), ("i32", (1 << 25) + 3), ("i64", ONE), ("i64", 1 << 22)])
def test_counts_reject_what_the_sample_allows(raja, name, n):
    """The sample and the counts run, the first scatter is launched and ends at
    once, no block sorts follow: the digit passes sort."""
    route = check(raja, name, 4, False, "spike", n)
    assert route[:4] == (1, 1, 1, 0) and route[4] > 0


@pytest.mark.parametrize("name,n", [
    ("u32", (1 << 18) + 1), ("i32", ONE), ("f32", ONE - 5), ("u64", (1 << 18) + 3), ("f64", ONE), ("i64", (1 << 22) + 1),
    ("f64", (1 << 22) + 7), ("i32", (1 << 25) + 1)])
def test_refused_keys(raja, name, n):
    """Keys whose digits the partition counts after its sample has refused them:
    in place at any alignment, both directions, 0, 4 and 8 value bytes."""
    for vb, desc, shift in ((4, False, 1), (0, True, 0), (8, True, 3), (4, False, 0)):
        route = check(raja, name, vb, desc, "few", n, shift)
        # one level counts and launches its scatter without the answer, two levels do not
        assert route[:4] == {0: (0, 0, 0, 0), 1: (1, 1, 1, 0), 2: (1, 0, 0, 0)}[levels(name, vb, n)]
        assert route[4] > 0


def test_sorted_and_reversed(raja):
    for n in (1_000_003, 5_000_011):
        for rev in (False, True):
            x = torch.arange(n, device=DEV, dtype=torch.int32)
            raw = (x.flip(0) if rev else x).contiguous()
            k, v = raw.clone(), torch.arange(n, device=DEV, dtype=torch.int32)
            raja.sort_pairs(k, v)
            assert torch.equal(k, x) and torch.equal(v, raw), (n, rev)


@pytest.mark.parametrize("name,how,n", [("u64", "uniform", 1 << 22), ("u64", "few", 1 << 22), ("u32", "uniform", 2_000_003)])
def test_behind_a_long_queue(raja, name, how, n):
    """The host polls the device's answers while tens of milliseconds of other
    work on the stream come first."""
    room = torch.empty(1 << 28, dtype=torch.int32, device=DEV)
    g = torch.Generator(device=DEV)
    g.manual_seed(n)
    raw, keys = keys_of(name, how, n, g)
    order = torch.sort(bits_of(raw, name), stable=True).indices
    k, v = keys.clone(), torch.arange(n, device=DEV, dtype=torch.int32)
    torch.cuda.synchronize()
    for i in range(60):
        room.fill_(i)
    raja.sort_pairs(k, v)
    assert torch.equal(k.view(raw.dtype), raw[order]) and torch.equal(v.to(torch.int64), order)
