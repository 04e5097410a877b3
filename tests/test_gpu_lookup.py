"""GPU parity: table multiplicities around the sizes at which the histogram changes shape (copies per entry, slices of the
table, rows of the workspace, one launch or two) and tables that go through the hash, against numpy counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from tests.gpu_util import rand_field, to_dev, to_np  # noqa: E402


def _counts(x, table):
    """First occurrence collects."""
    keys, first = np.unique(table, return_index=True)
    at = np.minimum(np.searchsorted(keys, x), len(keys) - 1)
    hit = keys[at] == x
    return np.bincount(first[at[hit]], minlength=len(table)).astype(np.uint64)


def _check(x, table):
    from verinf_amd.prover import cuda_primitives as cp
    dx, dt = to_dev(x), to_dev(table)
    want = _counts(x, table)
    assert np.array_equal(to_np(cp.lookup_multiplicities(dx, dt)), want)
    mult = to_dev(np.arange(len(table), dtype=np.uint64))
    cp.lookup_multiplicities_into(dx, dt, mult)
    assert np.array_equal(to_np(mult), want + np.arange(len(table), dtype=np.uint64))


@pytest.mark.parametrize("n_x", [1, 8192, 8193, 300001])
@pytest.mark.parametrize("n_table", [1, 63, 1024, 1025, 32768, 32769, 65536, 100003])
def test_range_tables(n_x, n_table):
    rng = np.random.default_rng(n_x + n_table)
    x = rng.integers(0, n_table + max(1, n_table // 8), n_x).astype(np.uint64)         # some beyond the table
    x[: n_x // 3] = n_table // 2                                                       # many of one entry
    x[-1] = np.uint64((1 << 64) - 1)
    _check(x, np.arange(n_table, dtype=np.uint64))


@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 1, (1 << 23) + 5])                 # 64 slices of 32768 entries, and more
@pytest.mark.parametrize("n_x", [50000, 200001])
def test_tables_of_many_slices(n_x, n):
    rng = np.random.default_rng(3)
    x = rng.integers(0, n + 1000, n_x).astype(np.uint64)
    x[:100] = n - 1
    _check(x, np.arange(n, dtype=np.uint64))
    _check(x * np.uint64(3), np.arange(n, dtype=np.uint64)[::-1] * np.uint64(3))


@pytest.mark.parametrize("n_x,n_table", [(1, 1), (1000, 3), (50001, 300), (200000, 4097), (100000, 40000)])
def test_other_tables(n_x, n_table):
    table = rand_field((n_table,), 7 + n_table)
    table[n_table // 2:] = table[: n_table - n_table // 2][::-1]                       # every entry twice, later ones unused
    table[-1] = 0
    rng = np.random.default_rng(n_table)
    x = table[rng.integers(0, n_table, n_x)]
    x[::7] = rand_field((len(x[::7]),), 9)
    _check(x, table)


@pytest.mark.parametrize("n_table", [512, 4096, 4097, 65536, 1 << 20])
def test_a_table_changed_in_place_is_looked_at_again(n_table):
    """The same storage holds a range, then one entry that is not its index (at either end and inside), then a range again."""
    from verinf_amd.prover import cuda_primitives as cp
    dt = to_dev(np.arange(n_table, dtype=np.uint64))
    rng = np.random.default_rng(n_table)
    x = np.concatenate([rng.integers(0, n_table, 200000).astype(np.uint64), [n_table + 5] * 9]).astype(np.uint64)
    x[:50] = 0
    x[50:90] = n_table - 1
    x[90:120] = n_table // 2
    dx = to_dev(x)
    for at in (None, 0, n_table - 1, n_table // 2, None):
        table = np.arange(n_table, dtype=np.uint64)
        if at is not None:
            table[at] = n_table + 5
        dt.copy_(to_dev(table))
        assert np.array_equal(to_np(cp.lookup_multiplicities(dx, dt)), _counts(x, table)), at


@pytest.mark.parametrize("n_x,n_table", [(100, 3000), (300001, 3000), (100000, 8192), (131073, 8192), (5000, 70000), (300001, 70000)])
def test_a_promised_range_needs_no_table(n_x, n_table):
    """table_is_range = 1 through the C ABI: no table is read."""
    from verinf_amd import _lib
    L = _lib.lib()
    x = np.random.default_rng(n_x).integers(0, n_table + 100, n_x).astype(np.uint64)
    dx, want = to_dev(x), _counts(x, np.arange(n_table, dtype=np.uint64))
    need = L.vi_lookup_histogram_workspace_bytes(n_x, n_table, 1)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    mult = to_dev(np.full(n_table, 7, dtype=np.uint64))
    for accumulate, plus in ((1, 7), (0, 0)):
        _lib.check(L.vi_lookup_histogram(dx.data_ptr(), n_x, None, n_table, 1, accumulate, mult.data_ptr(), ws.data_ptr(), need, _lib.stream_ptr()))
        assert np.array_equal(to_np(mult), want + np.uint64(plus))


def test_captured_calls_of_both_kinds_of_table():
    """The launches of a call do not depend on what the table holds: a graph captured over a range counts right after its
    table has become another one."""
    from verinf_amd.prover import cuda_primitives as cp
    n_x, n_table = 200000, 5000
    dx = to_dev(np.random.default_rng(1).integers(0, n_table, n_x).astype(np.uint64))
    dt = to_dev(np.arange(n_table, dtype=np.uint64))
    mult = torch.zeros(n_table, dtype=torch.int64, device="cuda").view(torch.uint64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        cp.lookup_multiplicities_into(dx, dt, mult)
        mult.view(torch.int64).zero_()
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        cp.lookup_multiplicities_into(dx, dt, mult)
    tables = [np.arange(n_table, dtype=np.uint64), rand_field((n_table,), 3), np.arange(n_table, dtype=np.uint64)[::-1].copy()]
    want = np.zeros(n_table, dtype=np.uint64)
    for i, table in enumerate(tables):
        dt.copy_(to_dev(table))
        x = table[np.random.default_rng(i).integers(0, n_table, n_x)]
        dx.copy_(to_dev(x))
        g.replay()
        torch.cuda.synchronize()
        want += _counts(x, table)
        assert np.array_equal(to_np(mult), want), i


def test_a_table_beyond_the_hash():
    """More than 2^30 entries: a range is indexed, another table searched from the front."""
    from verinf_amd.prover import cuda_primitives as cp
    n_table = (1 << 30) + 7
    table = torch.arange(n_table, dtype=torch.int64, device="cuda")
    x = np.array([0, n_table - 1, n_table - 1, n_table, 12345] + [5] * 30, dtype=np.uint64)
    got = cp.lookup_multiplicities(to_dev(x), table.view(torch.uint64)).view(torch.int64)
    assert got[[0, 5, 12345, n_table - 1]].tolist() == [1, 30, 1, 2] and int(got.sum()) == 34
    table[n_table - 1] = 3                                     # entries near the front only: a search walks up to them
    got = cp.lookup_multiplicities(to_dev(x[4:]), table.view(torch.uint64)).view(torch.int64)
    assert got[[5, 12345]].tolist() == [30, 1] and int(got.sum()) == 31
    del got, table
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n_table", [3000, 40000])
@pytest.mark.parametrize("skip", [0, 4, 8])
def test_scratch_of_any_alignment(n_table, skip):
    from verinf_amd import _lib
    L = _lib.lib()
    table = rand_field((n_table,), 4)
    x = table[np.random.default_rng(2).integers(0, n_table, 300000)]
    dx, dt = to_dev(x), to_dev(table)
    need = L.vi_lookup_histogram_workspace_bytes(len(x), n_table, 0)
    ws = torch.full((need + skip + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    mult = torch.empty(n_table, dtype=torch.uint64, device="cuda")
    _lib.check(L.vi_lookup_histogram(dx.data_ptr(), len(x), dt.data_ptr(), n_table, 0, 0, mult.data_ptr(), ws.data_ptr() + skip, need, _lib.stream_ptr()))
    assert np.array_equal(to_np(mult), _counts(x, table))
    assert bool((ws[:skip] == 0x5A).all()) and bool((ws[need + skip:] == 0x5A).all())


@pytest.mark.parametrize("n_x,n_table", [(131073, 8192), (140001, 8193), (300001, 65535), (1500001, 65536), (140001, 65537), (400000, 131073),
                                         (256 * 65535, 65536), (256 * 65535 + 1, 65536)])
@pytest.mark.parametrize("kind", ["range", "one entry", "other"])
def test_counters_of_16_bits(n_x, n_table, kind):
    """Tables from 8192 entries on: one and two slices, odd lengths, up to as many look-ups of one entry as such a counter holds."""
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(n_x + n_table)
    at = rng.integers(0, n_table, n_x)
    at[:n_x if kind == "one entry" else n_x // 3] = n_table - 1
    table = np.arange(n_table, dtype=np.uint64)
    if kind == "other":
        table = table * np.uint64(0x9E3779B97F4A7C15)          # different, as the factor is odd
    print(n_x, n_table, kind, flush=True)
    x = table[at]
    got = to_np(cp.lookup_multiplicities(to_dev(x), to_dev(table)))
    assert np.array_equal(got, np.bincount(at, minlength=n_table).astype(np.uint64))


@pytest.mark.parametrize("n_table", [8192, 8193, 16384, 16385, 32768])
@pytest.mark.parametrize("n_x", [131073, 1500001, 256 * 65535])
def test_few_entries_of_16_bit_counters(n_x, n_table):
    """Four, two and one copy per entry, whose sums are what a counter holds at most."""
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(n_x + n_table)
    few = np.array([0, 1, 2, n_table // 2, n_table - 2, n_table - 1], dtype=np.uint64)
    print(n_x, n_table, flush=True)
    for hot in (few, few[-1:]):
        x = hot[rng.integers(0, len(hot), n_x)]
        want = np.bincount(x.astype(np.int64), minlength=n_table).astype(np.uint64)
        for table in (np.arange(n_table, dtype=np.uint64), rng.permutation(n_table).astype(np.uint64)):
            got = to_np(cp.lookup_multiplicities(to_dev(x), to_dev(table)))
            assert np.array_equal(got, want[table.astype(np.int64)])
