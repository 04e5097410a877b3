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
    cp._range_table_cache.clear()                              # tables of this test come and go at the same addresses
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
