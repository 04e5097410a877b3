"""The kernels that compile whole on the CPU (cpu_build/simt), against the oracle, as a program of its own: the test runs it
under AddressSanitizer, where every numpy array is a heap block of exactly its size."""
import ctypes
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(os.path.dirname(HERE)))
from oracle import oracle as O  # noqa: E402

P = O.P
I64, VP, SZ = ctypes.c_int64, ctypes.c_void_p, ctypes.c_size_t


def field(shape, seed):
    rng = np.random.default_rng(seed)
    a = rng.integers(0, 1 << 63, size=shape, dtype=np.uint64) * np.uint64(2) + rng.integers(0, 2, size=shape, dtype=np.uint64)
    return a % np.uint64(P)


def ptr(a):
    return a.ctypes.data if a is not None else None


def scratch(nbytes):
    """nbytes of garbage from an address that is a multiple of 8 only, nothing behind them."""
    a = np.full(nbytes + 8, 0xA5, dtype=np.uint8)
    assert a.ctypes.data % 16 == 0
    return a[8:]


def lookup(so):
    L = ctypes.CDLL(so)
    L.vi_lookup_histogram_workspace_bytes.restype = SZ
    L.vi_lookup_histogram_workspace_bytes.argtypes = [I64, I64, ctypes.c_int]
    L.vi_lookup_histogram.argtypes = [VP, I64, VP, I64, ctypes.c_int, ctypes.c_int, VP, VP, SZ, VP]
    L.vi_lookup_multiplicities.argtypes = [VP, I64, VP, I64, ctypes.c_int, VP, VP]

    def check(x, table, promised=0):
        n_x, n_t = len(x), len(table)
        keys, first = np.unique(table, return_index=True)
        at = np.minimum(np.searchsorted(keys, x), len(keys) - 1)
        hit = keys[at] == x if n_x else np.zeros(0, bool)
        want = np.bincount(first[at[hit]], minlength=n_t).astype(np.uint64)
        need = L.vi_lookup_histogram_workspace_bytes(n_x, n_t, promised)
        for accumulate, before in ((1, 7), (0, 12345)):
            mult, ws = np.full(n_t, before, dtype=np.uint64), scratch(need)
            rc = L.vi_lookup_histogram(ptr(x), n_x, None if promised else ptr(table), n_t, promised, accumulate, ptr(mult), ptr(ws), need, None)
            assert rc == 0 and np.array_equal(mult, want + np.uint64(before if accumulate else 0)), (n_x, n_t, promised, accumulate)
        mult = np.zeros(n_t, dtype=np.uint64)
        if n_x < 1000:
            assert L.vi_lookup_multiplicities(ptr(x), n_x, ptr(table), n_t, promised, ptr(mult), None) == 0
            assert np.array_equal(mult, want)

    # one and several groups, copies per entry, both sides of the small table, slices, one atomic per look-up
    for n_x, n_t in ((0, 5), (1, 1), (9000, 3), (500, 1024), (9001, 1025), (300, 4096), (9001, 4096), (9001, 4097), (700, 8191), (900, 8192),
                     (131073, 8192), (9001, 32771), (140001, 32772)):
        rng = np.random.default_rng(n_x + n_t)
        span = np.arange(n_t, dtype=np.uint64)
        x = rng.integers(0, n_t + n_t // 8 + 1, n_x).astype(np.uint64)
        x[-1:] = (1 << 64) - 1
        check(x, span)
        check(x, span, promised=1)
        if n_x > 100000:                                       # long runs, less often
            continue
        odd = span.copy()                                      # all but a range: the last entry, then the first
        odd[-1] = n_t + 1
        check(x, odd)
        odd[0] = 5 % n_t
        check(x, odd)
        table = field(n_t, n_x)
        table[n_t // 2:] = table[:n_t - n_t // 2][::-1]        # entries twice
        y = table[rng.integers(0, n_t, n_x)]
        y[::3] = field(len(y[::3]), 3)
        check(y, table)
    print("lookup", flush=True)


if __name__ == "__main__":
    globals()[sys.argv[1]](sys.argv[2])
    print("OK")
