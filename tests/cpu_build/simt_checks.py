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

    def counts(x, table):
        keys, first = np.unique(table, return_index=True)
        at = np.minimum(np.searchsorted(keys, x), len(keys) - 1)
        hit = keys[at] == x if len(x) else np.zeros(0, bool)
        return np.bincount(first[at[hit]], minlength=len(table)).astype(np.uint64)

    # the first calls of the library, whose tags are known: scratch that holds slots of that very tag, naming any index or none, in
    # some of the slots and in all of them
    tags = [1 << 63 | (n * 0x9E3779B97F4A7C15 & (1 << 33) - 1) << 30 for n in range(2)]
    rng = np.random.default_rng(0)
    n_t = 5000
    table = field(n_t, 1)
    table[::4] = np.arange(0, n_t, 4)                          # some entries are their own index
    table[1::4] = table[rng.integers(0, n_t, len(table[1::4]))]
    x = np.concatenate([table[rng.integers(0, n_t, 9001)], np.arange(0, 600, dtype=np.uint64)])
    ws = scratch(L.vi_lookup_histogram_workspace_bytes(len(x), n_t, 0))
    slots = ws[(-ws.ctypes.data) % 16:][:8 << 14].view(np.uint64)
    mult = np.empty(n_t, dtype=np.uint64)
    for tag, share in zip(tags, (0.4, 1.0)):
        taken = rng.random(len(slots)) < share
        slots[taken] = (np.uint64(tag) | rng.integers(0, 2 * n_t, len(slots)).astype(np.uint64))[taken]
        assert L.vi_lookup_histogram(ptr(x), len(x), ptr(table), n_t, 0, 0, ptr(mult), ptr(ws), len(ws), None) == 0
        assert np.array_equal(mult, counts(x, table)), share
        found = int(ws[(-ws.ctypes.data) % 16:][8 << 14:][:4].view(np.uint32)[0])
        assert found == (7 if share == 1.0 else 3)             # off and on the diagonal, and entries without a slot
    for seed in (2, 3):                                        # the same scratch again, with slots of the calls before
        table = np.random.default_rng(seed).permutation(table)
        assert L.vi_lookup_histogram(ptr(x), len(x), ptr(table), n_t, 0, 0, ptr(mult), ptr(ws), len(ws), None) == 0
        assert np.array_equal(mult, counts(x, table))

    def check(x, table, promised=0):
        n_x, n_t = len(x), len(table)
        want = counts(x, table)
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
                     (131073, 8192), (140001, 8193), (131073, 16384), (140001, 16385), (9001, 32771), (140001, 32772), (140001, 65539)):
        rng = np.random.default_rng(n_x + n_t)
        span = np.arange(n_t, dtype=np.uint64)
        x = rng.integers(0, n_t + n_t // 8 + 1, n_x).astype(np.uint64)
        x[-1:] = (1 << 64) - 1
        check(x, span)
        check(x, span, promised=1)
        odd = span.copy()                                      # all but a range: the last entry, then the first
        odd[-1] = n_t + 1
        check(x, odd)
        if n_t > 4097:                                         # long runs, less often
            continue
        odd[0] = 5 % n_t
        check(x, odd)
        table = field(n_t, n_x)
        table[n_t // 2:] = table[:n_t - n_t // 2][::-1]        # entries twice
        y = table[rng.integers(0, n_t, n_x)]
        y[::3] = field(len(y[::3]), 3)
        check(y, table)
    print("lookup", flush=True)


def _ntt_lib(so):
    L = ctypes.CDLL(so)
    for name in ("vi_ntt_workspace_bytes", "vi_ntt_best_workspace_bytes"):
        getattr(L, name).restype, getattr(L, name).argtypes = SZ, [I64, I64]
    L.vi_ntt_batched.argtypes = [VP, I64, I64, ctypes.c_int, VP, SZ, VP]
    L.vi_coset_lde_workspace_bytes.restype, L.vi_coset_lde_workspace_bytes.argtypes = SZ, [I64, I64, I64]
    L.vi_coset_lde_min_workspace_bytes.restype, L.vi_coset_lde_min_workspace_bytes.argtypes = SZ, [I64, I64]
    L.vi_coset_lde_launches.restype, L.vi_coset_lde_launches.argtypes = I64, [I64, I64, I64, SZ]
    L.vi_coset_lde.argtypes = [VP, I64, I64, I64, I64, I64, ctypes.c_uint64, VP, I64, VP, SZ, VP]
    L.vi_coset_lde_coeffs.argtypes = [VP, I64, I64, I64, I64, I64, ctypes.c_uint64, VP, I64, VP, I64, VP, SZ, VP]
    L.vi_coset_extend.argtypes = [VP, I64, I64, I64, I64, I64, ctypes.c_uint64, VP, I64, VP, SZ, VP]
    L.simt_launches.restype = ctypes.c_long
    return L


def ntt(so):
    """Transforms through vi_ntt_batched: every length class, at the batch sizes that take few-row kernels."""
    L = _ntt_lib(so)
    row_switch = os.environ.get("VI_NTT_ROW") != "0"

    def run(rows, inverse, ws_bytes=None):
        m, n = rows.shape
        ws = scratch(L.vi_ntt_best_workspace_bytes(m, n) if ws_bytes is None else ws_bytes)
        before = L.simt_launches()
        rc = L.vi_ntt_batched(ptr(rows), m, n, inverse, ptr(ws) if len(ws) else None, len(ws), None)
        return rc, L.simt_launches() - before

    for logn, m in [(1, 3), (2, 5), (3, 1), (3, 130), (4, 70), (5, 33), (6, 1), (7, 9), (8, 5), (9, 3), (10, 2), (11, 1), (11, 3), (12, 1), (12, 3), (13, 2),
                    (14, 1), (15, 1), (16, 1), (17, 1)]:
        n = 1 << logn
        raw = field((m, n), logn + m)
        raw[-1, -2:] = [(1 << 64) - 1, P + 1]
        want = raw % np.uint64(P)
        a = raw.copy()
        rc, launches = run(a, 0)
        assert rc == 0 and np.array_equal(a, O.ntt_rows(want)), (logn, m)
        if 3 <= logn <= 11:                                    # the single launch, or the passes the switch asks for
            assert launches == (1 if row_switch or logn < 10 else 2), (logn, launches)
        rc, _ = run(a, 1)
        assert rc == 0 and np.array_equal(a, want), (logn, m)
        if logn >= 12:                                         # one row of scratch: the rows one after the other
            a = raw.copy()
            rc, _ = run(a, 0, 8 * n)
            assert rc == 0 and np.array_equal(a, O.ntt_rows(want)), (logn, m)
        # without scratch: rows of up to 2^12 points need none, unless the switch asks for their two passes
        a = raw.copy()
        rc, _ = run(a, 0, 0)
        assert (rc == 0) == (logn <= (12 if row_switch else 9)), (logn, rc)
        if rc == 0:
            assert np.array_equal(a, O.ntt_rows(want))
    print("ntt", flush=True)


def lde(so):
    """Extensions through the three entry points: values, coefficients beside and in place, from coefficients; strided sources of
    any width, one to 32 cosets, scratch for all rows and for one."""
    L = _ntt_lib(so)

    def check(logK, log_rho, m, w, shift):
        K, N = 1 << logK, 1 << (logK + log_rho)
        stride = w + 3
        flat = field((m - 1) * stride + w, logK + w)           # the last row ends with its last word
        src = np.lib.stride_tricks.as_strided(flat, (m, w), (8 * stride, 8))
        rows = np.ascontiguousarray(src)
        want = O.coset_lde_rows(rows, K, N, shift)
        padded = np.zeros((m, K), dtype=np.uint64)
        padded[:, :w] = rows
        want_c = O.ntt_rows(padded, inverse=True)
        for nbytes in (L.vi_coset_lde_workspace_bytes(m, K, N), L.vi_coset_lde_min_workspace_bytes(K, N)):
            ws = scratch(nbytes)
            what = (logK, log_rho, m, w, nbytes)
            out = np.empty((m, N), dtype=np.uint64)
            before = L.simt_launches()
            assert L.vi_coset_lde(ptr(flat), m, w, stride, K, N, shift, ptr(out), N, ptr(ws), nbytes, None) == 0
            assert np.array_equal(out, want), what
            assert L.simt_launches() - before == L.vi_coset_lde_launches(m, K, N, nbytes), what
            out = np.empty((m, N), dtype=np.uint64)
            co = np.empty((m, K), dtype=np.uint64)
            assert L.vi_coset_lde_coeffs(ptr(flat), m, w, stride, K, N, shift, ptr(co), K, ptr(out), N, ptr(ws), nbytes, None) == 0
            assert np.array_equal(out, want) and np.array_equal(co, want_c), what
            co = np.empty((m, K), dtype=np.uint64)
            assert L.vi_coset_lde_coeffs(ptr(flat), m, w, stride, K, N, shift, ptr(co), K, None, N, ptr(ws), nbytes, None) == 0
            assert np.array_equal(co, want_c), what
            out = np.empty((m, N), dtype=np.uint64)
            assert L.vi_coset_extend(ptr(co), m, K, K, K, N, shift, ptr(out), N, ptr(ws), nbytes, None) == 0
            assert np.array_equal(out, want), what
            own, out = padded.copy(), np.empty((m, N), dtype=np.uint64)
            assert L.vi_coset_lde_coeffs(ptr(own), m, K, K, K, N, shift, ptr(own), K, ptr(out), N, ptr(ws), nbytes, None) == 0
            assert np.array_equal(out, want) and np.array_equal(own, want_c), what

    for logK in range(1, 13):
        for log_rho in (0, 1, 2, 3, 5):
            if logK + log_rho > 14:
                continue
            K = 1 << logK
            check(logK, log_rho, 3 if logK < 10 else 1, [1, K - 1, K][(logK + log_rho) % 3] or 1, 7)
    for logK, log_rho, m, w in ((3, 1, 300, 5), (6, 2, 70, 64), (10, 3, 2, 600), (11, 3, 1, 2048), (13, 1, 2, 5000), (13, 2, 1, 8192), (14, 0, 1, 100),
                                (14, 2, 1, 9000)):
        check(logK, log_rho, m, w, 11)
    check(10, 2, 257, 1000, 11)                                # rows in one launch
    print("lde", flush=True)


def small(shape, seed, fill):
    """Signed 16-bit numbers mod p: any, the largest, the lowest."""
    x = np.random.default_rng(seed).integers(-(1 << 15), 1 << 15, shape)
    x[:] = {"top": (1 << 15) - 1, "low": -(1 << 15)}.get(fill.split()[-1], x)
    return np.where(x < 0, x.astype(np.uint64) + np.uint64(P), x.astype(np.uint64))


def matmul(so):
    """Products through residues: every tile shape with remainders, one unit of the inner dimension and several, the largest sums of
    either sign, words at and above p, slices of the inner dimension."""
    L = ctypes.CDLL(so)
    L.simt_matmul_workspace.restype, L.simt_matmul_workspace.argtypes = SZ, [I64] * 3
    L.simt_matmul.argtypes = [VP, VP, VP, I64, I64, I64, VP]
    L.simt_tile_workspace.restype, L.simt_tile_workspace.argtypes = SZ, [I64, ctypes.c_int]
    L.simt_tile.restype, L.simt_tile.argtypes = None, [VP, VP, VP, I64, I64, I64, ctypes.c_int, VP]
    for m, k, n, fill in ((1, 1, 1, None), (3, 17, 70, "any"), (64, 64, 64, "top"), (65, 100, 65, "half"), (130, 33, 130, None), (5, 8193, 3, "top"),
                          (120, 70, 250, 4), (128, 64, 256, 4), (128, 130, 128, 2), (67, 5, 100, 2), (65, 4001, 66, 2),
                          (3, 17, 70, "i16"), (64, 64, 128, "i16 top"), (65, 129, 130, "i16"), (5, 1030, 3, "i16 low"), (70, 65, 40, "over a"), (40, 130, 300, "over b"),
                          # residues by one workgroup per slab; more items than workgroups cut up
                          (3, 8190, 2, "any"), (2, 32768, 3, "i16")):
        print("matmul", m, k, n, fill, flush=True)
        A, B = field((m, k), m), field((k, n), n)
        if fill == "top":
            A[:], B[:] = P - 1, P - 1
        elif fill == "half":                                   # the words of largest size as signed numbers
            A[:], B[:] = 0x8080808080808080, 0x7F7F7F7F7F7F7F7F
            B[::2] += np.uint64(1)
        elif isinstance(fill, str) and fill != "any":          # 16-bit signed numbers, the last word of A or B one beyond them
            A[:] = small((m, k), 1, fill)
            B[:] = small((k, n), 2, fill)
            if fill.startswith("over"):
                (A if fill == "over a" else B)[-1, -1] = (1 << 15) if fill == "over a" else P - (1 << 15) - 1
        elif fill == "any":
            A[:, ::3] = np.uint64((1 << 64) - 1) - A[:, ::3] % np.uint64(1 << 20)
            B[::2] = np.uint64((1 << 64) - 1) - B[::2] % np.uint64(1 << 33)
        C = np.empty((m, n), dtype=np.uint64)
        if fill in (2, 4):                                     # one tile of 128 x 64 fill
            ws = scratch(L.simt_tile_workspace(k, fill))
            L.simt_tile(ptr(A), ptr(B), ptr(C), m, k, n, fill, ptr(ws))
        else:
            ws = scratch(L.simt_matmul_workspace(m, k, n))
            assert L.simt_matmul(ptr(A), ptr(B), ptr(C), m, k, n, ptr(ws)) == 0
        rows = sorted({0, m // 2, m - 1})
        want = (A[rows].astype(object).dot(B.astype(object)) % P).astype(np.uint64)
        assert np.array_equal(C[rows], want), (m, k, n, fill)


def tables(so):
    """The tables of a call stay until its launches are queued, whatever other threads' calls evict in between."""
    L = _ntt_lib(so)
    for K, N in ((64, 128), (1 << 13, 1 << 14)):               # the single launch, and passes
        a, out = field((2, K), 1), np.empty((2, N), dtype=np.uint64)
        ws = scratch(L.vi_coset_lde_workspace_bytes(2, K, N))
        L.simt_other_shifts(40)
        assert L.vi_coset_lde(ptr(a), 2, K, K, K, N, 7, ptr(out), N, ptr(ws), len(ws), None) == 0
        assert np.array_equal(out, O.coset_lde_rows(a, K, N, 7))
    print("tables", flush=True)


# Sums that take every route of vi_sumcheck_prove_coins: products with kernels of their own, the hadamard gate, sums under a common
# factor (table 0) in all their forms, other sums in registers, in memory and beyond one descriptor.
SUMS = {
    "one": [(5, [0])],
    "two": [(7, [0, 1])],
    "three": [(1, [0, 1, 2])],
    "four": [(3, [0, 1, 2, 3])],
    "gate": [(3, [0, 1, 2]), (P - 3, [0, 3])],
    "products": [(3, [0, 1, 2]), (5, [0, 3, 4])],
    "singles": [(3, [0, 1]), (P - 7, [2, 0]), (11, [0, 3])],
    "constant": [(3, [0, 1]), (P - 2, [0])],
    "only a constant beside products": [(3, [0, 1, 2]), (9, [0])],
    "mixed": [(3, [0, 1, 2]), (P - 3, [0, 3]), (9, [4, 0]), (6, [0, 5, 5]), (P - 6, [0, 5]), (4, [0])],
    "shared": [(3, [0, 1, 2]), (5, [1, 0, 3]), (7, [2, 3, 0]), (8, [0, 1]), (0, [0, 1, 3])],
    "common twice": [(3, [0, 0, 1]), (5, [0, 0]), (2, [1, 2, 0])],
    "many": [(k + 1, [0, k % 37 + 1]) for k in range(50)] + [(k + 2, [0, k + 1, k + 18]) for k in range(20)],
    "registers": [(3, [0, 1]), (4, [2, 3])],
    "memory": [(k + 3, [k, k + 1, 10 - k]) for k in range(10)],
    "degree four": [(2, [0, 1, 2, 3]), (3, [0, 4])],
    "rewritten": [(2, [0, 1, 2])] + [(k + 2, [0, 3 + k]) for k in range(130)],
}


def sumcheck(so):
    """Proofs with work buffers and scratch of exactly the stated sizes, tables apart from them and folded in place."""
    L = ctypes.CDLL(so)
    L.vi_sumcheck_prove_coins_workspace_bytes.restype, L.vi_sumcheck_prove_coins_workspace_bytes.argtypes = SZ, [I64]
    L.vi_sumcheck_prove_coins.argtypes = [VP, VP, ctypes.c_int, I64, VP, VP, VP, ctypes.c_int, VP, VP, VP, SZ, VP]
    L.simt_error.restype = ctypes.c_char_p
    L.simt_system_stores.argtypes = [VP]
    NO_WORD = np.uint64((1 << 64) - 1)

    def check(form, v, buffers):
        terms, size = SUMS[form], 1 << v
        n = 1 + max(max(fs) for _, fs in terms)
        print("sumcheck", form, v, buffers, flush=True)
        tabs = [field(size, 100 * v + t) for t in range(n)]
        raw = [t.copy() for t in tabs]
        raw[0][0], raw[-1][-1] = NO_WORD, np.uint64(P)         # caller words at and above p
        tabs[0][0], tabs[-1][-1] = int(NO_WORD) % P, 0
        coins = field(v, v)
        src = [t.copy() for t in raw]
        work = src if buffers == "in place" else [np.full(max(size // 2, 1), 0xA5A5A5A5, dtype=np.uint64) for _ in range(n)]
        off = np.cumsum([0] + [len(fs) for _, fs in terms]).astype(np.int32)
        idx = np.array([f for _, fs in terms for f in fs], dtype=np.int32)
        coeffs = np.array([c for c, _ in terms], dtype=np.uint64)
        samples = np.full(8 * v, NO_WORD, dtype=np.uint64)
        stores = [L.simt_system_stores(samples.ctypes.data + 8 * x) for x in range(8 * v)]
        ws = scratch(L.vi_sumcheck_prove_coins_workspace_bytes(size))
        rc = L.vi_sumcheck_prove_coins((VP * n)(*[t.ctypes.data for t in src]), (VP * n)(*[t.ctypes.data for t in work]), n, size, ptr(off), ptr(idx),
                                       ptr(coeffs), len(terms), ptr(coins), ptr(samples), ptr(ws), len(ws), None)
        assert rc == 0, L.simt_error()
        _, want, _ = O.sumcheck_prove(tabs, terms, [int(c) for c in coins])
        deg = max(len(fs) for _, fs in terms)
        assert samples.reshape(v, 8)[:, :deg + 1].tolist() == want, (form, v, buffers)
        # the host may poll the samples: each is stored once, and past the caches
        for x in range(8 * v):
            at = samples.ctypes.data + 8 * x
            assert L.simt_system_stores(at) - stores[x] == (x % 8 <= deg), (form, v, x)
        if buffers == "apart":
            assert all(np.array_equal(a, b) for a, b in zip(src, raw)), "caller's table was modified"

    if "SIMT_CUS" in os.environ:
        # passes over more columns than the chip holds (four workgroups a CU): pieces from a counter, all tables' entries through LDS.  The
        # first pass alone, and the first two, where three workgroups of the second add up what the first has left, however few CUs there are
        cus = int(os.environ["SIMT_CUS"])
        for form in ("one", "two", "three", "four", "gate"):
            if cus == 1:
                check(form, 14, "apart")
                check(form, 16, "in place")
            # a second pass of 32 pieces for three workgroups' 48 wavefronts (36 for four tables), and of 64 and 128
            if cus < 3:
                check(form, 16 + cus, "apart")
            else:
                check(form, 18, "in place")
                if form in ("three", "gate"):
                    check(form, 19, "apart")
        print("sumcheck", flush=True)
        return
    # lengths below the lanes of a wavefront, one to eight entries a lane, one pass of three rounds and two, each with every remainder
    for form, terms in SUMS.items():
        common = sum(len(fs) <= 3 and 0 in fs for _, fs in terms) == len(terms) > 1
        for v in ((1, 6, 8, 9, 10, 11, 12) if common and len(terms) < 20 else (1, 6, 10) if len(terms) > 20 else (2, 5, 9, 11)):
            check(form, v, "apart")
        for v in (2, 10 if len(terms) < 20 else 7):
            check(form, v, "in place")
    print("sumcheck", flush=True)


def mle(so):
    """eq vectors and evaluations, one table and several, full groups of four tables and remainders, on both sides of sixteen entries to
    a thread; rows apart, results and scratch of exactly the stated sizes."""
    L = ctypes.CDLL(so)
    L.vi_mle_eval_workspace_bytes.restype, L.vi_mle_eval_workspace_bytes.argtypes = SZ, [I64]
    L.vi_mle_eval.argtypes = [VP, I64, I64, VP, ctypes.c_int, VP, VP, SZ, VP]
    L.vi_eq_vector.argtypes = [VP, ctypes.c_int, ctypes.c_int, VP, VP]
    for n, k in ((0, 1), (1, 2), (2, 5), (3, 4), (4, 3), (7, 9), (12, 5), (17, 5), (18, 1), (18, 5)):
        print("mle", n, k, flush=True)
        size, pitch = 1 << n, (1 << n) + (3 if n < 10 else 0)
        point = field(max(n, 1), n + 1)[:n]
        tabs = field(k * pitch, n + k)[:(k - 1) * pitch + size]
        for t in range(k):                                     # words at and above p in every table
            tabs[t * pitch + (7 * t) % size] = np.uint64((1 << 64) - 1 - t)
            tabs[t * pitch + (7 * t + 3) % size] = np.uint64(P)
        out, ws = np.empty(k, dtype=np.uint64), scratch(L.vi_mle_eval_workspace_bytes(k))
        assert L.vi_mle_eval(ptr(tabs), k, pitch, ptr(point), n, ptr(out), ptr(ws), len(ws), None) == 0
        rows = [tabs[t * pitch:t * pitch + size] for t in range(k)]
        assert out.tolist() == [O.mle_eval(r % np.uint64(P), [int(z) for z in point]) for r in rows], (n, k)
        if n < 13:
            eq = np.empty(size, dtype=np.uint64)
            assert L.vi_eq_vector(ptr(point), n, 0, ptr(eq), None) == 0 and np.array_equal(eq, O.eq_vector([int(z) for z in point]))


def blake3(so):
    """Pads of one, four and eight words to a thread, rows that share a workgroup and rows over several; digests and trees, four lanes to a
    compression and one."""
    L = ctypes.CDLL(so)
    L.vi_pad_rows.argtypes = [VP, I64, VP, I64, I64, I64, I64, VP, VP]
    L.vi_hash_columns_workspace_bytes.restype, L.vi_hash_columns_workspace_bytes.argtypes = SZ, [I64, I64]
    L.vi_hash_columns.argtypes = [VP, I64, I64, I64, VP, VP, SZ, VP]
    L.vi_merkle_tree_nodes.restype, L.vi_merkle_tree_nodes.argtypes = I64, [I64]
    L.vi_merkle_tree.argtypes = [VP, I64, VP, VP]
    seed = np.arange(32, dtype=np.uint8) * np.uint8(7)
    for rows, ell, width in ((1, 0, 1), (3, 5, 5), (7, 2, 19), (5, 100, 257), (300, 11, 17), (2, 8100, 9000),
                             (1030, 500, 512), (3, 180000, 180001), (8, 65530, 65537), (8200, 1020, 1024)):
        print("pad", rows, ell, width, flush=True)
        pitch = ell + 1
        msgs = field(rows * pitch, rows)[:(rows - 1) * pitch + ell]
        out = np.empty((rows, width), dtype=np.uint64)
        assert L.vi_pad_rows(ptr(seed), (1 << 32) - 2, ptr(msgs) if ell else None, rows, ell, pitch, width, ptr(out), None) == 0
        for r in range(rows):
            assert np.array_equal(out[r, :ell], msgs[r * pitch:r * pitch + ell]), (rows, ell, width, r)
        if width > ell:
            numbers = (np.arange(rows, dtype=np.uint64) + np.uint64((1 << 32) - 2)) % np.uint64(1 << 32)
            want = O.row_prg(seed.tobytes(), 0, rows, width - ell, numbers)
            assert np.array_equal(out[:, ell:], want), (rows, ell, width)
    for m, n in ((0, 3), (1, 5), (12, 256), (128, 70), (129, 70), (300, 65), (700, 33)):
        print("hash", m, n, flush=True)
        mat, digests = field((max(m, 1), n), m), np.empty((n, 32), dtype=np.uint8)
        ws = scratch(L.vi_hash_columns_workspace_bytes(m, n))
        assert L.vi_hash_columns(ptr(mat), m, n, n, ptr(digests), ptr(ws), len(ws), None) == 0
        assert np.array_equal(digests, O.hash_columns(mat[:m])), (m, n)
        nodes = np.empty((L.vi_merkle_tree_nodes(n), 32), dtype=np.uint8)
        assert L.vi_merkle_tree(ptr(digests), n, ptr(nodes), None) == 0
        assert np.array_equal(nodes, np.concatenate(O.merkle_levels(digests)[1:])), n


if __name__ == "__main__":
    globals()[sys.argv[1]](sys.argv[2])
    print("OK")
