"""GPU parity of the single-launch transforms and extensions of short rows: every row length and direction, ragged batches,
narrow and strided sources, coefficients beside, in place and alone, one to many cosets -- against the oracle, and against
the multi-pass kernels by running the same rows inside a batch too large for the single launch."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402
from tests.gpu_util import P, rand_field, to_dev, to_np  # noqa: E402


@pytest.fixture(scope="module")
def cp():
    from verinf_amd.prover import cuda_primitives
    return cuda_primitives


@pytest.mark.parametrize("logn", range(3, 12))
@pytest.mark.parametrize("m", [1, 3, 129])
def test_transforms(cp, logn, m):
    n = 1 << logn
    a = rand_field((m, n), 10 * logn + m)
    a[0, :3] = [P - 1, 0, P - 1]
    raw = a.copy()
    raw[-1, -2:] = [np.uint64((1 << 64) - 1), np.uint64(P + 1)]                        # words that are not canonical
    a[-1, -2:] = [np.uint64(((1 << 64) - 1) % P), 1]
    d = to_dev(raw)
    cp.ntt_forward_batched(d)
    fwd = to_np(d)
    assert np.array_equal(fwd, O.ntt_rows(a))
    big = to_dev(np.concatenate([a] * ((1 << 20) // a.size + 1)))                      # the multi-pass kernels
    cp.ntt_forward_batched(big)
    assert np.array_equal(to_np(big)[-m:], fwd)
    cp.ntt_inverse_batched(d)
    assert np.array_equal(to_np(d), a)
    inv = to_dev(a)
    cp.ntt_inverse_batched(inv)
    assert np.array_equal(to_np(inv), O.ntt_rows(a, inverse=True))


@pytest.mark.parametrize("logk", range(3, 13))
@pytest.mark.parametrize("log_rho", [0, 1, 2, 3, 5])
@pytest.mark.parametrize("m", [1, 5])
def test_extensions(cp, logk, log_rho, m):
    K, N = 1 << logk, 1 << (logk + log_rho)
    for w in (K, K - 3, 1):
        a = rand_field((m, w), 100 * logk + 10 * log_rho + w)
        wide = torch.empty((m, w + 5), dtype=torch.int64, device="cuda").view(torch.uint64)
        wide.view(torch.int64)[:, :w] = to_dev(a).view(torch.int64)
        src = wide[:, :w]                                                              # strided rows
        want = O.coset_lde_rows(a, K, N, 7)
        assert np.array_equal(to_np(cp.coset_lde(src, K, N)), want)
        coeffs, code = cp.coset_lde_with_coeffs(src, K, N)
        assert np.array_equal(to_np(code), want)
        only, none = cp.coset_lde_with_coeffs(src, K, N, need_codewords=False)
        assert none is None and torch.equal(only, coeffs)
        assert np.array_equal(to_np(cp.coset_extend(coeffs, K, N)), want)
        back = coeffs.clone()
        cp.ntt_forward_batched(back)
        assert np.array_equal(to_np(back)[:, :w], a)
    full = rand_field((m, K), 9 + logk)
    own = to_dev(full)
    coeffs, code = cp.coset_lde_with_coeffs(own, K, N, in_place=True)
    assert coeffs.data_ptr() == own.data_ptr()
    assert np.array_equal(to_np(code), O.coset_lde_rows(full, K, N, 7))
    back = coeffs.clone()
    cp.ntt_forward_batched(back)
    assert np.array_equal(to_np(back), full)


@pytest.mark.parametrize("logk,log_rho,m", [(5, 1, 70000), (6, 2, 9000), (10, 1, 1100), (8, 2, 1025), (12, 2, 300), (9, 3, 300)])
def test_larger_batches(cp, logk, log_rho, m):
    """All cosets in one workgroup, and the first batches beyond the single launch."""
    K, N = 1 << logk, 1 << (logk + log_rho)
    a = rand_field((m, K), logk)
    got = to_np(cp.coset_lde(to_dev(a), K, N))
    rows = sorted({0, 1, m // 3, m // 2, m - 2, m - 1})
    assert np.array_equal(got[rows], O.coset_lde_rows(np.ascontiguousarray(a[rows]), K, N, 7))
    coeffs, code = cp.coset_lde_with_coeffs(to_dev(a), K, N, in_place=True)
    assert np.array_equal(to_np(code), got)


@pytest.mark.parametrize("logk", range(5, 10))
@pytest.mark.parametrize("log_rho", range(5))
def test_passes_over_short_rows_in_parts_of_tiles(cp, logk, log_rho):
    """Batches beyond the single launch whose last tile of 4096 words holds one row or lacks one, from rows of any width and stride:
    against the single launch over slices of the batch, and the last rows against the oracle."""
    K, N = 1 << logk, 1 << (logk + log_rho)
    tile = max(1, 4096 // N)
    for m in ((5 << 20) // 2 // N // tile * tile + 1, (3 << 20) // N // tile * tile - 1):
        for w in (K, K - 3, K // 2 + 1):
            a = torch.randint(-(1 << 63), (1 << 63) - 1, (m, w + 5), dtype=torch.int64, device="cuda",
                              generator=torch.Generator(device="cuda").manual_seed(m + w)).view(torch.uint64)
            src = a[:, :w]
            coeffs, code = cp.coset_lde_with_coeffs(src, K, N)
            assert torch.equal(cp.coset_lde(src, K, N), code)
            assert torch.equal(cp.coset_extend(coeffs, K, N), code)
            step = (1 << 18) // N
            for i in range(0, m, step):
                some, want = cp.coset_lde_with_coeffs(src[i:i + step], K, N)
                assert torch.equal(coeffs[i:i + step], some) and torch.equal(code[i:i + step], want), (m, w, i)
            words = to_np(src[m - 2:].contiguous()) % np.uint64(P)
            assert np.array_equal(to_np(code[m - 2:]), O.coset_lde_rows(np.ascontiguousarray(words), K, N, 7))
        rows = torch.randint(-(1 << 63), (1 << 63) - 1, (m << log_rho, K), dtype=torch.int64, device="cuda").view(torch.uint64)[:-1]
        for transform in (cp.ntt_forward_batched, cp.ntt_inverse_batched):
            whole = rows.clone()
            transform(whole)
            step = (1 << 18) // K
            for i in range(0, rows.shape[0], step):
                some = rows[i:i + step].clone()
                transform(some)
                assert torch.equal(whole[i:i + step], some), (m, i)


@pytest.mark.parametrize("logk,log_rho", [(7, 0), (7, 1), (5, 2), (9, 1)])
def test_a_small_workspace_takes_the_same_extension(cp, logk, log_rho):
    """Rows enough for the passes, with a workspace for all of them (two launches), for a third, and for one row (one launch)."""
    from verinf_amd import _lib
    L = _lib.lib()
    K, N = 1 << logk, 1 << (logk + log_rho)
    m = (5 << 20) // N + 1
    src = to_dev(rand_field((m, K), logk + log_rho))
    one = L.vi_coset_lde_min_workspace_bytes(K, N)
    want = cp.coset_lde(src, K, N)
    for rows, launches in ((m, 2), (m // 3, None), (1, 1)):
        assert launches is None or L.vi_coset_lde_launches(m, K, N, one * rows) == launches
        ws = torch.empty(one * rows, dtype=torch.uint8, device="cuda")
        out = torch.zeros_like(want)
        rc = L.vi_coset_lde(src.data_ptr(), m, K, K, K, N, 7, out.data_ptr(), N, ws.data_ptr(), ws.numel(), None)
        torch.cuda.synchronize()
        assert rc == 0 and torch.equal(out, want), rows


@pytest.mark.parametrize("logn", range(12, 21))
def test_transforms_of_longer_rows(cp, logn):
    """Few rows (two or three launches of four points per thread) against the oracle and against a batch beyond them."""
    n = 1 << logn
    m = 1 if logn > 18 else 3
    a = rand_field((m, n), logn)
    raw = a.copy()
    raw[-1, -2:] = [np.uint64((1 << 64) - 1), np.uint64(P + 1)]                        # words that are not canonical
    a[-1, -2:] = [np.uint64(((1 << 64) - 1) % P), 1]
    d = to_dev(raw)
    cp.ntt_forward_batched(d)
    fwd = to_np(d)
    assert np.array_equal(fwd, O.ntt_rows(a))
    big = to_dev(np.concatenate([a] * ((1 << (22 if logn == 17 else 20)) // a.size + 1)))
    cp.ntt_forward_batched(big)
    assert np.array_equal(to_np(big)[-m:], fwd)
    cp.ntt_inverse_batched(d)
    assert np.array_equal(to_np(d), a)
    inv = to_dev(a)
    cp.ntt_inverse_batched(inv)
    assert np.array_equal(to_np(inv), O.ntt_rows(a, inverse=True))


# rows of 2^10 and 2^11 with up to four cosets have the single launch
@pytest.mark.parametrize("logk,log_rho", [(k, r) for r in (0, 1, 2, 3, 5) for k in range(10, 19) if (k > 11 or r >= 3) and k + r <= 21])
def test_extensions_of_longer_rows(cp, logk, log_rho):
    K, N = 1 << logk, 1 << (logk + log_rho)
    m = max(1, min(3, (1 << 20) // N)) if logk > 11 else (1 << 20) // N + 1
    for w in (K, K // 2 + 3, 1):
        a = rand_field((m, w), 100 * logk + 10 * log_rho + w)
        wide = torch.empty((m, w + 5), dtype=torch.int64, device="cuda").view(torch.uint64)
        wide.view(torch.int64)[:, :w] = to_dev(a).view(torch.int64)
        src = wide[:, :w]                                                              # strided rows
        code = cp.coset_lde(src, K, N)
        rows = sorted({0, m - 1})
        assert np.array_equal(to_np(code)[rows], O.coset_lde_rows(np.ascontiguousarray(a[rows]), K, N, 7))
        coeffs, again = cp.coset_lde_with_coeffs(src, K, N)
        assert torch.equal(again.view(torch.int64), code.view(torch.int64))
        only, none = cp.coset_lde_with_coeffs(src, K, N, need_codewords=False)
        assert none is None and torch.equal(only.view(torch.int64), coeffs.view(torch.int64))
        assert torch.equal(cp.coset_extend(coeffs, K, N).view(torch.int64), code.view(torch.int64))
        back = coeffs.clone()
        cp.ntt_forward_batched(back)
        assert np.array_equal(to_np(back)[:, :w], a)
        own = torch.zeros((m, K), dtype=torch.int64, device="cuda").view(torch.uint64)
        own.view(torch.int64)[:, :w] = to_dev(a).view(torch.int64)
        held, again = cp.coset_lde_with_coeffs(own, K, N, in_place=True)
        assert held.data_ptr() == own.data_ptr()
        assert torch.equal(held.view(torch.int64), coeffs.view(torch.int64)) and torch.equal(again.view(torch.int64), code.view(torch.int64))


# m rows take one set of launches, m + 1 another
@pytest.mark.parametrize("logk,log_rho,m", [(6, 2, 8192), (7, 2, 4096), (10, 3, 64), (10, 3, 3559), (11, 1, 4096), (12, 0, 128), (12, 0, 256), (12, 0, 485),
                                            (12, 1, 64), (12, 1, 128), (12, 2, 502), (13, 2, 151), (14, 2, 65), (16, 1, 8), (16, 2, 8), (18, 2, 11)])
def test_extensions_on_both_sides_of_the_switch(cp, logk, log_rho, m):
    K, N = 1 << logk, 1 << (logk + log_rho)
    a = to_dev(rand_field((m + 1, K), logk))
    few, more = cp.coset_lde(a[:m], K, N).view(torch.int64), cp.coset_lde(a, K, N).view(torch.int64)
    assert torch.equal(few, more[:m])
    for row in (0, m - 1):
        assert np.array_equal(to_np(more[row].view(torch.uint64)), O.coset_lde_rows(to_np(a[row:row + 1]), K, N, 7)[0])


_CAPTURE = """
import torch
from tests.gpu_util import rand_field, to_dev
from verinf_amd.prover import cuda_primitives as cp
for logn, first, then in ((5, 3, 1 << 16), (6, 1 << 15, 3), (8, 3, 1 << 13), (10, 1 << 11, 2), (11, 2, 1 << 10),
                          (12, 4, 1 << 9), (13, 1 << 8, 4)):
    n = 1 << logn
    cp.ntt_forward_batched(to_dev(rand_field((first, n), 1)))
    src = [to_dev(rand_field((then, n), 2 + i)) for i in range(3)]
    buf = src[0].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        cp.ntt_forward_batched(buf)
    for s in src:
        buf.copy_(s)
        g.replay()
        torch.cuda.synchronize()
        cp.ntt_forward_batched(s)
        assert torch.equal(buf.view(torch.int64), s.view(torch.int64)), logn
print("captured")
"""


_CAPTURE_EXTENSIONS = """
import torch
from tests.gpu_util import rand_field, to_dev
from verinf_amd.prover import cuda_primitives as cp
for logk, log_rate, first, then in ((9, 2, 3, 1 << 12), (10, 2, 3, 1 << 10), (11, 1, 1 << 11, 2), (12, 2, 2, 1 << 8), (12, 1, 1 << 10, 2), (14, 2, 64, 2)):
    k, n = 1 << logk, 1 << (logk + log_rate)
    cp.coset_lde(to_dev(rand_field((first, k), 1)), k, n, 7)
    src = [to_dev(rand_field((then, k), 2 + i)) for i in range(3)]
    buf = src[0].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = cp.coset_lde(buf, k, n, 7)
    for s in src:
        buf.copy_(s)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int64), cp.coset_lde(s, k, n, 7).view(torch.int64)), (logk, then)
print("captured")
"""


@pytest.mark.parametrize("calls", [_CAPTURE, _CAPTURE_EXTENSIONS], ids=["transforms", "extensions"])
def test_a_captured_call_finds_the_tables_of_another_batch_size(calls):
    """A call of one batch size prepares its row length for all of them: the other kernels capture with nothing left to
    upload.  In a process of its own, where no other test has prepared anything."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", calls], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("captured\n"), r.stderr[-2000:]
