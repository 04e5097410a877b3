"""GPU parity: gl_matmul at the edges of its tiles, blocks and slices, on the VALU (few rows) and on the matrix cores
(many rows), against Python big-int sums (bit-exact); larger results by sampled rows and columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from tests.gpu_util import P, rand_field, to_dev, to_np  # noqa: E402


@pytest.mark.parametrize("m,k,n,fill", [
    # VALU: row remainders of a lane's tile, slices over wavefronts and over workgroups, one row streamed
    (9, 33, 65, None), (17, 500, 129, None), (13, 16, 64, None), (1, 20, 40000, None), (8, 3000, 40, "top"), (1, 2048, 33000, "any"),
    # matrix cores: 64 x 64, 128 x 128 and 128 x 256 tiles with remainders, inner dimensions around a step and a slice,
    # the largest sums, words at and above p, columns in several blocks
    (64, 1000, 3000, None), (65, 1023, 2999, "any"), (129, 700, 4097, None), (700, 257, 2100, "any"), (1025, 65, 4300, None),
    (130, 8192, 130, "top"), (131, 8193, 129, "half"), (200, 16400, 70, "any"), (100, 40, 250001, None)])
def test_matmul_edges(m, k, n, fill):
    from verinf_amd.prover import cuda_primitives as cp
    A, B = rand_field((m, k), 1 + m), rand_field((k, n), 2 + n)
    if fill == "top":
        A[:], B[:] = P - 1, P - 1
    elif fill == "half":                                        # the word of largest size as a signed number, both signs
        A[:], B[:] = 0x8080808080808080, 0x7F7F7F7F7F7F7F7F
        B[::2] += 1
    elif fill == "any":                                         # words that are not canonical
        A[:, ::3] = np.uint64((1 << 64) - 1) - A[:, ::3] % np.uint64(1 << 20)
        B[::2] = np.uint64((1 << 64) - 1) - B[::2] % np.uint64(1 << 33)
    print(m, k, n, fill, flush=True)
    got = to_np(cp.gl_matmul(to_dev(A), to_dev(B)))
    assert got.shape == (m, n)
    budget = 4_000_000 // k                                     # entries checked
    rows = sorted({0, m // 2, m - 1, min(m - 1, 63)})
    cols = np.unique(np.linspace(0, n - 1, max(2, budget // len(rows))).astype(int)) if n * len(rows) > budget else np.arange(n)
    want = (A[rows].astype(object).dot(B[:, cols].astype(object)) % P).astype(np.uint64)
    assert np.array_equal(got[np.ix_(rows, cols)], want)


@pytest.mark.parametrize("skip", [0, 8])
def test_scratch_of_any_alignment(skip):
    from verinf_amd import _lib
    L = _lib.lib()
    m, k, n = 130, 70, 150
    A, B = rand_field((m, k), 1), rand_field((k, n), 2)
    dA, dB, C = to_dev(A), to_dev(B), torch.empty((m, n), dtype=torch.uint64, device="cuda")
    while (need := L.vi_gl_matmul_workspace_bytes(m, k, n)) < 18 * 128 * 128:           # a size of the matrix cores
        m *= 2
        A = rand_field((m, k), 1)
        dA, C = to_dev(A), torch.empty((m, n), dtype=torch.uint64, device="cuda")
    ws = torch.full((need + skip + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    _lib.check(L.vi_gl_matmul(dA.data_ptr(), dB.data_ptr(), C.data_ptr(), m, k, n, ws.data_ptr() + skip, need, _lib.stream_ptr()))
    assert np.array_equal(to_np(C), (A.astype(object).dot(B.astype(object)) % P).astype(np.uint64))
    assert bool((ws[:skip] == 0x5A).all()) and bool((ws[need + skip:] == 0x5A).all())


# 16-bit signed numbers: tiles of 64 x 128 and 128 x 128 with remainders, steps and slices of the inner dimension with remainders,
# the largest sums, one word of A or B a step beyond the range (then the residues do the product)
@pytest.mark.parametrize("m,k,n", [(40, 64, 3000), (64, 1000, 3001), (65, 1023, 2999), (129, 700, 4097), (1025, 65, 4300), (300, 9000, 500),
                                   (128, 8192, 128), (100, 32768, 70), (100, 32769, 70)])
@pytest.mark.parametrize("fill", ["any", "top", "low", "over a", "over b"])
def test_matmul_of_small_numbers(m, k, n, fill):
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(m)
    lo, hi = {"top": ((1 << 15) - 1, 1 << 15), "low": (-(1 << 15), 1 - (1 << 15))}.get(fill, (-(1 << 15), 1 << 15))
    A, B = rng.integers(lo, hi, (m, k)), rng.integers(lo, hi, (k, n))
    if fill == "over a":
        A[-1, -1] = 1 << 15
    if fill == "over b":
        B[-1, -1] = -(1 << 15) - 1
    dA, dB = (to_dev(np.where(x < 0, x.astype(np.uint64) + np.uint64(P), x.astype(np.uint64))) for x in (A, B))
    print(m, k, n, fill, flush=True)
    got = to_np(cp.gl_matmul(dA, dB))
    rows = sorted({0, m // 2, m - 1, min(m - 1, 63)})
    want = A[rows] @ B                                          # below 2^45
    assert np.array_equal(got[rows], np.where(want < 0, want.astype(np.uint64) + np.uint64(P), want.astype(np.uint64)))
    ones = to_np(cp.gl_matmul(dA, to_dev(np.ones((k, 300), dtype=np.uint64))))[:, 299]        # every row
    want = A.sum(axis=1)
    assert np.array_equal(ones, np.where(want < 0, want.astype(np.uint64) + np.uint64(P), want.astype(np.uint64)))


@pytest.mark.parametrize("m", list(range(1, 11)) + [13, 17, 21, 24])
@pytest.mark.parametrize("k,n", [(9, 65), (1300, 129), (3000, 64), (700, 4097)])
def test_few_rows(m, k, n):
    """Every number of rows to a lane, one and several blocks of rows, one to 64 slices of the inner dimension."""
    from verinf_amd.prover import cuda_primitives as cp
    A, B = rand_field((m, k), m), rand_field((k, n), n)
    A[0, :], B[:, -1] = P - 1, P - 1
    got = to_np(cp.gl_matmul(to_dev(A), to_dev(B)))
    cols = np.unique(np.linspace(0, n - 1, min(n, 3_000_000 // (m * k) + 2)).astype(int))
    assert np.array_equal(got[:, cols], (A.astype(object).dot(B[:, cols].astype(object)) % P).astype(np.uint64))


# residues by three workgroups a slab and by one (340 slabs and more), of one block and of the first of several; words that the first
# launch's sample sees and does not see
@pytest.mark.parametrize("m,k,n", [(256, 1088, 1024), (256, 1089, 1025), (64, 760, 1070), (300, 9000, 500), (100, 16400, 300), (70, 40, 120001)])
@pytest.mark.parametrize("kind", ["field", "mixed", "few"])
def test_matmul_of_arbitrary_words(m, k, n, kind):
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(m + k)
    A = rand_field((m, k), 1) if kind == "field" else rng.integers(0, 1 << 15, (m, k)).astype(np.uint64)
    B = rng.integers(0, 1 << 15, (k, n)).astype(np.uint64) if kind == "few" else rand_field((k, n), 2)
    if kind == "few":                                           # a word of A, and a column of B
        A[m // 2, k // 3] = P - 12345678901
        B[:, n - 1] = rand_field((k,), 3)
    print(m, k, n, kind, flush=True)
    got = to_np(cp.gl_matmul(to_dev(A), to_dev(B)))
    rows = sorted({0, m // 2, m - 1})
    cols = np.unique(np.concatenate([[n - 1], np.linspace(0, n - 1, 1 + 1_000_000 // k).astype(int)]))
    want = (A[rows].astype(object).dot(B[:, cols].astype(object)) % P).astype(np.uint64)
    assert np.array_equal(got[np.ix_(rows, cols)], want)
    one = to_np(cp.gl_matmul(to_dev(A), to_dev(np.ones((k, 300), dtype=np.uint64))))[:, 299]              # every row
    assert np.array_equal(one, (A.astype(object).sum(axis=1) % P).astype(np.uint64))
