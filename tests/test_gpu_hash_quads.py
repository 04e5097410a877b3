"""GPU parity of the four-lane BLAKE3 forms: column digests around the size at which one lane per column takes over, block and
chunk remainders, trees of every small leaf count, and padded rows -- against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402
from tests.gpu_util import rand_field, to_dev, to_np  # noqa: E402


@pytest.mark.parametrize("m", [0, 1, 7, 8, 9, 127, 128, 129, 300])
@pytest.mark.parametrize("n", [1, 15, 64, 65, 4096])
def test_column_digests(m, n):
    from verinf_amd.prover import cuda_primitives as cp
    a = rand_field((m, n), 3 * m + n) if m else np.zeros((0, n), dtype=np.uint64)
    assert np.array_equal(to_np(cp.hash_columns_streamed(to_dev(a))), O.hash_columns(a))


@pytest.mark.parametrize("m,n", [(16, 16384), (16, 16385), (256, 8192), (257, 8192)])
def test_column_digests_around_the_switch(m, n):
    from verinf_amd.prover import cuda_primitives as cp
    a = rand_field((m, n), m)
    got = to_np(cp.hash_columns_streamed(to_dev(a)))
    cols = [0, 1, n // 2, n - 2, n - 1]
    assert np.array_equal(got[cols], O.hash_columns(np.ascontiguousarray(a[:, cols])))


@pytest.mark.parametrize("m,n", [(9, 131072), (9, 131073), (129, 65536), (129, 65537), (129, 131073), (300, 43520), (300, 43777)])
def test_column_digests_around_two_wavefronts_per_simd(m, n):
    """Chunks and merges on both sides of the launch size from which sums and exclusive ors have the long encoding."""
    from verinf_amd.prover import cuda_primitives as cp
    a = rand_field((m, n), m)
    got = to_np(cp.hash_columns_streamed(to_dev(a)))
    cols = [0, 1, n // 2, n - 2, n - 1]
    assert np.array_equal(got[cols], O.hash_columns(np.ascontiguousarray(a[:, cols])))
    rows = 9 if n > 100000 else 1                          # pads: a word a thread, both sides as well
    seed = torch.arange(32, dtype=torch.uint8, device="cuda")
    pads = to_np(cp.row_prg(seed, 5, rows, n // 8))
    assert np.array_equal(pads[-1], O.row_prg(bytes(range(32)), 4 + rows, 1, n // 8)[0])


def test_trees_of_every_small_size():
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(1)
    for k in list(range(1, 70)) + [127, 129, 255, 256, 257, 511, 512, 513, 700, 1025, 5000]:
        leaves = rng.integers(0, 256, (k, 32), dtype=np.uint8)
        root, levels = cp.merkle_build_blake3(torch.from_numpy(leaves).cuda())
        want = O.merkle_levels(leaves)
        assert len(levels) == len(want)
        for got, ref in zip(levels, want):
            assert np.array_equal(to_np(got), ref), k
        assert to_np(root).tobytes() == want[-1][0].tobytes()


@pytest.mark.parametrize("m,ell,width,stride", [(1, 1, 4, 1), (3, 0, 8, 5), (5, 48, 64, 48), (33, 100, 128, 131), (7, 64, 64, 64)])
def test_padded_rows(m, ell, width, stride):
    from verinf_amd.prover import cuda_primitives as cp
    seed = bytes(range(40, 72))
    wide = rand_field((m, stride), 5)
    padded = torch.empty((m, width), dtype=torch.uint64, device="cuda")
    cp.pad_rows(torch.tensor(list(seed), dtype=torch.uint8, device="cuda"), 4_000_000_000, to_dev(wide)[:, :ell], padded)
    want = np.concatenate([wide[:, :ell], O.row_prg(seed, 4_000_000_000, m, width - ell)], axis=1) if width > ell else wide[:, :ell]
    assert np.array_equal(to_np(padded), want)


@pytest.mark.parametrize("m,ell,width", [(1023, 300, 512), (1025, 511, 512), (8200, 40, 64), (30000, 7, 19), (200000, 1, 3), (37, 9001, 16383), (150, 40000, 65536)])
def test_padded_rows_in_larger_batches(m, ell, width):
    """One, four and eight words a thread; rows whose words do not divide over the lanes."""
    from verinf_amd.prover import cuda_primitives as cp
    seed = bytes(range(7, 39))
    messages = torch.randint(0, 1 << 62, (m, ell), dtype=torch.int64, device="cuda").view(torch.uint64)
    padded = torch.empty((m, width), dtype=torch.uint64, device="cuda")
    cp.pad_rows(torch.tensor(list(seed), dtype=torch.uint8, device="cuda"), 11, messages, padded)
    assert torch.equal(padded[:, :ell], messages)
    for r in {0, 1, m // 2, m - 1}:
        assert np.array_equal(to_np(padded[r, ell:]), O.row_prg(seed, 11 + r, 1, width - ell)[0]), r


def test_a_message_of_one_chunk_without_workspace_is_refused():
    from verinf_amd import _lib
    mat = to_dev(rand_field((8, 64), 1))
    out = torch.zeros(64 * 32, dtype=torch.uint8, device="cuda")
    ws = torch.empty(64, dtype=torch.uint8, device="cuda")
    for ptr, size in ((None, 0), (ws.data_ptr(), 64)):
        assert _lib.lib().vi_hash_columns(mat.data_ptr(), 8, 64, 64, out.data_ptr(), ptr, size, _lib.stream_ptr()) != 0
    assert not out.any()
