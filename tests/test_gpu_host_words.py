"""Small results read back through pinned memory and small operands sent inside a launch, at the edges of their sizes,
with other work queued before them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from tests.gpu_util import P, to_np  # noqa: E402


@pytest.mark.parametrize("nbytes", [4, 8, 12, 32, 1020, 4096, 5000 * 4, 1 << 20])
def test_read_back(nbytes):
    from verinf_amd import _lib
    src = torch.randint(0, 256, (nbytes + 8,), dtype=torch.uint8, device="cuda")
    for _ in range(3):
        src += 1                                              # the bytes are those after the queued work
        assert _lib.read_back(src, nbytes) == to_np(src)[:nbytes].tobytes()
    with pytest.raises(_lib.VerinfHipError):
        _lib.read_back(src, nbytes + 1)


@pytest.mark.parametrize("n", [0, 1, 12, 63, 64, 448, 449, 5000])
def test_upload_of_python_integers(n):
    from verinf_amd import _lib
    rng = np.random.default_rng(n)
    for lo, hi in ((0, 1 << 62), (0, P), (P - 3, 1 << 64), (-5, 1 << 70)):       # canonical, not canonical, beyond a word
        values = [int(rng.integers(0, 1 << 62)) * (hi - lo) // (1 << 62) + lo for _ in range(n)]
        t = _lib.upload_words(_lib.field_words(values))
        assert tuple(t.shape) == (1, n) and t.dtype == torch.uint64
        assert to_np(t)[0].tolist() == [v % P for v in values]
    assert to_np(_lib.upload_words(_lib.field_words(np.arange(3, dtype=np.uint64))))[0].tolist() == [0, 1, 2]


def test_waiting_for_words():
    """Results that are there already, arguments that make no sense, and a stream that has nothing more to write."""
    from verinf_amd import _lib
    L = _lib.lib()
    host, view = _lib.pinned_words(64, _lib.stream_ptr())
    view[:24] = _lib.NO_WORD
    view.reshape(-1)[:24].reshape(3, 8)[:, :5] = 7
    assert L.vi_wait_words(host.data_ptr(), 3, 8, 5, _lib.stream_ptr()) == 0
    assert L.vi_wait_words(host.data_ptr(), 0, 8, 5, _lib.stream_ptr()) == 0
    torch.cuda.synchronize()
    assert L.vi_wait_words(host.data_ptr(), 3, 8, 6, _lib.stream_ptr()) == -2 and b"drained" in L.vi_last_error()
    assert L.vi_wait_words(host.data_ptr(), 3, 4, 5, None) == -1 and L.vi_wait_words(host.data_ptr() + 4, 1, 1, 1, None) == -1
    assert L.vi_wait_words(None, 1, 1, 1, None) == -1
