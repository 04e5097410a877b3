"""Small results read back through pinned memory and small operands sent inside a launch, at the edges of their sizes,
with other work queued before them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from tests.gpu_util import P, rand_field, to_dev, to_np  # noqa: E402


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


class _Fails(list):
    """A mask polynomial that can be evaluated once, for its challenge, and then no more."""
    reads = 0

    def __reversed__(self):
        self.reads += 1
        if self.reads > 1:
            raise KeyboardInterrupt
        return super().__reversed__()


@pytest.mark.parametrize("left", ["proof", "evaluation", "between calls"])
def test_a_call_left_between_its_launches_and_its_results(left, monkeypatch):
    """The kernels of a call that an exception ended write their results all the same; the next call on the stream gets its own."""
    import random
    from oracle import oracle as O
    from verinf_amd import _lib
    from verinf_amd.layergkr import gpu
    from verinf_amd.prover import cuda_primitives as cp
    rng = random.Random(1)
    v = 10
    coins = [rng.randrange(P) for _ in range(v)]
    tabs = [rand_field(1 << v, t) for t in range(4)]
    dev = [to_dev(t) for t in tabs]
    slow = torch.ones((2048, 2048), dtype=torch.int64, device="cuda").view(torch.uint64)
    gpu.mle_eval_t(dev[0], coins)
    gpu.prove_terms_gpu([(1, dev[2:])], lambda i: coins[i], P)
    torch.cuda.synchronize()
    for _ in range(40):
        cp.gl_matmul(slow, slow)                               # a few milliseconds in front of the kernels of the call
    with monkeypatch.context() as m, pytest.raises(KeyboardInterrupt):
        if left == "between calls":                            # the second interrupt: nothing is waited for
            m.setattr(_lib._Words, "__exit__", lambda self, *error: None)
        if left == "evaluation":
            def interrupted(*args):
                raise KeyboardInterrupt
            m.setattr(_lib.lib(), "vi_wait_words", interrupted)
            gpu.mle_eval_t(dev[0], coins)
        else:
            gpu.prove_terms_gpu([(1, dev[:2])], lambda i: coins[i], P, mask=lambda deg, mu: _Fails([1, 2, 3]))
    if left == "evaluation":
        assert gpu.mle_eval_t(dev[1], coins) == O.mle_eval(tabs[1], coins)
    claim, polys, _, _ = gpu.prove_terms_gpu([(1, dev[2:])], lambda i: coins[i], P)
    want_claim, want_samples, _ = O.sumcheck_prove(tabs[2:], [(1, [0, 1])], coins)
    assert claim == want_claim and [[y for _, y in s] for s in polys] == want_samples


def test_a_call_within_another_ones_wait_has_words_of_its_own():
    from verinf_amd import _lib
    sp = _lib.stream_ptr()
    with _lib.polled_words(8, sp) as outer:
        outer.view[:8] = 5
        with _lib.polled_words(8, sp) as inner:
            assert inner is not outer and inner.view[0] == _lib.NO_WORD and outer.view[0] == 5
    assert not outer.polled and not inner.polled
