"""The Python wrappers on several streams and host threads at once: scratch buffers are kept per (purpose,
device, stream) and the sumcheck's pinned sample words per (thread, stream), so concurrent callers must not
disturb each other.  Each thread's results are compared bit for bit with the oracle."""
import random
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402
from tests.gpu_util import P, rand_field, to_dev, to_np  # noqa: E402


def test_wrappers_from_two_threads_on_their_own_streams():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from verinf_amd import _lib
    from verinf_amd.layergkr import gpu
    from verinf_amd.prover import cuda_primitives as cp

    jobs = [(1 << 12, 1 << 14, 37, 51), (1 << 13, 1 << 15, 19, 52)]
    results, errors = {}, []

    def work(i):
        try:
            K, N, m, seed = jobs[i]
            stream = torch.cuda.Stream()                        # default priority
            msgs = rand_field((m, K), seed)
            tabs = [rand_field(1 << 14, seed + 10 + j) for j in range(3)]
            coins = [random.Random(seed).randrange(P) for _ in range(14)]
            with torch.cuda.stream(stream):
                d_msgs = to_dev(msgs)
                d_tabs = [to_dev(t) for t in tabs]
                outs = []
                for _ in range(6):                              # keep both streams busy at the same time
                    code = cp.coset_lde(d_msgs, K, N, 7)
                    rows = d_msgs.clone()
                    cp.ntt_forward_batched(rows)
                    claim, polys, _, _ = gpu.prove_terms_gpu([(1, d_tabs)], lambda r: coins[r], P)
                    outs.append((code, rows, claim, polys))
                stream.synchronize()
            results[i] = (msgs, tabs, coins, [(to_np(c), to_np(r), cl, po) for c, r, cl, po in outs])
        except Exception as exc:                                # surfaced by the main thread
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i, (K, N, m, seed) in enumerate(jobs):
        msgs, tabs, coins, outs = results[i]
        want_code = O.coset_lde_rows(msgs, K, N, 7)
        want_rows = O.ntt_rows(msgs)
        want_claim, want_samples, _ = O.sumcheck_prove(tabs, [(1, [0, 1, 2])], coins)
        for code, rows, claim, polys in outs:
            assert np.array_equal(code, want_code)
            assert np.array_equal(rows, want_rows)
            assert claim == want_claim and [[y for _, y in s] for s in polys] == want_samples
    # one scratch buffer per stream that was used, none shared
    keys = [k for k in _lib._ws_cache if k[0] == "lde"]
    assert len({k[2] for k in keys}) >= 2
    _lib.release_workspaces()
    assert not _lib._ws_cache


@pytest.mark.parametrize("n_table", [100, 5000, 40000])
def test_look_ups_on_two_streams_add_into_one_table(n_table):
    """lookup_multiplicities_into adds: calls on streams without an order between them lose no counts."""
    from verinf_amd.prover import cuda_primitives as cp
    rng = np.random.default_rng(n_table)
    table = to_dev(np.arange(n_table, dtype=np.uint64))
    for n_x in (5000, 300000):                                   # one workgroup per slice, and rows added up by a second launch
        xs = [rng.integers(0, n_table, n_x).astype(np.uint64) for _ in range(2)]
        dev = [to_dev(x) for x in xs]
        mult = torch.zeros(n_table, dtype=torch.int64, device="cuda").view(torch.uint64)
        torch.cuda.synchronize()
        streams, rounds = [torch.cuda.Stream(), torch.cuda.Stream()], 40
        for _ in range(rounds):
            for s, x in zip(streams, dev):
                with torch.cuda.stream(s):
                    cp.lookup_multiplicities_into(x, table, mult)
        torch.cuda.synchronize()
        want = sum(np.bincount(x.astype(np.int64), minlength=n_table) for x in xs) * rounds
        assert np.array_equal(to_np(mult), want.astype(np.uint64))


def _two_threads(job, count=2):
    """job(i) on `count` threads that switch as often as the interpreter can, all on the default stream."""
    import sys
    errors, gate = [], threading.Barrier(count)

    def work(i):
        try:
            gate.wait()
            job(i)
        except BaseException as exc:                             # surfaced by the main thread
            errors.append(exc)

    before = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(count)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(before)
    assert not errors, errors


def test_threads_that_share_a_stream_do_not_share_a_call():
    """Calls of several launches through scratch: the launches of two threads' calls on one stream do not mix, also while the
    scratch grows."""
    from verinf_amd import _lib
    from verinf_amd.layergkr import gpu
    from verinf_amd.prover import cuda_primitives as cp
    _lib.release_workspaces()

    def inputs(i):
        tabs = [rand_field(1 << (10 + i), 70 + 10 * i + j) for j in range(3)]
        table = np.arange(5000 + 3000 * i, dtype=np.uint64)
        return {"lde": rand_field((5 + 40 * i, 1 << 13), 61 + i), "ntt": rand_field((3 + 9 * i, 1 << 14), 63 + i),
                "a": rand_field((70 + 60 * i, 300), 65 + i), "b": rand_field((300, 500 + 300 * i), 67 + i),
                "x": np.random.default_rng(i).integers(0, len(table), 200000 + 100000 * i).astype(np.uint64), "table": table,
                "hash": rand_field((300 + 100 * i, 64), 69 + i), "sum": rand_field(70000 + i, 80 + i), "tabs": tabs,
                "mat": np.stack(tabs), "coins": [random.Random(i + 7 * j).randrange(P) for j in range(10 + i)]}

    data = [inputs(i) for i in range(2)]
    dev = [{k: [to_dev(t) for t in v] if k == "tabs" else (v if k == "coins" else to_dev(v)) for k, v in d.items()} for d in data]

    def calls(d):
        rows = d["ntt"].clone()
        cp.ntt_forward_batched(rows)
        claim, polys, _, _ = gpu.prove_terms_gpu([(1, d["tabs"])], lambda r: d["coins"][r], P)
        return [cp.coset_lde(d["lde"], 1 << 13, 1 << 15), rows, cp.gl_matmul(d["a"], d["b"]), cp.lookup_multiplicities(d["x"], d["table"]),
                cp.hash_columns_streamed(d["hash"]), gpu.gl_sum(d["sum"])], claim, polys, gpu.mle_eval_t(d["mat"], d["coins"])

    out = {0: [], 1: []}
    _two_threads(lambda i: out[i].extend(calls(dev[i]) for _ in range(25)))
    torch.cuda.synchronize()
    for i in range(2):
        d = data[i]
        want = [O.coset_lde_rows(d["lde"], 1 << 13, 1 << 15, 7), O.ntt_rows(d["ntt"]), None,
                np.bincount(d["x"].astype(np.int64), minlength=len(d["table"])).astype(np.uint64), O.hash_columns(d["hash"]), None]
        want[2] = (d["a"].astype(object).dot(d["b"].astype(object)) % P).astype(np.uint64)
        want[5] = np.array([sum(int(v) for v in d["sum"]) % P], dtype=np.uint64)
        want_claim, want_samples, _ = O.sumcheck_prove(d["tabs"], [(1, [0, 1, 2])], d["coins"])
        want_ends = [O.mle_eval(t, d["coins"]) for t in d["tabs"]]
        for tensors, claim, polys, ends in out[i]:
            for k, (got, w) in enumerate(zip(tensors, want)):
                assert np.array_equal(to_np(got), w), k
            assert claim == want_claim and [[y for _, y in s] for s in polys] == want_samples and ends == want_ends


def test_interactive_proofs_on_one_stream_in_step():
    """Two provers whose coins wait for each other in every round: neither holds what the other one needs."""
    from verinf_amd.layergkr import gpu
    n_rounds, gate = 9, threading.Barrier(2, timeout=60)
    tabs = [[rand_field(1 << n_rounds, 90 + 10 * i + j) for j in range(3)] for i in range(2)]
    dev = [[to_dev(t) for t in ts] for ts in tabs]
    coins = [random.Random(5).randrange(P) for _ in range(n_rounds)]
    out = [None, None]

    def job(i):
        def coin(rnd, samples):
            gate.wait()
            return coins[rnd]
        out[i] = gpu.prove_terms_gpu_interactive([(1, dev[i]), (3, dev[i][:2])], coin, P)

    _two_threads(job)
    for i in range(2):
        want_claim, want_samples, _ = O.sumcheck_prove(tabs[i], [(1, [0, 1, 2]), (3, [0, 1])], coins)
        assert out[i][0] == want_claim and [[y for _, y in s] for s in out[i][1]] == want_samples


def test_a_graph_keeps_its_scratch_when_later_calls_outgrow_it():
    """Captured calls that use scratch, replayed after larger calls on the same stream took bigger buffers and other tensors
    took the memory that the smaller ones had."""
    from verinf_amd import _lib
    from verinf_amd.layergkr import gpu
    from verinf_amd.prover import cuda_primitives as cp
    _lib.release_workspaces()
    side = torch.cuda.Stream()

    def calls(lde, rows, a, b, x, table, mat, vec):
        rows = rows.clone()
        cp.ntt_forward_batched(rows)
        return [cp.coset_lde(lde, 1 << 13, 1 << 15), rows, cp.gl_matmul(a, b), cp.lookup_multiplicities(x, table), cp.hash_columns_streamed(mat),
                gpu.gl_sum(vec)]

    def inputs(scale, seed):
        shapes = ((2 * scale, 1 << 13), (2 * scale, 1 << 14), (80 * scale, 200), (200, 400 * scale))
        table = np.arange(6000 * scale, dtype=np.uint64)
        x = np.random.default_rng(seed).integers(0, len(table), 150000).astype(np.uint64)
        return [*(to_dev(rand_field(s, seed + i)) for i, s in enumerate(shapes)), to_dev(x), to_dev(table), to_dev(rand_field((300 * scale, 64), seed + 9)),
                to_dev(rand_field(5000 * scale, seed + 10))]

    args, side_args = inputs(1, 1), inputs(8, 50)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls(*args)                                             # tables are uploaded here, and small scratch is cached
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        outs = calls(*args)
    with torch.cuda.stream(side):
        calls(*side_args)
    side.synchronize()
    others = [torch.full((1 << s,), 0x5A, dtype=torch.uint8, device="cuda") for s in range(10, 24) for _ in range(2)]
    for seed in (1, 20, 40):
        for old, new in zip(args, inputs(1, seed)):
            old.copy_(new)
        want = calls(*args)
        g.replay()
        torch.cuda.synchronize()
        for k, (got, w) in enumerate(zip(outs, want)):
            assert np.array_equal(to_np(got), to_np(w)), (seed, k)
        assert all(bool((o == 0x5A).all()) for o in others)
