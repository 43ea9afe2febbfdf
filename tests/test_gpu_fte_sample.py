"""The shared threshold sample when its pieces are late (forced from the host:
one try, then every workgroup scores what is missing itself), bit for bit
against the CPU oracle: synchronous queries, queries queued on both lanes,
and two engines queueing at once."""
import threading

import numpy as np
import pytest

import oracle
import topk_amd

pytestmark = pytest.mark.gpu

# (n, d, m, k): fewer workgroups than pieces' takers, ragged pieces, deep ranks, runtime-width scores
CASES = [((1 << 19) + 1, 3, 2, 16), (1_300_003, 8, 8, 64), (2_100_001, 20, 20, 1000), (4_194_301, 5, 1, 1)]


def _store(n, d):
    return topk_amd.generate(n, d, topk_amd.INDEPENDENT, 3)


@pytest.mark.parametrize("polls", [1, 2, 0])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_late_sample(gpu, case, polls):
    n, d, m, k = case
    x = _store(n, d)
    rng = np.random.default_rng(n)
    w, attr = rng.uniform(-0.2, 1.0, d).astype(np.float32), rng.permutation(d)[:m]
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, attr)
    with topk_amd.Engine(x) as eng:
        eng.set_tuning("sample_polls", polls)
        for grid in (0, 5):
            eng.set_tuning("stream_grid", grid)
            for _ in range(2):
                ids, sc, thr = eng.fte(k, w, attr)
                assert np.array_equal(ids, rid) and np.array_equal(sc.view(np.uint32), rsc.view(np.uint32))
                assert thr == rthr


def _queue(eng, queries, k):
    import torch
    ids = [torch.empty(k, dtype=torch.int64, device="cuda") for _ in queries]
    sc = [torch.empty(k, dtype=torch.float32, device="cuda") for _ in queries]
    for i, (w, attr) in enumerate(queries):
        eng.fte_async(k, w, attr, ids[i].data_ptr(), sc[i].data_ptr())
    eng.sync()
    return [t.cpu().numpy().view(np.uint64) for t in ids], [t.cpu().numpy() for t in sc]


def _ordered(n, kind):
    """One column whose score order follows the ids."""
    i = np.arange(n, dtype=np.float32) / np.float32(n)
    if kind == "best-first":
        return i[::-1].copy().reshape(1, n)
    if kind == "best-last":
        return i.reshape(1, n)
    x = topk_amd.generate(n, 1, topk_amd.INDEPENDENT, 2) * np.float32(0.5)
    at = n // 128 // 16 * 16 * 40  # the first object of a sampled chunk
    x[0, at:at + 2000] += np.linspace(1, 0.5, 2000, dtype=np.float32)
    return x


@pytest.mark.parametrize("kind", ["best-first", "best-last", "clustered"])
@pytest.mark.parametrize("n,ks", [(524_289, (14, 18, 300)), (700_001, (14, 24, 1024)), (1 << 20, (14, 16, 36, 64, 1000)),
                                  (1_048_577, (16, 1000)), (2_097_153, (256, 1000))])
def test_queued_queries_on_stores_in_score_order(gpu, kind, n, ks):
    # nothing re-runs a queued query: its threshold holds for ordered stores too
    x = _ordered(n, kind)
    w = np.ones(1, np.float32)
    with topk_amd.Engine(x) as eng:
        for k in ks:
            ids, sc = _queue(eng, [(w, [0])] * 2, k)
            rid, rsc, _ = oracle.fte_topk(x, n, k, w, [0])
            for j in range(2):
                assert np.array_equal(ids[j], rid) and np.array_equal(sc[j], rsc), k


@pytest.mark.parametrize("polls", [1, 0])
def test_late_sample_with_queries_queued_on_both_lanes(gpu, polls):
    n, d, k = 1_300_003, 8, 32
    x = _store(n, d)
    rng = np.random.default_rng(1)
    queries = [(rng.uniform(0.1, 1.0, d).astype(np.float32), rng.permutation(d)[:3 + i % 6]) for i in range(16)]
    want = [oracle.fte_topk(x, n, k, w, a) for w, a in queries]
    with topk_amd.Engine(x) as a, topk_amd.Engine(x) as b:
        got = {}
        for e in (a, b):
            e.set_tuning("sample_polls", polls)
        threads = [threading.Thread(target=lambda e=e, i=i: got.setdefault(i, _queue(e, queries, k)))
                   for i, e in enumerate((a, b))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for i in range(2):
        for j, (rid, rsc, _) in enumerate(want):
            assert np.array_equal(got[i][0][j], rid) and np.array_equal(got[i][1][j], rsc), (i, j)


@pytest.mark.parametrize("kind", ["best-first", "best-last", "one-value", "two-values", "few-below"])
@pytest.mark.parametrize("n,k", [(4097, 1024), (6000, 1000), (8191, 1024), (65_521, 10), (1 << 19, 64), (1 << 20, 1),
                                 (1 << 20, 10), (1 << 20, 256), (1 << 20, 1000)])
def test_select_of_many_candidates(gpu, kind, n, k):
    # candidates past the select's LDS: spread by score, all tied, and an interval too full for it
    if kind in ("best-first", "best-last"):
        x = _ordered(n, kind)
    else:
        x = np.full((1, n), 0.75, np.float32)
        if kind == "two-values":
            x[0, ::2] = 0.25
        if kind == "few-below":
            x[0, n // 2:n // 2 + 90] = 0.25
    w = np.ones(1, np.float32)
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, [0])
    with topk_amd.Engine(x) as eng:
        for _ in range(2):
            ids, sc, thr = eng.fte(k, w, [0])
            assert np.array_equal(ids, rid) and np.array_equal(sc, rsc) and thr == rthr
        if kind.startswith("best"):
            assert eng.stats()["fallback"] == 0  # one run


@pytest.mark.parametrize("n", [1, 4095, 100_003, 1 << 19])
@pytest.mark.parametrize("k", [1, 31, 33, 163, 164, 256, 257, 1024])
def test_queued_queries_on_small_stores(gpu, n, k):
    # the prefix's top k listed by the seed, or the prefix streamed again
    x = _store(n, 3)
    w = np.array([0.5, -0.2, 1.0], np.float32)
    rid, rsc, _ = oracle.fte_topk(x, n, k, w, [2, 0, 1])
    with topk_amd.Engine(x) as eng:
        ids, sc = _queue(eng, [(w, [2, 0, 1])] * 3, k)
    c = rid.size  # min(k, n), then padding
    for j in range(3):
        assert np.array_equal(ids[j][:c], rid) and np.array_equal(sc[j][:c], rsc)
        assert np.all(ids[j][c:] == np.uint64(0xFFFFFFFFFFFFFFFF)) and np.all(sc[j][c:] == -np.inf)


@pytest.mark.parametrize("n,values", [((1 << 21) + 5, 1), (3_000_001, 2), (5_000_003, 7)])
def test_tied_scores_take_one_run(gpu, n, values):
    # every chunk of the sample holds more ties than the threshold's rank
    rng = np.random.default_rng(values)
    x = rng.integers(0, values, size=(2, n)).astype(np.float32)
    w, k = np.array([0.5, 1.0], np.float32), 100
    rid, rsc, _ = oracle.fte_topk(x, n, k, w, [0, 1])
    with topk_amd.Engine(x) as eng:
        ids, sc, _ = eng.fte(k, w, [0, 1])
        assert np.array_equal(ids, rid) and np.array_equal(sc, rsc) and eng.stats()["fallback"] == 0
        qi, qs = _queue(eng, [(w, [0, 1])] * 2, k)
    for j in range(2):
        assert np.array_equal(qi[j], rid) and np.array_equal(qs[j], rsc)
