"""Candidate staging, item order and the choice of pass of the batched path
against the oracle (cpu/TPAc.h:209-254 findTopKsimdMQ), bit for bit."""
import numpy as np
import pytest

import topk_amd
from test_gpu_batch import make_queries, oracle_batch

pytestmark = pytest.mark.gpu


def check(eng, x, qs):
    ref = oracle_batch(x, x.shape[1], qs)
    for i, ((gi, gs, _), (ri, rs)) in enumerate(zip(eng.batch(qs), ref)):
        assert np.array_equal(gi, ri) and np.array_equal(gs.view(np.uint32), rs.view(np.uint32)), i


SHAPES = [(8, 4, 256), (8, 8, 512), (8, 16, 256), (8, 16, 512), (8, 4, 1024), (16, 2, 256), (16, 4, 512), (16, 8, 256),
          (20, 2, 512), (20, 4, 256)]


@pytest.mark.parametrize("d,vpt,bs", SHAPES)
def test_stage_fills(gpu, d, vpt, bs):
    """Few distinct values: every tile of a query is full of candidates and of
    ties, the stage overflows inside an item; 70 queries cross a lane block."""
    rng = np.random.default_rng(d * vpt + bs)
    n = 30_001
    x = (np.rint(rng.random((d, n)) * 3) / 3).astype(np.float32)
    for order in ("sorted", "shuffled"):
        qs = make_queries(rng, 70, d, [1, 64, 1024], order=order, mmax=4)
        with topk_amd.Engine(x) as eng:
            for name, v in (("batch_fused", 1), ("batch_vpt", vpt), ("batch_bs", bs)):
                eng.set_tuning(name, v)
            for qpi in (0, 16, 128):
                eng.set_tuning("batch_qpi", qpi)
                check(eng, x, qs)


@pytest.mark.parametrize("nq", [1, 3, 64, 65, 1024])
@pytest.mark.parametrize("d,n", [(6, 1), (8, 4097), (8, 262_144), (8, 262_145), (12, 16_384), (12, 16_385), (17, 5000)])
def test_choice_of_pass(gpu, d, n, nq):
    """Both sides of the limits between the two passes, and the smallest and
    largest query budgets the entries give."""
    rng = np.random.default_rng(n + nq)
    x = topk_amd.generate(n, d, topk_amd.ANTICORRELATED, n)
    qs = make_queries(rng, nq, d, [1, 16, 100])
    with topk_amd.Engine(x) as eng:
        check(eng, x, qs)
        eng.set_tuning("batch_fused", 1)
        check(eng, x, qs)


@pytest.mark.parametrize("n", [63, 64, 65, 129, 4096, 16_385, 300_007])
@pytest.mark.parametrize("levels", [2, 1000, 0])
def test_select_ends(gpu, n, levels):
    """Lists of 63 to 65 keys and more, k at both ends, few distinct values
    and many; single queries and batches over the same store."""
    rng = np.random.default_rng(n + levels)
    d = 5
    x = rng.random((d, n)).astype(np.float32)
    if levels:
        x = np.rint(x * levels).astype(np.float32) / np.float32(levels)
    ks = [k for k in (1, 2, 63, 64, 65, 66, 1024) if k <= n]
    qs = make_queries(rng, 3 * len(ks), d, ks)
    with topk_amd.Engine(x) as eng:
        check(eng, x, qs)
        ref = oracle_batch(x, n, qs)
        for (k, w, a), (ri, rs) in zip(qs, ref):
            for got in (eng.fte(k, w, a), eng.pta(k, w, a)):
                assert np.array_equal(got[0], ri) and np.array_equal(got[1].view(np.uint32), rs.view(np.uint32))


@pytest.mark.parametrize("nq", [17, 300, 1024, 1025])
@pytest.mark.parametrize("mode", [1, 2])
def test_many_second_passes(gpu, nq, mode):
    """Long lists over anticorrelated objects and weights of both signs: a
    third of the queries overflow their candidate list and rerun, few enough
    and too many for 64 slices each, in batches on both sides of 1024."""
    n, d = 1_000_003, 8
    qs = make_queries(np.random.default_rng(nq), nq, d, [512, 1024], mmin=5, wlo=-1.0)
    with topk_amd.Engine.generated(n, d, topk_amd.ANTICORRELATED, 5) as eng:
        eng.set_tuning("batch_fused", mode)
        got = eng.batch(qs)
        assert eng.stats()["retried"] > 2
        for i, (q, (gi, gs, gt)) in enumerate(zip(qs, got)):
            ri, rs, rt = eng.fte(*q)
            assert np.array_equal(gi, ri) and np.array_equal(gs.view(np.uint32), rs.view(np.uint32)) and gt == rt, i
