"""Batches over stores of repeated values, where every object of a value lies in
one partition of many chunks: results against the oracle, and no more work
items than a budget of 128 queries an item gives."""
import numpy as np
import pytest

import topk_amd
from test_gpu_batch import make_queries
from test_gpu_batch_items import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [1, 65, 300])
@pytest.mark.parametrize("values", [1, 2])
def test_partitions_of_many_chunks(gpu, values, nq):
    n, d = 300_007, 4
    rng = np.random.default_rng(values)
    x = (rng.integers(0, values, size=(d, n)) + 0.5).astype(np.float32)
    qs = make_queries(rng, nq, d, [1, 16, 100])
    with topk_amd.Engine(x) as eng:
        eng.set_tuning("batch_fused", 1)
        eng.set_tuning("batch_item", 2048)
        for qpi in (0, 16, 128):
            eng.set_tuning("batch_qpi", qpi)
            check(eng, x, qs)
            s = eng.stats()
            if qpi == 0 and values == 1:
                assert s["items"] <= -(-nq // 128) * -(-n // 2048)


@pytest.mark.parametrize("fused", [1, 2])
def test_large_partitions_keep_id_order(gpu, fused):
    # one partition holds every object; its first positions are the lowest ids,
    # so a seed threshold admits few ties and no query takes a second pass
    n, d, nq = 1_000_003, 3, 40
    x = np.full((d, n), 0.5, np.float32)
    qs = make_queries(np.random.default_rng(3), nq, d, [1, 16, 256])
    with topk_amd.Engine(x) as eng:
        eng.init(topk_amd.TOPK_INIT_PTA)
        eng.set_tuning("batch_fused", fused)
        check(eng, x, qs)
        s = eng.stats()
        assert s["fallback"] == 0 and s["partitions_scored"] == nq
        k, w, attr = qs[0]
        ids, _, _ = eng.pta(256, w, attr)
        assert np.array_equal(ids, np.arange(256, dtype=np.uint64)) and eng.stats()["fallback"] == 0


@pytest.mark.parametrize("nq", [1, 7, 8])
def test_few_queries_over_a_larger_store(gpu, nq):
    # the two passes' limit above 2^20 objects, over values that bounds rule out little of
    n, d = (1 << 20) + 4097, 5
    rng = np.random.default_rng(nq)
    x = (rng.random((d, n)) * (rng.random((d, n)) < 0.02)).astype(np.float32)
    qs = make_queries(rng, nq, d, [1, 64, 300])
    with topk_amd.Engine(x) as eng:
        check(eng, x, qs)
        assert (eng.stats()["items"] == 0) == (nq >= 8)  # the query-major pass has no work items
