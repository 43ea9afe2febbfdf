"""Queries queued before the store's values change (normalisation with a layout
rebuild, attribute reordering) answer for the values they were queued on."""
import numpy as np
import pytest

import topk_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", ["init", "normalize", "reorder"])
def test_queued_queries_see_the_store_they_were_queued_on(gpu, change):
    import torch
    n, d, k, nq = 1 << 24, 6, 32, 12
    rng = np.random.default_rng(5)
    queries = [(rng.uniform(0.1, 1.0, d).astype(np.float32), rng.permutation(d)[:4]) for _ in range(nq)]
    with topk_amd.Engine.generated(n, d, topk_amd.INDEPENDENT, 2) as eng:
        eng.init(topk_amd.TOPK_INIT_PTA)
        want = [eng.fte(k, w, a) for w, a in queries]
        ids = torch.empty((nq, k), dtype=torch.int64, device="cuda")
        sc = torch.empty((nq, k), dtype=torch.float32, device="cuda")
        for i, (w, a) in enumerate(queries):
            eng.fte_async(k, w, a, ids[i].data_ptr(), sc[i].data_ptr())
        if change == "init":
            eng.init(topk_amd.TOPK_INIT_NORMALIZE | topk_amd.TOPK_INIT_PTA)
        elif change == "normalize":
            eng.init(topk_amd.TOPK_INIT_NORMALIZE)
        else:
            eng.reorder_attr()
        eng.sync()
        got, gsc = ids.cpu().numpy().view(np.uint64), sc.cpu().numpy()
        for i, (rid, rsc, _) in enumerate(want):
            assert np.array_equal(got[i], rid) and np.array_equal(gsc[i], rsc), i
