"""Layout builds in little device memory: the build that keeps nothing per
object gives the same layout, a store whose layout just fits is built, and an
allocation that finds no room takes the build's kept scratch back."""
import gc

import numpy as np
import pytest

import topk_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,psize", [(1, 1, 1024), (4097, 5, 1024), (70_001, 9, 2048), (200_003, 32, 1024),
                                       (1_100_001, 6, 65536), (3_000_017, 4, 4096)])
def test_lean_build_gives_the_same_layout(gpu, n, d, psize):
    x = topk_amd.generate(n, d, topk_amd.ANTICORRELATED, 3)
    with topk_amd.Engine(x) as eng:
        eng.set_partition_size(psize)
        layouts = []
        for lean in (0, 1, 0, 1):
            eng.set_tuning("init_lean", lean)
            eng.init(topk_amd.TOPK_INIT_PTA)
            layouts.append(eng.pta_layout())
            w = np.linspace(1.0, 0.2, d, dtype=np.float32)
            got, want = (f(min(64, n), w, list(range(d))) for f in (eng.pta, eng.fte))
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]
            for q in ((min(64, n), w, list(range(d))), (1, -w, [0])):
                ids, sc, thr = eng.batch([q])[0]
                want = eng.fte(*q)
                assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1]) and thr == want[2]
        for got in layouts[1:]:
            for i, (a, b) in enumerate(zip(layouts[0], got)):
                if i or layouts[0][2].max() <= 8192:  # ids of larger partitions are not ordered
                    assert np.array_equal(a, b), i


def _filled(leave):
    """A block of device memory that leaves about `leave` bytes."""
    import torch
    gc.collect()
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    return torch.empty(free - leave, dtype=torch.uint8, device="cuda")


def test_builds_and_batches_in_what_is_left(gpu):
    import torch
    n, d = 1 << 24, 8
    w = np.linspace(1.0, 0.2, d, dtype=np.float32)
    rng = np.random.default_rng(0)
    queries = [(64, rng.uniform(0.1, 1.0, d).astype(np.float32), rng.permutation(d)) for _ in range(512)]
    with topk_amd.Engine.generated(n, d, topk_amd.INDEPENDENT, 1) as eng:
        want = eng.fte(64, w, list(range(d)))
        torch.zeros(1, device="cuda")
        free0, _ = torch.cuda.mem_get_info()
        eng.set_tuning("init_lean", 1)
        eng.init(topk_amd.TOPK_INIT_PTA)
        layout = free0 - torch.cuda.mem_get_info()[0]
        assert layout < n * (4 * d + 4) * 1.25  # columns, ids, statistics: nothing else is kept
        eng.reorder_attr()  # drops the layout
        eng.init(topk_amd.TOPK_INIT_PTA)
    with topk_amd.Engine.generated(n, d, topk_amd.INDEPENDENT, 1) as eng:
        hold = _filled(layout + (150 << 20))  # less than the 24 bytes an object of a usual build
        eng.init(topk_amd.TOPK_INIT_PTA)
        got = eng.pta(64, w, list(range(d)))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        del hold
        torch.cuda.empty_cache()
        eng.init(topk_amd.TOPK_INIT_PTA)  # keeps its scratch
        hold = _filled(64 << 20)
        res = eng.batch(queries)
        del hold
        torch.cuda.empty_cache()
        for q, r in list(zip(queries, res))[::101]:
            ref = eng.fte(*q)
            assert np.array_equal(r[0], ref[0]) and np.array_equal(r[1], ref[1])
