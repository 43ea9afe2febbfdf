"""Partition queries at the edges of the cut pass's groups: 4 to 64
partitions a wave, the last group partly filled, partitions of one object, and
candidate counts on both sides of the select's LDS room."""
import numpy as np
import pytest

import topk_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3000, 1024 * 257, 1024 * 700, 1024 * 1030, 1024 * 4096 + 5, 1024 * 5000 + 1, 66_100_003])
@pytest.mark.parametrize("d,distr", [(2, topk_amd.ANTICORRELATED), (9, topk_amd.CORRELATED), (17, topk_amd.INDEPENDENT)])
def test_group_edges(gpu, n, d, distr):
    if n > 10**7 and d > 2:
        pytest.skip("the widest groups once")
    rng = np.random.default_rng(n + d)
    with topk_amd.Engine.generated(n, d, distr, n) as eng:
        eng.set_partition_size(1024)
        eng.init(topk_amd.TOPK_INIT_PTA)
        for k in (1, 64, 1024):
            for m in (1, d):
                w = rng.uniform(0.1, 1.0, d).astype(np.float32)
                a = rng.permutation(d)[:m].astype(np.uint8)
                for _ in range(2):
                    got, want = eng.pta(k, w, a), eng.fte(k, w, a)
                    assert np.array_equal(got[0], want[0]), (k, m)
                    assert np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32)) and got[2] == want[2]


@pytest.mark.parametrize("levels", [1, 2, 5])
def test_crowded_candidates(gpu, levels):
    """Few distinct scores: ties at the threshold crowd the select."""
    rng = np.random.default_rng(levels)
    n, d = 200_003, 3
    x = (np.rint(rng.random((d, n)) * levels) / levels).astype(np.float32)
    w = np.array([1.0, 0.5, 0.25], np.float32)
    with topk_amd.Engine(x) as eng:
        eng.init(topk_amd.TOPK_INIT_PTA)
        for k in (1, 100, 1024):
            for a in ([0], [2, 0], [0, 1, 2]):
                a = np.array(a, np.uint8)
                got, want = eng.pta(k, w, a), eng.fte(k, w, a)
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]
