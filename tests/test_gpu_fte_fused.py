"""One-launch FTE (threshold sample, stream and select in one kernel) at the
edges of its plans, bit for bit against the CPU oracle: stores that fit the
select whole (4096 objects), the own sample (to 2^19), the shared sample and
the ticketed tiles above, rank / interval / radix selects, more workgroups
than the select scans in one wave."""
import numpy as np
import pytest

import oracle
import topk_amd

pytestmark = pytest.mark.gpu

# (n, d, m, k, distribution or "ties" / "sorted", stream_grid)
CASES = [
    (4095, 3, 2, 1024, 1, 0), (4096, 3, 3, 10, 1, 0), (4097, 3, 3, 10, 1, 0), (4111, 17, 17, 1000, 3, 0),
    (65_521, 4, 1, 1, 2, 0), (65_521, 9, 9, 257, 0, 0), (65_521, 2, 2, 64, "sorted", 0),
    (65_521, 2, 2, 300, "ties", 0), ((1 << 19) - 1, 5, 5, 1024, 3, 0), (1 << 19, 2, 2, 16, "ties", 0),
    ((1 << 19) + 1, 2, 2, 16, "ties", 0), ((1 << 19) + 1, 20, 20, 1024, 3, 0), ((1 << 19) + 1, 3, 2, 100, "sorted", 0),
    (2_100_001, 8, 8, 128, 0, 0), (2_101_249, 8, 8, 1, 1, 0), (3_000_001, 16, 16, 200, 2, 0),
    (3_000_001, 2, 2, 200, 1, 257), (3_000_001, 1, 1, 64, 1, 3), (3_000_001, 4, 3, 900, 3, 4096),
]


def _columns(n, d, kind):
    if kind == "ties":  # a few distinct values: long runs of equal scores
        return (np.random.default_rng(n).integers(0, 4, size=(d, n)) / 4.0).astype(np.float32)
    if kind == "sorted":  # neighbouring ids score alike, the best ones last
        return np.tile(np.arange(n, dtype=np.float32) / np.float32(n), (d, 1))
    return topk_amd.generate(n, d, kind, 7)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_one_launch_fte_matches_oracle(gpu, case):
    n, d, m, k, kind, grid = case
    x = _columns(n, d, kind)
    rng = np.random.default_rng(n + k)
    w = rng.uniform(-0.2, 1.0, d).astype(np.float32)
    attr = rng.permutation(d)[:m]
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, attr)
    with topk_amd.Engine(x) as eng:
        if grid:
            eng.set_tuning("stream_grid", grid)
        for _ in range(2):  # the first call leaves the pipeline's state clean
            ids, sc, thr = eng.fte(k, w, attr)
            assert np.array_equal(ids, rid)
            assert np.array_equal(sc.view(np.uint32), rsc.view(np.uint32)) and thr == rthr
