"""Plain queries whose last stream tile ends past the store, bit for bit
against the CPU oracle: wide tiles (one or two columns, tuned tiles) at the
end of the last column, the exact mode's offset start, the n-entry run with
as many workgroups as a grid may have, and a caller's own store."""
import ctypes

import numpy as np
import pytest

import oracle
import topk_amd
from topk_amd import _lib

pytestmark = pytest.mark.gpu

# (n, d, queried attributes, k, tuning); the last attribute is the end of the column store
CASES = [
    (8_388_609, 1, [0], 64, {}), (8_396_801, 2, [1], 5, {}), (10_000_000, 1, [0], 1000, {}),
    (5_000_001, 2, [0, 1], 200, {"fte_force_exact": 1}), (8_388_609, 2, [1], 200, {"fte_force_exact": 1}),
    (16_385, 3, [2, 0, 1], 20, {"stream_vpt": 8}), (40_001, 17, list(range(17)), 20, {"stream_vpt": 8}),
    (600_001, 4, [3, 2, 1], 20, {"stream_vpt": 8, "stream_grid": 4096}),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, [c[0], c[1], len(c[2]), c[3], *c[4]])))
def test_last_tile_past_the_store(gpu, case):
    n, d, attr, k, tuning = case
    x = topk_amd.generate(n, d, topk_amd.INDEPENDENT, 5)
    x[:, n - 3:] = 1.5  # the last vector's objects are the best ones
    w = np.random.default_rng(n).uniform(0.1, 1.0, d).astype(np.float32)
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, attr)
    with topk_amd.Engine(x) as eng:
        for name, v in tuning.items():
            eng.set_tuning(name, v)
        ids, sc, thr = eng.fte(k, w, attr)
    assert np.array_equal(ids, rid)
    assert np.array_equal(sc.view(np.uint32), rsc.view(np.uint32)) and thr == rthr


@pytest.mark.parametrize("m,vpt", [(12, 1), (13, 1), (6, 2), (7, 2), (3, 4), (4, 4), (1, 8), (2, 8)])
@pytest.mark.parametrize("divide", [0, 1])
def test_unrolled_and_runtime_widths(gpu, m, vpt, divide):
    # the two sides of the unrolling limit, at a ragged size with a second tile per workgroup
    n, k = 1_100_003 * vpt, 33
    x = topk_amd.generate(n, m, topk_amd.INDEPENDENT, 5)
    rng = np.random.default_rng(m)
    w, attr = rng.uniform(-0.3, 1.0, m).astype(np.float32), rng.permutation(m)
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, attr, divide=bool(divide))
    with topk_amd.Engine(x) as eng:
        eng.set_tuning("stream_vpt", vpt)
        eng.set_tuning("score_divide", divide)
        ids, sc, thr = eng.fte(k, w, attr)
    assert np.array_equal(ids, rid)
    assert np.array_equal(sc.view(np.uint32), rsc.view(np.uint32)) and thr == rthr


def test_every_object_a_candidate(gpu):
    # best objects last: the prefix admits the whole store, past the regular
    # buffer, so the run with an n-entry one answers
    n, k = 8_400_003, 64
    x = (np.arange(n, dtype=np.float32) / np.float32(n)).reshape(1, n)
    w = np.ones(1, np.float32)
    rid, rsc, rthr = oracle.fte_topk(x, n, k, w, [0])
    with topk_amd.Engine(x) as eng:
        eng.set_tuning("fte_force_exact", 1)
        for grid in (0, 4096):
            eng.set_tuning("stream_grid", grid)
            ids, sc, thr = eng.fte(k, w, [0])
            assert np.array_equal(ids, rid) and np.array_equal(sc, rsc) and thr == rthr, grid


@pytest.mark.parametrize("n,d,attr", [(8_388_609, 1, [0]), (4_200_001, 2, [0, 1])])
def test_callers_store_of_the_documented_size(gpu, n, d, attr):
    import torch
    k, ld = 64, (n + 3) // 4 * 4
    x = topk_amd.generate(n, d, topk_amd.INDEPENDENT, 5)
    buf = torch.zeros(d * ld + 8192, dtype=torch.float32, device="cuda")
    for m in range(d):
        buf[m * ld:m * ld + n] = torch.from_numpy(x[m]).cuda()
    ids = torch.empty(k, dtype=torch.int64, device="cuda")
    sc = torch.empty(k, dtype=torch.float32, device="cuda")
    st = torch.full((1,), 99, dtype=torch.int32, device="cuda")
    w, a = np.ones(d, np.float32), np.array(attr, np.uint8)
    p = ctypes.c_void_p
    rc = _lib.lib().topk_fte_noalloc(p(buf.data_ptr()), n, d, ld, k, a.size, w.ctypes.data_as(p), a.ctypes.data_as(p),
                                     p(ids.data_ptr()), p(sc.data_ptr()), p(0), p(st.data_ptr()),
                                     p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc == _lib.TOPK_OK and int(st[0]) == _lib.TOPK_OK
    rid, rsc, _ = oracle.fte_topk(x, n, k, w, attr)
    assert np.array_equal(ids.cpu().numpy().view(np.uint64), rid) and np.array_equal(sc.cpu().numpy(), rsc)
