"""The partition layout the device builds (sample, k-d tree, counting sort,
order inside a partition, bound statistics) against a plain numpy
restatement of its rules: at most one workgroup's subtree, device-wide tree
levels above it, uneven leaf counts, ties on the split values, partitions
past the sorted size."""
import numpy as np
import pytest

import topk_amd

pytestmark = pytest.mark.gpu


def _leaves(x, n, L):
    """Leaf of every object under the tree over the sample."""
    ns = min(n, max(L * 64, 1 << 20))
    rows = x[:, np.arange(ns, dtype=np.int64) * n // ns]
    leaf = np.empty(n, np.int64)

    def split(idx, objs, lo, nl):
        if nl == 1:
            leaf[objs] = lo
            return
        nleft = nl // 2
        v = rows[:, idx]
        axis = int(np.argmax((v.max(axis=1) - v.min(axis=1)).astype(np.float32)))
        order = idx[np.lexsort((idx, v[axis]))]
        mid = idx.size * nleft // nl
        at = rows[axis, order[mid]]
        below = x[axis, objs] < at
        split(np.sort(order[:mid]), objs[below], lo, nleft)
        split(np.sort(order[mid:]), objs[~below], lo + nleft, nl - nleft)

    split(np.arange(ns), np.arange(n), 0, L)
    return leaf


def _data(kind, n, d):
    if kind == "ties":
        return (np.random.default_rng(n).integers(0, 5, size=(d, n)) / 4.0).astype(np.float32) - np.float32(0.5)
    return topk_amd.generate(n, d, kind, 3)


@pytest.mark.parametrize("n,d,psize,kind", [
    (3000, 3, 1024, 1), (4097, 5, 1024, 2), (70_001, 8, 1024, 0), (70_001, 9, 2048, 3), (70_001, 2, 1024, "ties"),
    (200_003, 32, 1024, 1), (1_100_001, 4, 4096, 3), (1_100_001, 6, 65536, 1),
])
def test_layout_matches_restatement(gpu, n, d, psize, kind):
    x = _data(kind, n, d)
    L = (n + psize - 1) // psize
    leaf = _leaves(x, n, L)
    size = np.bincount(leaf, minlength=L)
    off = np.concatenate([[0], np.cumsum((size + 255) // 256 * 256)])
    with topk_amd.Engine(x) as eng:
        eng.set_partition_size(psize)
        for _ in range(2):  # a rebuild gives the same layout
            eng.init(topk_amd.TOPK_INIT_PTA)
            pid, poff, psz, pmax, pmin = eng.pta_layout()
            assert np.array_equal(psz, size) and np.array_equal(poff, off)
            for p in range(L):
                ids = np.flatnonzero(leaf == p)
                got = pid[off[p]:off[p] + size[p]]
                assert np.all(pid[off[p] + size[p]:off[p + 1]] == 0xFFFFFFFF)
                if size[p] <= 8192:
                    s = np.zeros(ids.size, np.float32)
                    for m in range(d):
                        s = s + x[m, ids]
                    ids = ids[np.lexsort((ids, -s.astype(np.float64)))]
                    assert np.array_equal(got, ids)
                else:
                    assert np.array_equal(np.sort(got), ids)
                if size[p]:
                    assert np.array_equal(pmax[p], x[:, ids].max(axis=1))
                    assert np.array_equal(pmin[p], x[:, ids].min(axis=1))
        k, w = min(64, n), np.linspace(1.0, 0.2, d, dtype=np.float32)
        want = eng.fte(k, w, list(range(d)))
        got = eng.pta(k, w, list(range(d)))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]) and got[2] == want[2]
        for q in ((k, w, list(range(d))), (1, -w, [0]), (min(16, n), w, [d - 1, 0])):
            ids, sc, thr = eng.batch([q])[0]
            want = eng.fte(*q)
            assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1]) and thr == want[2]
