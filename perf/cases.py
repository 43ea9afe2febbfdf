"""The work this engine is timed on, through its public entry points.

Stores hold the benchmark distributions (``Engine.generated``), queries carry
weights U(0.1, 1) (``weights`` = "random"), the same with every third one
negated ("signed"), or ones ("ones").  Kinds of work:

* ``fte``      one synchronous plain query (``Engine.fte``)
* ``async``    a run of plain queries left on the device (``fte_async`` + ``sync``)
* ``pta``      one synchronous query over the partition layout (``Engine.pta``)
* ``init``     normalisation and layout build of a resident store, then its
               first query (``Engine.init`` + ``Engine.pta``)
* ``batch``    one synchronous call over many queries, seed thresholds
* ``learned``  batches kept two in flight under a trained predictor
* ``csv``      a text file parsed to a table (``read_csv``)
"""
import tempfile

import numpy as np
import torch

import topk_amd

DISTRIBUTIONS = {"correlated": topk_amd.CORRELATED, "independent": topk_amd.INDEPENDENT,
                 "anticorrelated": topk_amd.ANTICORRELATED, "mixed": topk_amd.MIXED}
TRAIN_QUERIES = 16384  # predictor training set of a "learned" case
QUERIES_PER_BATCH = 1024


def _case(kind, n, d, m, k, dist="independent", weights="random", **more):
    return dict(kind=kind, n=n, d=d, m=m, k=k, dist=dist, weights=weights, **more)


def listed():
    return [
        # a lookup in a small table: nothing but the latency of one call
        dict(_case("fte", 16411, 6, 3, 10), name="fte-16k"),
        # the reference's CPU-runnable case: attributes 4..7, unit weights, k = 16
        dict(_case("fte", 1 << 20, 8, 4, 16, weights="ones"), name="fte-1m"),
        # real-data scores (divided by qq after every term), terms out of order, a ragged size
        dict(_case("fte", 8000003, 12, 7, 100, "anticorrelated", divide=True, shuffled=True), name="fte-8m-divide"),
        # wide queries with negative weights that want a long result list
        dict(_case("fte", 4194301, 20, 20, 1000, "mixed", "signed", shuffled=True), name="fte-4m-k1000"),
        # the plain query of the headline benchmark
        dict(_case("fte", 1 << 26, 8, 8, 64), name="fte-64m"),
        # a consumer on the device: back-to-back queries without host waits
        dict(_case("async", 16777213, 8, 5, 32, "correlated", queries=32), name="async-16m"),
        # the pruned query at the size the partition layout is quoted on
        dict(_case("pta", 1 << 28, 8, 8, 128, "anticorrelated"), name="pta-256m"),
        # what a store pays before its first pruned query
        dict(_case("init", 16777213, 8, 8, 64), name="init-16m"),
        # a small service call: a few dozen mixed queries, no tuning
        dict(_case("batch", 1 << 20, 8, 0, 16, "correlated", queries=32, tuned=False), name="batch-1m"),
        # the multi-query benchmark: mixed store, random attribute subsets, k in 16..256
        dict(_case("batch", 1 << 25, 16, 0, 256, "mixed", queries=QUERIES_PER_BATCH, tuned=True), name="batch-32m"),
        # the headline: a trained predictor, batches of 1024, two in flight
        dict(_case("learned", 1 << 26, 8, 8, 64, queries=4 * QUERIES_PER_BATCH), name="learned-64m"),
        # a text table read from a warm page cache
        dict(_case("csv", 524309, 8, 0, 0), name="csv-512k"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["fte", "fte", "fte", "async", "pta", "init", "batch", "batch", "learned", "csv"])
    dist = rng.choice(sorted(DISTRIBUTIONS))
    weights = rng.choice(["random", "random", "ones", "signed"])
    if kind == "fte":
        d = rng.randint(4, 24)
        n = _log_int(rng, 1 << 12, (1 << 26) * 8 // max(8, d))
        k = min(_log_int(rng, 1, 1024), n)
        return _case("fte", n, d, rng.randint(2, d), k, dist, weights, divide=rng.random() < 0.25,
                     shuffled=rng.random() < 0.5)
    if kind == "async":
        d = rng.randint(4, 12)
        return _case("async", _log_int(rng, 1 << 20, 1 << 25), d, rng.randint(2, d), _log_int(rng, 4, 256), dist,
                     weights, queries=rng.randint(8, 32))
    if kind == "pta":
        d = rng.randint(4, 16)
        return _case("pta", _log_int(rng, 1 << 20, (1 << 28) * 8 // max(8, 2 * d)), d, rng.randint(2, d),
                     _log_int(rng, 8, 256), rng.choice(["anticorrelated", "independent"]), "random")
    if kind == "init":
        d = rng.randint(4, 16)
        return _case("init", _log_int(rng, 1 << 18, 1 << 24), d, d, _log_int(rng, 8, 128), "independent", "random")
    if kind == "batch":
        d = rng.randint(6, 16)
        return _case("batch", _log_int(rng, 1 << 18, 1 << 24), d, 0, _log_int(rng, 16, 256), dist, "random",
                     queries=_log_int(rng, 8, 1024), tuned=rng.random() < 0.5)
    if kind == "learned":
        return _case("learned", _log_int(rng, 1 << 22, 1 << 26), 8, 8, _log_int(rng, 16, 64), "independent", "random",
                     queries=4 * _log_int(rng, 64, QUERIES_PER_BATCH))
    return _case("csv", _log_int(rng, 1 << 12, 1 << 19), rng.randint(2, 12), 0, 0, dist, "random")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _weights(case, rng):
    if case["weights"] == "ones":
        return np.ones(case["d"], np.float32)
    w = rng.uniform(0.1, 1.0, case["d"]).astype(np.float32)
    if case["weights"] == "signed":
        w[2::3] *= -1
    return w


def _queries(case, seed):
    """(k, weights by attribute id, attributes) per query of a case."""
    rng = np.random.default_rng(seed)
    d, kind = case["d"], case["kind"]
    out = []
    for _ in range(case.get("queries", 1)):
        if kind == "batch":  # each its own attribute subset, weights and k
            m = int(rng.integers(max(2, d // 4), d + 1))
            attr = np.sort(rng.permutation(d)[:m])
            k = int(rng.integers(min(16, case["k"]), case["k"] + 1))
        else:
            m, k = case["m"], case["k"]
            attr = rng.permutation(d)[:m] if case.get("shuffled") else np.arange(d - m, d)
        out.append((k, _weights(case, rng), attr.astype(np.uint8)))
    return out


def prepare(case, seed):
    kind, n, d = case["kind"], case["n"], case["d"]
    if kind == "csv":
        f = tempfile.NamedTemporaryFile(suffix=".csv")
        topk_amd.write_csv(f.name, topk_amd.generate(n, d, DISTRIBUTIONS[case["dist"]], seed))
        return {"kind": kind, "file": f}
    eng = topk_amd.Engine.generated(n, d, DISTRIBUTIONS[case["dist"]], seed)
    queries = _queries(case, seed)
    s = {"kind": kind, "eng": eng, "queries": queries}
    if case.get("divide"):
        eng.set_tuning("score_divide", 1)
    if kind == "async":
        s["ids"] = torch.zeros(len(queries), case["k"], dtype=torch.int64, device="cuda")
        s["scores"] = torch.zeros(len(queries), case["k"], dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    if kind == "pta":
        eng.init(topk_amd.TOPK_INIT_PTA)
    if kind in ("batch", "learned"):
        eng.init(topk_amd.TOPK_INIT_PTA)
        per = len(queries) // 4 if kind == "learned" else len(queries)
        s["batches"] = [eng.prepare_batch(queries[i:i + per]) for i in range(0, len(queries), per)]
        for b in s["batches"]:  # slots past a query's own k stay zero
            b.ids[:] = 0
            b.scores[:] = 0
        if kind == "learned":
            train = dict(case, queries=TRAIN_QUERIES)
            eng.learned_train(_queries(train, seed + 0x5eed))
        if case.get("tuned", True):
            eng.batch_autotune(s["batches"][0])
    return s


def run(s):
    kind = s["kind"]
    if kind == "csv":
        return topk_amd.read_csv(s["file"].name)[0]
    eng, queries = s["eng"], s["queries"]
    if kind == "fte":
        k, w, attr = queries[0]
        ids, scores, thr = eng.fte(k, w, attr)
    elif kind == "pta":
        k, w, attr = queries[0]
        ids, scores, thr = eng.pta(k, w, attr)
    elif kind == "init":
        k, w, attr = queries[0]
        eng.init(topk_amd.TOPK_INIT_NORMALIZE | topk_amd.TOPK_INIT_PTA)
        ids, scores, thr = eng.pta(k, w, attr)
    elif kind == "async":
        for i, (k, w, attr) in enumerate(queries):
            eng.fte_async(k, w, attr, s["ids"][i].data_ptr(), s["scores"][i].data_ptr())
        eng.sync()
        return {"ids": s["ids"], "scores": s["scores"]}
    elif kind == "batch":
        b = s["batches"][0]
        eng.batch_run(b)
        ids, scores, thr = b.ids, b.scores, b.thr
    else:
        tickets = []
        for b in s["batches"]:
            if len(tickets) == 2:
                eng.batch_wait(tickets.pop(0))
            tickets.append(eng.batch_submit(b))
        for t in tickets:
            eng.batch_wait(t)
        return [{"ids": b.ids.view(np.int64), "scores": b.scores, "thr": b.thr} for b in s["batches"]]
    return {"ids": ids.view(np.int64), "scores": scores, "thr": thr}


def work(case):
    """Plain queries and ingest cannot do without one read of their columns or
    text; an indexed query cannot do without its layout's partition bounds
    (2 d + 2 values per 4096 objects) and its results."""
    kind, n, d, k = case["kind"], case["n"], case["d"], case["k"]
    nq = case.get("queries", 1)
    result = 12.0 * k
    bounds = (n / 4096 + 1) * (2 * d + 2) * 4.0
    if kind == "csv":
        return {"bytes": n * d * (9.0 + 4.0), "flops": 2.0 * n * d}
    if kind in ("fte", "async"):
        return {"bytes": nq * (4.0 * case["m"] * n + result), "flops": nq * 2.0 * case["m"] * n}
    if kind == "init":  # read and written once by the normalisation, read and written in partition order
        return {"bytes": 16.0 * d * n + bounds + result, "flops": 4.0 * n * d}
    batches = 4 if kind == "learned" else 1
    m = case["m"] or d / 2
    return {"bytes": batches * bounds + nq * (164.0 + result), "flops": nq * (n / 4096 + k) * 2.0 * m}


# ---------------------------------------------------------------------------
# the same in 64 bits (plain torch)
# ---------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _signed(x):
    x &= _M64
    return x - (1 << 64) if x >> 63 else x


def _shift(z, s):  # logical right shift of int64 bits
    return (z >> s) & ((1 << (64 - s)) - 1)


def _mix(z):  # SplitMix64's finaliser on int64 tensors (wrapping)
    z = z + _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shift(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shift(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shift(z, 31)


def _bits24(sk, i, slot, tag):
    return _shift(_mix((i * 64 + slot) * 16 + tag + sk), 40)


def _uniform(sk, i, slot):
    return _bits24(sk, i, slot, 0).float() * 2.0 ** -24


def _normal(sk, i, slot):
    s = sum(_bits24(sk, i, slot, t) for t in range(1, 13)) - 6 * 16777216
    return s.float() * 2.0 ** -24


def _columns(case, seed, lo, hi):
    """Objects [lo, hi) of a case's store as the generator defines them: binary32, (d, hi - lo)."""
    n, d, dist = case["n"], case["d"], case["dist"]
    i = torch.arange(lo, hi, dtype=torch.int64, device="cuda")
    sk = int(_mix(torch.tensor([_signed(seed ^ 0x5DEECE66D)], dtype=torch.int64))[0])

    def correlated():
        u = _uniform(sk, i, 63)
        return torch.stack([(u + _normal(sk, i, m) * 0.05).clamp(0, 1) for m in range(d)])

    def independent():
        return torch.stack([_uniform(sk, i, m) for m in range(d)])

    def anticorrelated():
        x = independent()
        total = torch.zeros_like(x[0])
        for m in range(d):
            total = total + x[m]
        c = (d * 0.5 + _normal(sk, i, 63) * 0.05 - total) / torch.tensor(float(d), device="cuda")
        return (x + c).clamp(0, 1)

    if dist != "mixed":
        return {"correlated": correlated, "independent": independent, "anticorrelated": anticorrelated}[dist]()
    return torch.where(i < n // 3, correlated(), torch.where(i < 2 * (n // 3), independent(), anticorrelated()))


def exact(case, seed):
    kind, n, d = case["kind"], case["n"], case["d"]
    nq = case.get("queries", 1)
    step = max(1, min(1 << 21, (1 << 27) // nq))  # objects scored at a time
    if kind == "csv":  # the values as the text gives them: six decimals
        x = torch.cat([_columns(case, seed, lo, min(n, lo + step)) for lo in range(0, n, step)], 1)
        return np.round(x.double().cpu().numpy() * 1e6) / 1e6
    lo_hi = None
    if kind == "init":
        parts = [_columns(case, seed, lo, min(n, lo + step)).double() for lo in range(0, n, step)]
        lo_hi = (torch.stack([p.amin(1) for p in parts]).amin(0)[:, None],
                 torch.stack([p.amax(1) for p in parts]).amax(0)[:, None])
        del parts
    queries = _queries(case, seed)
    coef = torch.zeros(nq, d, dtype=torch.float64, device="cuda")
    for q, (k, w, attr) in enumerate(queries):
        for j, a in enumerate(attr):
            scale = float(len(attr)) ** -(len(attr) - j) if case.get("divide") else 1.0
            coef[q, int(a)] += float(w[a]) * scale
    kmax = max(q[0] for q in queries)
    best = torch.empty(nq, 0, dtype=torch.float64, device="cuda")
    for lo in range(0, n, step):
        x = _columns(case, seed, lo, min(n, lo + step)).double()
        if lo_hi:
            x = (x - lo_hi[0]) / (lo_hi[1] - lo_hi[0])
        s = torch.topk(coef @ x, min(kmax, x.shape[1]), dim=1).values
        best = torch.cat([best, s], 1)
        best = torch.topk(best, min(kmax, best.shape[1]), dim=1).values
    best = best.cpu().numpy()
    scores = np.zeros((nq, kmax))
    thr = np.zeros(nq)
    for q, (k, _, _) in enumerate(queries):
        c = min(k, n)
        scores[q, :c] = best[q, :c]
        thr[q] = best[q, c - 1]
    if kind == "async":
        return {"ids": None, "scores": scores}
    if kind in ("fte", "pta", "init"):
        return {"ids": None, "scores": scores[0, :min(queries[0][0], n)], "thr": float(thr[0])}
    if kind == "batch":
        return {"ids": None, "scores": scores.ravel(), "thr": thr}
    per = nq // 4
    return [{"ids": None, "scores": scores[b * per:(b + 1) * per].ravel(), "thr": thr[b * per:(b + 1) * per]}
            for b in range(4)]
