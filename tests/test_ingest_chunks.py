"""Line counting over file chunks (256 KiB each) and the staged copies of the
text reader, at chunk edges."""
import functools

import numpy as np
import pytest

import oracle
import topk_amd

CHUNK = 256 << 10


@functools.lru_cache(maxsize=None)
def _text(total):
    """Text of one-value lines with blanks among them."""
    rng = np.random.default_rng(total)
    parts = [b"0.5", b"\n", b" \t", b"\r\n", b"7", b"\n\n", b"1e3 "]
    return (b"0.25\n" + b"".join(parts[i] for i in rng.integers(0, len(parts), total // 2)))[:total]


def _file(tmp_path, edges, total, end):
    t = bytearray(_text(total))
    for e, what in edges:
        if e + len(what) <= len(t):
            t[e:e + len(what)] = what
    p = tmp_path / "c.csv"
    p.write_bytes(bytes(t) + end)
    return p


def _count(p):
    return sum(1 for line in p.read_bytes().split(b"\n") if line.strip(b" \t\r\v\f"))


@pytest.mark.parametrize("total", [1, 5, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK, 9 * CHUNK + 17])
@pytest.mark.parametrize("what", [b"\n", b"\n\n", b" \n ", b"1\n", b"\n1", b" " * 400, b"1" * 400, b" " * 200 + b"1"],
                         ids=["nl", "nl2", "blank", "end", "start", "blanks", "digits", "last"])
def test_count_at_chunk_edges(tmp_path, total, what):
    for o in (-len(what), -1, 0):
        edges = [(c * CHUNK + o, what) for c in range(1, 10)]
        for end in (b"", b" ", b"3"):
            p = _file(tmp_path, edges, total, end)
            assert topk_amd.csv_count(str(p))[0] == _count(p)


def test_count_line_longer_than_chunks(tmp_path):
    p = tmp_path / "l.csv"
    p.write_bytes(b"1\n" + b" " * (3 * CHUNK) + b"\n2" + b" " * (2 * CHUNK) + b"\n\n" + b"3")
    assert topk_amd.csv_count(str(p)) == (3, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("n,d", [(3, 2), (9_000, 3), (60_001, 4), (400_003, 8)])
def test_read_through_slots(gpu, tmp_path, n, d):
    """One slot, several, and the last one partly filled, up and down; and the
    same table as a column file."""
    x = topk_amd.generate(n, d, topk_amd.INDEPENDENT, n)
    p = str(tmp_path / "t.csv")
    topk_amd.write_csv(p, x)
    want, _ = oracle.csv_read(p, n, d)
    got, rep = topk_amd.read_csv(p)
    assert np.array_equal(got, want) and rep["rows"] == n
    rm, _ = topk_amd.read_csv(p, rowmajor=True)
    assert np.array_equal(rm.T, want)
    topk_amd.write_colfile(str(tmp_path / "t.col"), want)
    with topk_amd.Engine.from_file(str(tmp_path / "t.col")) as eng:
        w, a = np.ones(d, np.float32), np.arange(d, dtype=np.uint8)
        with topk_amd.Engine(want) as ref:
            for u, v in zip(eng.fte(min(n, 9), w, a), ref.fte(min(n, 9), w, a)):
                assert np.array_equal(u, v)
