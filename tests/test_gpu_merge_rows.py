"""Batch inserts and removes whose rows sit at the edges of the row merge: rows
around the longest one merged by a wave, around a window of flat positions and
a piece of 64, runs of keys around what one lane places, rows that move to a
new slot, and keys at either end of a row."""
import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import assert_same_csr, need_gpu, say

pytestmark = pytest.mark.gpu
N = 20000


def _rows(lengths, rng):
    """One row per length, of that many spread ids."""
    src = np.repeat(np.arange(len(lengths)), lengths)
    dst = np.concatenate([np.sort(rng.choice(N, k, replace=False)) if k else
                          np.zeros(0, int) for k in lengths])
    return src.astype(np.uint32), dst.astype(np.uint32)


def _batch(lengths, keys, where, rng):
    """`keys` ids per row, at its low end, its high end or anywhere; one in
    four twice."""
    lo, hi = {"low": (0, 400), "high": (N - 400, N), "any": (0, N)}[where]
    rows = len(lengths)
    src = np.repeat(np.arange(rows), keys)
    dst = rng.integers(lo, hi, rows * keys)
    again = rng.random(len(src)) < 0.25
    src, dst = np.concatenate([src, src[again]]), np.concatenate([dst, dst[again]])
    at = rng.permutation(len(src))
    return src[at].astype(np.uint32), dst[at].astype(np.uint32)


@pytest.mark.parametrize("where", ["low", "high", "any"])
@pytest.mark.parametrize("keys", [1, 8, 9, 64, 65, 200])
@pytest.mark.parametrize("lengths", [
    [0] * 6000,
    list(range(0, 130)) * 50,
    [1500, 1527, 1528, 1535, 1536, 1537, 3, 0] * 90,
    [4095, 4096, 2048, 63, 64, 65, 1, 1400, 1400] * 80,
], ids=["empty", "short", "longest", "mixed"])
def test_rows(lengths, keys, where):
    _check(lengths, keys, where)


@pytest.mark.parametrize("rows,length,keys", [
    (3, 1000, 1450), (5, 0, 1530), (64, 900, 600), (4095, 60, 3),
    (4096, 700, 2), (4097, 700, 2), (4099, 30, 70), (16385, 100, 2)])
def test_row_counts(rows, length, keys):
    """Up to 4096 rows have a wave each, more share waves four at a time."""
    _check([length] * rows, keys, "any")


def _check(lengths, keys, where):
    need_gpu()
    rng = np.random.default_rng([keys, len(lengths)])
    g, og = S.SparseMatrixV(N), O.Graph(N)
    s, d = _rows(lengths, rng)
    if len(s):
        g.insert_batch(s, d)
        og.insert_batch(s, d)
    say("rows", len(lengths), "keys", keys, where)
    bs, bd = _batch(lengths, keys, where, rng)
    # half of the removed edges were never there
    rs, rd = _batch(lengths, keys, where, rng)
    rs[::2], rd[::2] = bs[:len(rs[::2])], bd[:len(rs[::2])]
    for _ in range(2):
        g.insert_batch(bs, bd)
        og.insert_batch(bs, bd)
        assert_same_csr(g, og, "insert")
        g.remove_batch(rs, rd)
        og.remove_batch(rs, rd)
        assert_same_csr(g, og, "remove")
