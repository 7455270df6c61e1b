"""The symmetry check: edges without a reverse that point up, down or both in
the (degree, id) order, with edge counts around a block's 2048.  A graph taken
for symmetric by mistake shows in BC, which then sums a vertex's paths over
its own row: 0 for a vertex reached by such an edge alone."""
import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import need_gpu, rel_close, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lone", ["none", "up", "down", "both"])
@pytest.mark.parametrize("pairs", [2047, 2048, 100000])
def test_edges_without_reverse(lone, pairs):
    need_gpu()
    rng = np.random.default_rng(pairs)
    n = max(64, pairs // 8)
    s = rng.integers(2, n - 2, pairs)
    d = rng.integers(2, n - 2, pairs)
    s, d = np.concatenate([s, d]), np.concatenate([d, s])
    hub = int(np.bincount(s, minlength=n).argmax())
    # up: from n - 1, which has no other edge, to the hub; down: from the hub
    # to 0; both: as many of one kind as of the other
    if lone in ("up", "both"):
        s, d = np.append(s, n - 1), np.append(d, hub)
    if lone in ("down", "both"):
        s, d = np.append(s, hub), np.append(d, 0)
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    og = O.Graph(n)
    og.insert_batch(s, d)
    off, cols = og.csr()
    g = S.SparseMatrixV(n)
    g.insert_batch(s, d)
    for src in (hub, int(s[0]), n - 1):
        say("bfs, bc", lone, pairs, len(cols), src)
        want, _ = O.bfs(off, cols, src)
        parent, level = S.EdgeMapVertexMap.BFS(g, src, levels=True)
        assert np.array_equal(level, want)
        assert np.array_equal(parent >= 0, want != S.UNREACHED)
        got = S.EdgeMapVertexMap.BC(g, src)
        ok, worst = rel_close(got, O.bc(off, cols, src), 1e-9, 1e-12)
        assert ok, worst
