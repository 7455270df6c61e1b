"""BFS where its top-down levels change hands: device-driven batches, the
one-block tail and host-sized pushes, with frontiers around the tile and cap
sizes, chains longer than any batch, and vertices without out-edges, many of
them in one frontier."""
import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import need_gpu, rel_close, say

pytestmark = pytest.mark.gpu
EMV = S.EdgeMapVertexMap


def _check(n, s, d, sources, sym=True):
    s, d = np.asarray(s, np.uint32), np.asarray(d, np.uint32)
    if sym:
        s, d = np.concatenate([s, d]), np.concatenate([d, s])
    og = O.Graph(n)
    og.insert_batch(s, d)
    off, cols = og.csr()
    g = S.SparseMatrixV(n)
    g.insert_batch(s, d)
    for src in sources:
        say("bfs", n, len(cols), src)
        want, _ = O.bfs(off, cols, src)
        parent, level = EMV.BFS(g, src, levels=True)
        assert np.array_equal(level, want)
        reached = want != S.UNREACHED
        assert np.array_equal(parent >= 0, reached) and parent[src] == src
        v = np.nonzero(reached)[0]
        v = v[v != src]
        p = parent[v]
        assert np.all(want[p] + 1 == want[v])
        # every tree edge is an edge: its key is among the graph's
        keys = np.repeat(np.arange(n, dtype=np.uint64), np.diff(off).astype(np.int64))
        keys = keys * np.uint64(n) + cols
        assert np.isin(p.astype(np.uint64) * np.uint64(n) + v.astype(np.uint64),
                       keys).all()
    return off, cols, g


@pytest.mark.parametrize("leaves", [1, 511, 512, 513, 2047, 2049, 131071,
                                    131073, 262145])
@pytest.mark.parametrize("sym", [True, False])
def test_stars_joined(leaves, sym):
    """A source, its leaves, and a second hub behind them: frontiers of 1,
    `leaves` and 1 vertices (leaves without out-edges when directed)."""
    need_gpu()
    n = leaves + 3
    leaf = np.arange(1, leaves + 1)
    s = np.concatenate([0 * leaf, leaf[::3], [leaves + 1]])
    d = np.concatenate([leaf, 0 * leaf[::3] + leaves + 1, [leaves + 2]])
    _check(n, s, d, [0, 1, leaves + 1, leaves + 2], sym)


@pytest.mark.parametrize("n", [2, 13, 14, 1500, 5000])
def test_chain(n):
    need_gpu()
    v = np.arange(n - 1)
    _check(n, v, v + 1, [0, n // 2, n - 1])


@pytest.mark.parametrize("degree", [1 << 20, (1 << 20) + 1])
def test_second_level_at_the_cap(degree):
    """In a graph too large to stay on the device, a second frontier of the
    cap's edges, or one more, and a third that reads its offsets."""
    need_gpu()
    hubs, n = 64, 1 << 21
    rng = np.random.default_rng(degree)
    per = np.full(hubs, (degree - hubs) // hubs)
    per[: degree - hubs - per.sum()] += 1  # with the source's edge: `degree`
    s = np.repeat(np.arange(1, hubs + 1), per)
    d = hubs + 1 + np.concatenate([rng.permutation(n - hubs - 1)[:k] for k in per])
    extra = rng.integers(hubs + 1, n, (2, 2 << 20))
    s = np.concatenate([np.zeros(hubs, int), s, extra[0]])
    d = np.concatenate([np.arange(1, hubs + 1), d, extra[1]])
    _check(n, s, d, [0])


@pytest.mark.parametrize("sym", [True, False])
def test_random_graph_any_source(sym):
    need_gpu()
    n = 300001
    rng = np.random.default_rng(3)
    s, d = rng.integers(0, n, 2 * n), rng.integers(0, n, 2 * n)
    _check(n, s, d, [0, 7, n - 1], sym)


CAP = 1 << 20  # most edges of a device-driven frontier in a graph of over 2^22


@pytest.mark.parametrize("sinks,edges", [
    (CAP + CAP // 2, 3000),   # the second frontier itself over the cap
    (CAP - 3000, 6000),       # degrees 2: sinks and edges 3000 over
    (CAP - 6000, 6000),       # edges with a sink counted as one: the cap
    (CAP - 5999, 6000),       # one over
    (CAP - 9000, 6000),       # vertices and edges together: the cap
    (CAP - 8999, 6000),       # one over
])
def test_directed_frontier_of_sinks(sinks, edges):
    """A frontier of about a cap's worth of vertices without out-edges, among
    them edges / 2 that lead on for three more levels, behind frontiers that
    only a push sized by the host expands."""
    need_gpu()
    on, first = edges // 2, CAP + 1
    src, a = 0, np.arange(1, first + 1)
    b = first + 1 + np.arange(sinks + on)
    c = b[-1] + 1 + np.arange(edges)
    e = c[-1] + 1 + np.arange(5)
    n = int(e[-1]) + 1 + 4096
    rng = np.random.default_rng(edges + sinks)
    lead = rng.permutation(b)[:on]
    parts = [(np.full(first, src), a), (a[np.arange(len(b)) % first], b),
             (np.repeat(lead, 2), c), (c[::7], np.full(len(c[::7]), e[0])),
             (e[:-1], e[1:])]
    # edges out of reach, up to a graph too large to stay on the device
    m = sum(len(x) for x, _ in parts)
    f = n - 4096 + rng.integers(0, 4096, (2, 3 << 20))
    s = np.concatenate([x for x, _ in parts] + [f[0]]).astype(np.uint32)
    d = np.concatenate([y for _, y in parts] + [f[1]]).astype(np.uint32)
    say("sinks", sinks, edges, m)
    off, cols, g = _check(n, s, d, [src], False)
    assert len(cols) > 1 << 22 and g.M() == len(cols)
    assert np.array_equal(EMV.BF(g, src), O.bf(off, cols, src))
    ok, worst = rel_close(EMV.BC(g, src), O.bc(off, cols, src), 1e-9, 1e-12)
    assert ok, worst


def _layers(flip, rng):
    """A source, 2^16 vertices behind it, and two more layers with degrees on
    both sides of every pull class (32, 128, 2048), the last with neighbours
    in the middle one only; flip: ids reversed, so rows are read from the
    other end."""
    near = np.arange(1, (1 << 16) + 1)
    per = {1: 20000, 8: 20000, 32: 3000, 33: 3000, 128: 600, 129: 600,
           2048: 100, 2049: 100, 6000: 30}
    degree = np.repeat(list(per), list(per.values()))
    mid = near[-1] + 1 + np.arange(len(degree))
    far = mid[-1] + 1 + np.arange(len(degree) // 10)
    ends = [(np.zeros(len(near), int), near)]
    for ids, back, deg in ((mid, near, degree), (far, mid, degree[::10])):
        s = np.repeat(ids, deg)
        ends.append((s, rng.choice(back, len(s))))
    s = np.concatenate([x for x, _ in ends])
    d = np.concatenate([y for _, y in ends])
    s, d = np.concatenate([s, near]), np.concatenate([d, rng.permutation(near)])
    extra = rng.choice(near, (2, 1200000))  # over 2^22 edges in all
    s, d = np.concatenate([s, extra[0]]), np.concatenate([d, extra[1]])
    n = int(far[-1]) + 2  # and one vertex of no edge
    return (n, n - 1 - s, n - 1 - d, n - 1) if flip else (n, s, d, 0)


@pytest.mark.parametrize("flip", [False, True])
def test_bottom_up_steps(flip):
    """A graph too large to stay on the device whose second and third steps
    are bottom-up, with vertices of every pull class found in each."""
    need_gpu()
    n, s, d, src = _layers(flip, np.random.default_rng(11))
    off, cols, g = _check(n, s, d, [src])
    assert len(cols) > 1 << 22
    alpha, beta = g.bfs_switch()
    level, _ = O.bfs(off, cols, src)
    deg = np.diff(off).astype(np.int64)
    size = [(level == k).sum() for k in range(4)]
    edges = [deg[level == k].sum() for k in range(4)]
    # the second step: over the cap, growing, and over the rest's share
    assert edges[1] > CAP and size[1] > size[0]
    assert edges[1] > (len(cols) - edges[0] - edges[1]) / alpha
    assert size[2] >= n / beta  # the third stays bottom-up
    for k in (2, 3):
        assert (np.histogram(deg[level == k], [1, 33, 129, 2049, 1 << 32])[0] > 0).all()


@pytest.mark.parametrize("flip", [False, True])
def test_one_edge_without_reverse(flip):
    """The same graph with one edge more, the only one of the vertex it ends
    at: bottom-up steps would miss that vertex."""
    need_gpu()
    n, s, d, src = _layers(flip, np.random.default_rng(11))
    lone, near = (0, n - 2 - 77) if flip else (n - 1, 1 + 77)
    s, d = np.concatenate([s, d, [near]]), np.concatenate([d, s, [lone]])
    off, cols, _ = _check(n, s, d, [src], False)
    assert O.bfs(off, cols, src)[0][lone] == 2
