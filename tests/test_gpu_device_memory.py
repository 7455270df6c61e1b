"""Device memory kept between graphs: graphs made and dropped in turn and from
several threads hold the right edges whatever their memory held before, and the
memory is given back when the free memory is asked for."""
import threading

import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import assert_same_csr, need_gpu, say

pytestmark = pytest.mark.gpu


def _round(seed, errors):
    try:
        rng = np.random.default_rng(seed)
        for i in range(6):
            n = int(rng.integers(2, 60000))
            m = int(rng.integers(1, 300000))
            s = rng.integers(0, n, m).astype(np.uint32)
            d = rng.integers(0, n, m).astype(np.uint32)
            g, og = S.SparseMatrixV(n), O.Graph(n)
            for lo in range(0, m, 100000):
                g.insert_batch(s[lo:lo + 100000], d[lo:lo + 100000])
            og.insert_batch(s, d)
            assert_same_csr(g, og, f"{seed}/{i} insert")
            g.remove_batch(s[::2], d[::2])
            og.remove_batch(s[::2], d[::2])
            assert_same_csr(g, og, f"{seed}/{i} remove")
            assert np.array_equal(S.EdgeMapVertexMap.BFS(g, 0, levels=True)[1],
                                  O.bfs(*og.csr(), 0)[0])
            g.close()
    except BaseException as e:  # noqa: BLE001 - reported by the main thread
        errors.append(e)


@pytest.mark.parametrize("threads", [1, 4])
def test_graphs_in_turn(threads):
    need_gpu()
    say("graphs from", threads, "threads")
    errors = []
    ts = [threading.Thread(target=_round, args=(100 * threads + t, errors))
          for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    if errors:
        raise errors[0]


def test_memory_is_given_back():
    need_gpu()
    S.SparseMatrixV(4).close()
    free0, _ = S.mem_info()
    n = 1 << 16
    s = np.arange(4000000, dtype=np.uint32) % n
    d = (np.arange(4000000, dtype=np.uint32) // 7) % n
    for _ in range(3):
        g = S.SparseMatrixV(n)
        g.insert_batch(s, d)
        g.close()
    free1, _ = S.mem_info()
    say("free before and after", free0, free1)
    assert free0 - free1 < 64 << 20  # the runtime's own slack
