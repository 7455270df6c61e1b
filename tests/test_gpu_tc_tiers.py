"""Triangle counts where the counting kernels' tables change: every out-list
length across the tier bounds, vertex 0 in and out of the lists, ids that only
differ above 24 bits, and vertex counts around the binning step."""
import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import need_gpu, say

pytestmark = pytest.mark.gpu
EMV = S.EdgeMapVertexMap


def _clique(ids):
    a, b = np.meshgrid(ids, ids)
    keep = a != b
    return a[keep].astype(np.uint32), b[keep].astype(np.uint32)


@pytest.mark.parametrize("k", [3, 17, 18, 65, 66, 130, 258, 514, 600])
@pytest.mark.parametrize("ids", ["low", "spread", "wide"])
def test_clique(k, ids):
    need_gpu()
    rng = np.random.default_rng(k)
    if ids == "low":  # vertex 0 is a member
        n, v = k, np.arange(k)
    elif ids == "spread":
        n = 70001
        v = rng.permutation(np.arange(1, n))[:k]
    else:  # pairs of ids equal in their low 24 bits
        n = (1 << 24) + 4096
        v = rng.permutation(4096)[:(k + 1) // 2]
        v = np.concatenate([v, v + (1 << 24)])[:k]
    g = S.SparseMatrixV(n)
    g.insert_batch(*_clique(v))
    say("clique", k, ids)
    assert EMV.TC(g) == k * (k - 1) * (k - 2) // 6


@pytest.mark.parametrize("n", [5, 1023, 1024, 1025, 20011])
@pytest.mark.parametrize("directed", [False, True])
def test_random_with_hub(n, directed):
    """A random graph, vertex 0 joined to most others (directed rows take the
    lists of smaller ids instead of the oriented ones)."""
    need_gpu()
    rng = np.random.default_rng(n)
    s, d = rng.integers(0, n, 12 * n), rng.integers(0, n, 12 * n)
    hub = np.arange(1, n, 2)
    s, d = np.concatenate([s, hub]), np.concatenate([d, 0 * hub])
    if not directed:
        s, d = np.concatenate([s, d]), np.concatenate([d, s])
    else:
        s, d = np.concatenate([s, 0 * hub]), np.concatenate([d, hub])
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    og = O.Graph(n)
    og.insert_batch(s, d)
    g = S.SparseMatrixV(n)
    g.insert_batch(s, d)
    say("tc", n, directed)
    assert EMV.TC(g) == O.tc(*og.csr())
