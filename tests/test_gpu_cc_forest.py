"""CC labels on symmetric graphs whose hubs sit at either end of the ids, with
several large components, chains and isolated vertices, on both sides of the
sizes at which the forest's schedule changes (2^14 and 2^17 vertices), and
chains within and across the blocks of 256 that the first hook is followed in."""
import time

import numpy as np
import pytest

import sstgraph_amd as S
from oracle import oracle as O
from tests.gpu_common import need_gpu, say

pytestmark = pytest.mark.gpu
EMV = S.EdgeMapVertexMap


def _edges(shape, n, rng):
    if shape in ("rmat", "rmat_low"):  # hubs at the top / at the bottom
        scale = n.bit_length() - 1
        s, d = O.rmat(1 << scale, 7, 8 << scale)
        if shape == "rmat_low":
            s, d = n - 1 - s.astype(np.int64), n - 1 - d.astype(np.int64)
    elif shape == "er":
        s, d = rng.integers(0, n, 4 * n), rng.integers(0, n, 4 * n)
    elif shape == "blocks":  # nine components of random edges, hubs on top
        s = rng.integers(0, n, 6 * n)
        d = s - s % 9 + 9 * rng.integers(0, 1 + n // 90, 6 * n) + s % 9
        d = np.where((d < n) & (d % 9 == s % 9), d, s)
    elif shape in ("path", "path_hub"):  # one chain; edges mostly at the top
        s, d = np.arange(0, n - 1), np.arange(1, n)
        if shape == "path_hub":
            k = min(n - 1, 4096)
            top = rng.integers(n - 1 - k, n - 1, (2, 4 * n))
            s, d = np.concatenate([s, top[0]]), np.concatenate([d, top[1]])
    elif shape == "ladder":  # two chains and their rungs
        s, d = np.arange(0, n - 2), np.arange(2, n)
        s, d = np.concatenate([s, s[::2]]), np.concatenate([d, s[::2] + 1])
    else:  # chains: a vertex's neighbours are next to it
        s = np.arange(0, n - 1)
        s = s[s % 1000 != 0]
        d = s + 1
    s, d = np.asarray(s, np.uint32), np.asarray(d, np.uint32)
    return np.concatenate([s, d]), np.concatenate([d, s])


@pytest.mark.parametrize("shape", ["rmat", "rmat_low", "er", "blocks", "chains"])
@pytest.mark.parametrize("n", [1, 255, 16383, 16384, 65537, 131071, 131073])
def test_labels_match_oracle(shape, n):
    _check(shape, n)


@pytest.mark.parametrize("shape", ["path", "path_hub", "ladder"])
@pytest.mark.parametrize("n", [3, 256, 257, 512, 513, 20001, 131072, 300001])
def test_chains_across_blocks(shape, n):
    _check(shape, n)


def _check(shape, n):
    need_gpu()
    rng = np.random.default_rng(n)
    s, d = _edges(shape, n, rng)
    og = O.Graph(n)
    og.insert_batch(s, d)
    off, cols = og.csr()
    g = S.SparseMatrixV(n)
    g.insert_batch(s, d)
    say("cc", shape, n)
    want = O.cc(off, cols)
    for _ in range(2):
        assert np.array_equal(EMV.CC(g), want)


def test_many_graphs_hubs_at_either_end():
    need_gpu()
    rng = np.random.default_rng(1)
    made = [(n, *_edges(shape, n, rng)) for shape, n in
            (("rmat", 4096), ("rmat_low", 4096), ("blocks", 70001),
             ("chains", 5000), ("rmat", 65536), ("er", 9), ("path", 100),
             ("path_hub", 300), ("path", 77), ("path_hub", 1001))]
    M = S.MultiGraph([n for n, _, _ in made])
    M.insert_batches([(i, s, d) for i, (_, s, d) in enumerate(made)])
    for _ in range(3):  # recorded, then replayed
        M.run([0] * len(made), pr_iters=1)
        label = M.results()["label"]
        for i, (n, s, d) in enumerate(made):
            og = O.Graph(n)
            og.insert_batch(s, d)
            assert np.array_equal(M.part(label, i), O.cc(*og.csr())), i


def test_ordered_chain_is_not_walked():
    """A path numbered along its edges takes no longer than one with its ids
    shuffled (it took four times as long while its one chain was walked)."""
    need_gpu()
    n = 1 << 22
    best = []
    for ids in (np.arange(n), np.random.default_rng(5).permutation(n)):
        ids = ids.astype(np.uint32)
        s, d = np.concatenate([ids[:-1], ids[1:]]), np.concatenate([ids[1:], ids[:-1]])
        g = S.SparseMatrixV(n)
        g.insert_batch(s, d)
        out, ts = S.DeviceArray(n, np.uint32), []
        for _ in range(9):
            t = time.perf_counter()
            assert S.lib().sstg_cc(g.handle, out.ptr, S.SSTG_DEVICE_PTRS) == 0
            ts.append(time.perf_counter() - t)
        assert not out.to_host().any()
        best.append(min(ts))
        g.close()
    say("ordered, shuffled (us):", *[int(t * 1e6) for t in best])
    assert best[0] < 2 * best[1]
