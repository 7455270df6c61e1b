"""The workloads whose speed this framework is judged by.

Each case is work that a program using the framework has it do, through the
Python binding or the C ABI behind it: batch updates of a dynamic graph, a
whole-graph load, and the traversals and reductions over it.  Graphs are rMat
with the effective quadrant probabilities of the reference's generator
(0.25 / 0.05 / 0.05 / 0.65) or Erdos-Renyi, drawn here from a seed; "ef" is
the number of generated edges per vertex, and "sym" graphs get every edge in
both directions, as undirected graphs are stored.
"""
import ctypes
import math

import numpy as np
import torch

import sstgraph_amd as S
from sstgraph_amd import workloads

DEVICE = "cuda"
QUADRANTS = (0.25, 0.05, 0.05, 0.65)
DAMPING = 0.85


def listed():
    return [
        # a trickle of updates to a large live graph: 1,000 edges inserted,
        # a few memberships asked, the edges retracted
        {"name": "update_1e3", "kind": "update", "graph": "rmat", "scale": 24,
         "ef": 16, "sym": True, "batch": 1000},
        # bulk ingestion into the same graph, ten million edges at a time
        {"name": "update_1e7", "kind": "update", "graph": "rmat", "scale": 24,
         "ef": 16, "sym": True, "batch": 10000000},
        # a served graph: an update batch arrives in host memory, a traversal
        # has to see it, the batch is retracted again
        {"name": "stream_1e5", "kind": "stream", "graph": "rmat", "scale": 22,
         "ef": 16, "sym": True, "batch": 100000},
        # loading a graph: an edge list into a new graph, and its CSR out
        {"name": "build_s20", "kind": "build", "graph": "rmat", "scale": 20,
         "ef": 16, "sym": True},
        # a traversal of a small graph, where launches and waits count
        {"name": "bfs_s16", "kind": "bfs", "graph": "rmat", "scale": 16,
         "ef": 16, "sym": True, "source": "hub"},
        # the same of a large one
        {"name": "bfs_s24", "kind": "bfs", "graph": "rmat", "scale": 24,
         "ef": 16, "sym": True, "source": "hub"},
        # the harness's PageRank, in 64 bits
        {"name": "pagerank_s24", "kind": "pagerank", "graph": "rmat",
         "scale": 24, "ef": 16, "sym": True, "iters": 20, "bits": 64},
        # PageRank with compensated 32-bit sums on a graph without hubs, whose
        # vertex count is no power of two
        {"name": "pagerank_f32_er", "kind": "pagerank", "graph": "er",
         "n": 3000001, "ef": 10, "sym": True, "iters": 10, "bits": 32},
        # betweenness, components and triangles of a mid-size social graph
        {"name": "bc_s22", "kind": "bc", "graph": "rmat", "scale": 22,
         "ef": 16, "sym": True, "source": "hub"},
        {"name": "cc_s24", "kind": "cc", "graph": "rmat", "scale": 24,
         "ef": 16, "sym": True},
        {"name": "tc_s22", "kind": "tc", "graph": "rmat", "scale": 22,
         "ef": 16, "sym": True},
        # many small graphs analysed together: BFS, components and PageRank of
        # each, results taken to the host
        {"name": "multi_64", "kind": "multi", "graphs": 64, "spec": 3,
         "iters": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update", "update", "update", "stream", "build", "bfs",
                       "bfs", "pagerank", "pagerank", "bc", "cc", "tc", "multi"])
    if kind == "multi":
        return {"kind": kind, "graphs": _log(rng, 8, 64),
                "spec": rng.randint(4, 1000), "iters": rng.randint(5, 12)}
    top = {"update": 23, "stream": 22, "build": 20, "bfs": 23, "pagerank": 22,
           "bc": 22, "cc": 23, "tc": 21}[kind]
    c = {"kind": kind, "graph": rng.choice(["rmat", "rmat", "er"])}
    if c["graph"] == "rmat":
        c["scale"] = rng.randint(12, top)
    else:
        c["n"] = _log(rng, 1 << 12, 1 << top) | 1
    c["ef"] = rng.randint(6, 16)
    # components, triangles and the served stream are those of undirected
    # graphs; the others also run along one-directional edges
    c["sym"] = kind in ("cc", "tc", "stream", "bc") or rng.random() < 0.8
    if kind in ("update", "stream"):
        c["batch"] = _log(rng, 100, 3000000 if kind == "update" else 300000) | 1
    if kind in ("bfs", "bc"):
        c["source"] = rng.choice(["hub", "any"])
    if kind == "pagerank":
        c["iters"] = rng.randint(5, 20)
        c["bits"] = rng.choice([64, 64, 32])
    return c


# ------------------------------------------------------------------ inputs
def _vertices(case):
    return 1 << case["scale"] if case["graph"] == "rmat" else case["n"]


def _pairs(case, count, gen):
    """count generated edges as two int32 tensors (ids below 2^31)."""
    if case["graph"] == "er":
        n = case["n"]
        return [torch.randint(0, n, (count,), generator=gen, device=DEVICE,
                              dtype=torch.int32) for _ in range(2)]
    a, b, c, _ = QUADRANTS
    src = torch.zeros(count, dtype=torch.int32, device=DEVICE)
    dst = torch.zeros(count, dtype=torch.int32, device=DEVICE)
    for _ in range(case["scale"]):
        r = torch.rand(count, generator=gen, device=DEVICE)
        src.mul_(2).add_(r >= a + b)
        dst.mul_(2).add_(((r >= a) & (r < a + b)) | (r >= a + b + c))
    return [src, dst]


def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    return gen


def _graph_edges(case, gen):
    src, dst = _pairs(case, case["ef"] * _vertices(case), gen)
    if case["sym"]:
        return torch.cat([src, dst]), torch.cat([dst, src])
    return src, dst


def _some(src, dst, count, gen):
    """count edges picked from an edge list."""
    at = torch.randint(0, src.numel(), (count,), generator=gen, device=DEVICE)
    return src[at], dst[at]


def _multi_edges(case, seed):
    """Vertex counts, edge counts and the edges (local ids) of many graphs."""
    gen = _generator(seed)
    sizes, counts, srcs, dsts = [], [], [], []
    for kind, scale, param, _ in workloads.c4_specs(case["graphs"], case["spec"]):
        n = 1 << scale
        one = {"graph": kind, "scale": scale, "n": n}
        s, d = _pairs(one, workloads.c4_edge_count((kind, scale, param, 0)), gen)
        sizes.append(n)
        counts.append(2 * s.numel())
        srcs += [s, d]
        dsts += [d, s]
    return sizes, counts, torch.cat(srcs), torch.cat(dsts)


class _OnDevice(S.DeviceArray):
    """A tensor's memory as the binding's device array; the tensor owns it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.count = tensor.numel()
        self.dtype = np.dtype(str(tensor.dtype).replace("torch.", ""))
        self.nbytes = self.count * tensor.element_size()
        self.ptr = ctypes.c_void_p(tensor.data_ptr())

    def free(self):
        pass


def _source(case, src, n, gen):
    if case["source"] == "hub":
        return int(torch.bincount(src, minlength=n).argmax())
    return int(src[int(torch.randint(0, src.numel(), (1,), generator=gen,
                                     device=DEVICE))])


def _check(status, what):
    if status != S.SSTG_OK:
        raise S.SSTGError(status, what)


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind == "multi":
        sizes, counts, src, dst = _multi_edges(case, seed)
        torch.cuda.synchronize()
        st["multi"] = S.MultiGraph(sizes)
        st["multi"].insert_batches_device(np.arange(len(sizes)), counts,
                                          _OnDevice(src), _OnDevice(dst))
        # each graph's BFS starts at the first generated edge's end
        starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
        st["sources"] = src[torch.from_numpy(starts).to(DEVICE)].cpu().numpy()
        return st
    gen = _generator(seed)
    n = _vertices(case)
    src, dst = _graph_edges(case, gen)
    torch.cuda.synchronize()
    if kind == "build":
        # room for the CSR's columns, of which there are at most as many as pairs
        st.update(n=n, src=_OnDevice(src), dst=_OnDevice(dst),
                  off=torch.empty(n + 1, dtype=torch.int64, device=DEVICE),
                  cols=torch.zeros(src.numel(), dtype=torch.int32, device=DEVICE))
        torch.cuda.synchronize()
        return st
    g = st["graph"] = S.SparseMatrixV(n)
    g.insert_batch(_OnDevice(src), _OnDevice(dst))
    if kind in ("update", "stream"):
        # four fifths fresh edges, one fifth edges that the graph has
        b = case["batch"]
        fresh = _pairs(case, b - b // 5, gen)
        known = _some(src, dst, b // 5, gen)
        bs, bd = (torch.cat([f, k]) for f, k in zip(fresh, known))
        if kind == "stream":  # the served graph stays undirected
            bs, bd = torch.cat([bs, bd]), torch.cat([bd, bs])
            st["batch"] = [x.cpu().numpy().view(np.uint32) for x in (bs, bd)]
        else:
            # memberships: half of the batch's edges, half of the graph's
            some = _some(bs, bd, b // 2, gen)
            old = _some(src, dst, b - b // 2, gen)
            st["batch"] = [_OnDevice(x) for x in (bs, bd)]
            st["ask"] = [torch.cat([s, o]) for s, o in zip(some, old)]
            st["has"] = torch.empty(b, dtype=torch.uint8, device=DEVICE)
    if kind in ("bfs", "bc", "stream"):
        st["source"] = _source(dict(case, source=case.get("source", "hub")),
                               src, n, gen)
    if kind in ("bfs", "stream"):
        st["parent"] = _OnDevice(torch.empty(n, dtype=torch.int32, device=DEVICE))
        st["level"] = _OnDevice(torch.empty(n, dtype=torch.int32, device=DEVICE))
    if kind in ("pagerank", "bc", "cc"):
        wide = {"bc": torch.float64, "cc": torch.int32}.get(
            kind, torch.float64 if case.get("bits") == 64 else torch.float32)
        st["out"] = _OnDevice(torch.empty(n, dtype=wide, device=DEVICE))
    torch.cuda.synchronize()
    return st


# -------------------------------------------------------------------- runs
def run(st):
    kind = st["kind"]
    lib = S.lib()
    if kind == "update":
        g, (src, dst), (rows, cols) = st["graph"], st["batch"], st["ask"]
        g.insert_batch(src, dst)
        inserted = g.M()
        _check(lib.sstg_has_batch(g.handle, rows.data_ptr(), cols.data_ptr(),
                                  rows.numel(), st["has"].data_ptr(),
                                  S.SSTG_DEVICE_PTRS), "has_batch")
        g.remove_batch(src, dst)
        return {"inserted": inserted, "has": st["has"], "left": g.M()}
    if kind == "stream":
        g, (src, dst) = st["graph"], st["batch"]
        g.insert_batch(src, dst)
        inserted = g.M()
        S.EdgeMapVertexMap.BFS(g, st["source"], out=(st["parent"], st["level"]))
        g.remove_batch(src, dst)
        return {"inserted": inserted, "level": st["level"].tensor, "left": g.M()}
    if kind == "build":
        g = S.SparseMatrixV(st["n"])
        g.insert_batch(st["src"], st["dst"])
        _check(lib.sstg_export_csr(g.handle, st["off"].data_ptr(),
                                   st["cols"].data_ptr(), S.SSTG_DEVICE_PTRS),
               "export_csr")
        g.close()
        return {"offsets": st["off"], "columns": st["cols"]}
    if kind == "bfs":
        # any valid parents will do and they differ from run to run, so the
        # parents are asked for and the levels are what is compared
        S.EdgeMapVertexMap.BFS(st["graph"], st["source"],
                               out=(st["parent"], st["level"]))
        return st["level"].tensor
    if kind == "pagerank":
        g, out, iters = st["graph"], st["out"], st["case"]["iters"]
        if st["case"]["bits"] == 64:
            S.EdgeMapVertexMap.PR_S(g, iters, DAMPING, out=out)
        else:
            _check(lib.sstg_pagerank_f32k(g.handle, iters, DAMPING, out.ptr,
                                          S.SSTG_DEVICE_PTRS), "pagerank")
        return out.tensor
    if kind == "bc":
        _check(lib.sstg_bc(st["graph"].handle, st["source"], st["out"].ptr,
                           S.SSTG_DEVICE_PTRS), "bc")
        return st["out"].tensor
    if kind == "cc":
        _check(lib.sstg_cc(st["graph"].handle, st["out"].ptr,
                           S.SSTG_DEVICE_PTRS), "cc")
        return st["out"].tensor
    if kind == "tc":
        return S.EdgeMapVertexMap.TC(st["graph"])
    if kind == "multi":
        st["multi"].run(st["sources"], pr_iters=st["case"]["iters"],
                        damping=DAMPING)
        r = st["multi"].results()
        return {k: r[k] for k in ("level", "label", "rank")}
    raise ValueError(kind)


# -------------------------------------------------------------------- work
def _rmat_cells(scale):
    """(cells, probability, on the diagonal) of the cell classes of an rMat
    adjacency matrix: a cell's probability depends on how often each quadrant
    was taken."""
    a, b, _, d = QUADRANTS
    for i in range(scale + 1):          # quadrant 0
        for j in range(scale + 1 - i):  # quadrants 1 and 2 together
            k = scale - i - j
            cells = math.comb(scale, i) * math.comb(scale - i, j) * 2 ** j
            yield cells, a ** i * b ** j * d ** k, j == 0


def _edges(case, drawn):
    """Expected distinct edges without self-loops after `drawn` pairs."""
    if case["graph"] == "er":
        n = case["n"]
        return n * (n - 1.0) * -math.expm1(-drawn / (n * float(n)))
    return sum(c * -math.expm1(-drawn * p)
               for c, p, diagonal in _rmat_cells(case["scale"]) if not diagonal)


def _rows(case, batch):
    """[(rows, probability that a batch of that many edges touches one,
    probability of a pair's row)] by row class."""
    if case["graph"] == "er":
        p = 1.0 / case["n"]
        return [(case["n"], -math.expm1(-batch * p), p)]
    one = QUADRANTS[2] + QUADRANTS[3]
    s = case["scale"]
    ps = [(math.comb(s, z), (1 - one) ** z * one ** (s - z)) for z in range(s + 1)]
    return [(c, -math.expm1(-batch * p), p) for c, p in ps]


def _update_bytes(case, m, pairs):
    """One batch insert or remove: the pairs read once, each touched row read
    and written once, and its degree and place."""
    classes = _rows(case, pairs)
    touched = sum(c * t for c, t, _ in classes)
    ids = sum(c * t * m * p for c, t, p in classes)
    return 8.0 * pairs + 8.0 * ids + 16.0 * touched


def work(case):
    kind = case["kind"]
    if kind == "multi":
        m = n = 0.0
        for g, scale, param, _ in workloads.c4_specs(case["graphs"], case["spec"]):
            one = {"graph": g, "scale": scale, "n": 1 << scale}
            m += _edges(one, 2 * workloads.c4_edge_count((g, scale, param, 0)))
            n += 1 << scale
        # BFS and components read the edges and write a word a vertex each;
        # every PageRank iteration reads the edges, the degrees and the ranks
        # and writes the ranks
        return {"bytes": 2 * (4 * m + 8 * n) + case["iters"] * (4 * m + 24 * n),
                "flops": case["iters"] * (m + 3 * n)}
    n = float(_vertices(case))
    drawn = case["ef"] * n * (2 if case["sym"] else 1)
    m = _edges(case, drawn)
    if kind == "update":
        b = case["batch"]
        return {"bytes": 2 * _update_bytes(case, m, b) + 13.0 * b, "flops": 0}
    if kind == "stream":
        b = 2 * case["batch"]
        return {"bytes": 2 * _update_bytes(case, m, b) + 4 * m + 16 * n, "flops": 0}
    if kind == "build":
        return {"bytes": 8 * drawn + 8 * n + 4 * m, "flops": 0}
    if kind == "bfs":  # degrees and places, the edges, levels and parents
        return {"bytes": 4 * m + 20 * n, "flops": 0}
    if kind == "pagerank":
        w = case["bits"] // 8
        return {"bytes": case["iters"] * (4 * m + (8 + 2 * w) * n),
                "flops": case["iters"] * (m + 3 * n)}
    if kind == "bc":  # once down and once up
        return {"bytes": 8 * m + 44 * n, "flops": 2 * m + 4 * n}
    if kind == "cc":
        return {"bytes": 4 * m + 16 * n, "flops": 0}
    if kind == "tc":
        return {"bytes": 4 * m + 12 * n, "flops": 0}
    raise ValueError(kind)


# ------------------------------------------------------------------- exact
def _distinct(n, src, dst):
    """The graph's edges as int64 rows and columns, by row."""
    src, dst = src.long(), dst.long()
    keys = torch.unique((src * n + dst)[src != dst])
    return torch.div(keys, n, rounding_mode="floor"), keys % n


def _pagerank(n, rows, cols, iters, share):
    """share: 1 / the vertex count of each vertex's graph."""
    deg = torch.bincount(rows, minlength=n).double()
    x = share.clone()
    for _ in range(iters):
        c = torch.where(deg > 0, x / deg.clamp(min=1), torch.zeros_like(x))
        x = torch.zeros_like(x).index_add_(0, rows, c[cols])
        x = DAMPING * x + (1 - DAMPING) * share
    return x


def _levels(n, rows, cols, source):
    level = torch.full((n,), -1, dtype=torch.int64, device=DEVICE)
    level[source] = 0
    depth = 0
    while True:
        ends = cols[level[rows] == depth]
        ends = ends[level[ends] < 0]
        if not ends.numel():
            return level, depth
        depth += 1
        level[ends] = depth


def _betweenness(n, rows, cols, source):
    level, depth = _levels(n, rows, cols, source)
    steps = []
    for d in range(depth):
        at = (level[rows] == d) & (level[cols] == d + 1)
        steps.append((rows[at], cols[at]))
    sigma = torch.zeros(n, dtype=torch.float64, device=DEVICE)
    sigma[source] = 1
    for u, v in steps:
        sigma.index_add_(0, v, sigma[u])
    delta = torch.zeros_like(sigma)
    for u, v in reversed(steps):
        delta.index_add_(0, u, sigma[u] / sigma[v] * (1 + delta[v]))
    return delta


def exact(case, seed):
    kind = case["kind"]
    if kind == "multi":
        sizes, counts, src, dst = _multi_edges(case, seed)
        size = torch.tensor(sizes, device=DEVICE)
        base = torch.repeat_interleave(size.cumsum(0) - size,
                                       torch.tensor(counts, device=DEVICE))
        n = sum(sizes)
        rows, cols = _distinct(n, src + base, dst + base)
        share = 1.0 / torch.repeat_interleave(size, size).double()
        return {"level": None, "label": None,
                "rank": _pagerank(n, rows, cols, case["iters"], share)}
    if kind not in ("pagerank", "bc"):
        return None  # whole numbers
    gen = _generator(seed)
    n = _vertices(case)
    src, dst = _graph_edges(case, gen)
    rows, cols = _distinct(n, src, dst)
    if kind == "bc":
        return _betweenness(n, rows, cols, _source(case, src, n, gen))
    share = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEVICE)
    return _pagerank(n, rows, cols, case["iters"], share)
