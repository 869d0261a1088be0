"""The workloads this library is timed on, through its public entry points.

Each case names what a program does with the library (``op``) and the graph it
does it on.  Graphs are the two kinds the library's benchmark and tests use:
Erdos-Renyi (``er``: flat, degrees near their mean) and R-MAT with the
Graph500 quadrant weights (``rmat``: skewed, long hub lists), with ``n``
vertices and exactly ``edges`` distinct undirected edges.  They are made here with torch (on the GPU when there is one) and oriented by
(degree, id) into the DAG that a program gets from ``Graph.orientation()``.

ops
  count      Context.count of a resident graph: every later count of a graph
             that a program uploaded once
  partition  Context.count of one part of a split DAG with its halo: what one
             GPU of several does
  solver     TCSolver(g), nothing kept: the whole drop-in call on a host DAG
             (``context``: whether the program holds a Context for it)
  local      Context.count_local: the count attributed to edges, vertices and
             the parts of a split, as asked for
  batch      Batch.count: many small graphs resident together, one call
  serve      Server: requests submitted one after another, all results polled
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hetegeneous_parallel_programming_amd import Graph
from hetegeneous_parallel_programming_amd.graph import PartitionedGraph
from hetegeneous_parallel_programming_amd.solver import Context, Server, TCSolver

_RMAT = (0.57, 0.19, 0.19)  # quadrant weights a, b, c (d = 1 - a - b - c)
_PARTS = 4                  # parts of a split, as in the library's own split benchmark
_ELEMENTS = 1 << 26         # streamed ids expanded at a time by exact()
_EXACT_MOST = 3 << 30       # streamed ids above which exact() would take too long


def listed():
    return [
        # a small graph counted over and over (an ego network, a unit of a sweep): latency
        {"name": "count_er_1k", "op": "count", "kind": "er", "n": 1000, "edges": 16000},
        # a mid-size skewed graph, just past what one plain launch counts well
        {"name": "count_rmat_30k", "op": "count", "kind": "rmat", "n": 30011, "edges": 12 * 30011},
        # an ordinary skewed graph
        {"name": "count_rmat_s18", "op": "count", "kind": "rmat", "n": 1 << 18, "edges": 15 << 18},
        # the headline graph of the benchmark
        {"name": "count_rmat_s22", "op": "count", "kind": "rmat", "n": 1 << 22, "edges": 64000000},
        # a large flat graph (mesh- or random-like): short lists, many rows
        {"name": "count_er_2m", "op": "count", "kind": "er", "n": 2000003, "edges": 33000000},
        # one GPU's share of a graph split over four
        {"name": "partition_rmat_s21", "op": "partition", "kind": "rmat", "n": 1 << 21, "edges": 15 << 21},
        # the drop-in call on a small graph, in a program that holds a context
        {"name": "solver_er_16k", "op": "solver", "context": True, "kind": "er", "n": 16384, "edges": 250007},
        # the drop-in call on a large graph, as a program with one graph makes it
        {"name": "solver_rmat_s20", "op": "solver", "context": False, "kind": "rmat", "n": 1 << 20, "edges": 15 << 20},
        # every attribution at once: clustering coefficients, edge support, split accounting
        {"name": "local_rmat_s19", "op": "local", "edge_counts": True, "vertex_counts": True, "part_counts": True,
         "kind": "rmat", "n": 1 << 19, "edges": 15 << 19},
        # edge support (truss-like filters) with the split's sums
        {"name": "edges_rmat_s20", "op": "local", "edge_counts": True, "vertex_counts": False, "part_counts": True,
         "kind": "rmat", "n": 1 << 20, "edges": 15 << 20},
        # the benchmark's mix of graphs (256 to 65536 vertices, mean degree 4 to 64)
        {"name": "batch_mix_512", "op": "batch", "graphs": 512, "n_low": 256, "n_high": 65536},
        # the same mix arriving as requests, with the benchmark's 1% of large ones
        {"name": "serve_mix_256", "op": "serve", "graphs": 256, "n_low": 256, "n_high": 65536,
         "large": 2, "large_n": 1 << 20, "large_edges": 15 << 20},
    ]


def draw(rng):
    def log_int(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    op = rng.choice(["count", "count", "count", "partition", "solver", "local", "batch", "serve"])
    if op == "batch":
        low = log_int(64, 4096)
        return {"op": op, "graphs": log_int(16, 512), "n_low": low, "n_high": low + log_int(64, 60000)}
    if op == "serve":
        low = log_int(64, 4096)
        return {"op": op, "graphs": log_int(16, 256), "n_low": low, "n_high": low + log_int(64, 60000),
                "large": rng.choice([0, 1]), "large_n": log_int(1 << 17, 1 << 20),
                "large_edges": log_int(1 << 20, 1 << 24)}
    kind = rng.choice(["er", "rmat"])
    most = {"count": 64000000, "partition": 31000000, "solver": 15000000, "local": 7500000}[op]
    edges = log_int(4000, most)
    n = max(math.isqrt(16 * edges), int(edges / rng.uniform(3.0 if kind == "rmat" else 8.0, 24.0)))
    case = {"op": op, "kind": kind, "n": n, "edges": edges}
    if op == "solver":
        case["context"] = rng.choice([True, False])
    if op == "local":
        asked = rng.choice([(True, True, True), (True, False, False), (False, True, False), (False, False, True),
                            (True, False, True)])
        case.update(zip(("edge_counts", "vertex_counts", "part_counts"), asked))
    return case


# ---- graphs ------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed, stream):
    g = torch.Generator(device=_device())
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _rmat_pairs(levels, gen):
    """R-MAT endpoints; levels: per pair, how many quadrant choices it makes."""
    a, b, c = _RMAT
    src = torch.zeros(levels.numel(), dtype=torch.int64, device=levels.device)
    dst = torch.zeros_like(src)
    for level in range(int(levels.max()) if levels.numel() else 0):
        x = torch.rand(levels.numel(), generator=gen, device=levels.device)
        on = levels > level
        src = torch.where(on, 2 * src + (x >= a + b), src)
        dst = torch.where(on, 2 * dst + (((x >= a) & (x < a + b)) | (x >= a + b + c)), dst)
    return src, dst


def _distinct(n, src, dst):
    """The distinct undirected edges of these vertex pairs, as lo * n + hi."""
    keep = src != dst
    lo, hi = torch.minimum(src, dst)[keep], torch.maximum(src, dst)[keep]
    return torch.unique(lo * n + hi)


def _dag(n, pair):
    """(rowptr, colidx) of the graph of these distinct edges, oriented by (degree, id)."""
    lo, hi = pair // n, pair % n
    degree = torch.bincount(lo, minlength=n) + torch.bincount(hi, minlength=n)
    up = degree[lo] <= degree[hi]  # ids ascend, so a tie goes from lo to hi
    key = torch.sort(torch.where(up, lo * n + hi, hi * n + lo))[0]
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    torch.cumsum(torch.bincount(key // n, minlength=n), 0, out=rowptr[1:])
    return rowptr, key % n


def _single(kind, n, edges, seed, stream=0):
    gen = _generator(seed, stream)
    dev = _device()
    pair = torch.empty(0, dtype=torch.int64, device=dev)
    while pair.numel() < edges:  # duplicates and loops are drawn again
        count = edges + edges // 8 if pair.numel() == 0 else 2 * (edges - pair.numel()) + 1024
        if kind == "er":
            src = torch.randint(0, n, (count,), generator=gen, device=dev)
            dst = torch.randint(0, n, (count,), generator=gen, device=dev)
        else:
            src, dst = _rmat_pairs(torch.full((count,), max(1, (n - 1).bit_length()), device=dev), gen)
            inside = (src < n) & (dst < n)
            src, dst = src[inside], dst[inside]
        pair = torch.unique(torch.cat([pair, _distinct(n, src, dst)]))
    kept = torch.randperm(pair.numel(), generator=gen, device=dev)[:edges]
    return _dag(n, pair[kept])


def _mix(case, seed):
    """The benchmark's mix as one DAG over all vertices, and each graph's first
    vertex: sizes spread over their logarithm, mean degrees 4 to 64, Erdos-Renyi
    and R-MAT in turn."""
    dev = _device()
    count, low, high = case["graphs"], case["n_low"], case["n_high"]
    rng = np.random.RandomState(int(seed) % (1 << 32))
    n = np.exp(rng.uniform(math.log(low), math.log(high + 1), count)).astype(np.int64).clip(low, high)
    pairs = np.maximum(1, (n * rng.uniform(4.0, 64.0, count) / 2).astype(np.int64))
    first = np.concatenate([[0], np.cumsum(n)])
    which = torch.repeat_interleave(torch.arange(count, device=dev), torch.from_numpy(pairs).to(dev))
    size = torch.from_numpy(n).to(dev)[which]
    gen = _generator(seed, 1)
    u = (torch.rand(which.numel(), generator=gen, device=dev, dtype=torch.float64) * size).long()
    v = (torch.rand(which.numel(), generator=gen, device=dev, dtype=torch.float64) * size).long()
    scale = torch.tensor([int(x - 1).bit_length() for x in n], device=dev)[which]
    ru, rv = _rmat_pairs(torch.where(which % 2 == 1, scale, torch.zeros_like(scale)), gen)
    rmat = which % 2 == 1
    u, v = torch.where(rmat, ru, u), torch.where(rmat, rv, v)
    inside = (u < size) & (v < size)
    base = torch.from_numpy(first[:-1]).to(dev)[which]
    total = int(first[-1])
    rowptr, colidx = _dag(total, _distinct(total, (u + base)[inside], (v + base)[inside]))
    return rowptr, colidx, first


def _host(rowptr, colidx):
    return rowptr.cpu().numpy(), colidx.to(torch.int32).cpu().numpy()


def _split_mix(rowptr, colidx, first):
    rowptr, colidx = _host(rowptr, colidx)
    graphs = []
    for a, b in zip(first[:-1], first[1:]):
        e0, e1 = rowptr[a], rowptr[b]
        graphs.append(Graph.from_csr(rowptr[a:b + 1] - e0, colidx[e0:e1] - np.int32(a)))
    return graphs


def _bounds(n):
    return np.array([n * p // _PARTS for p in range(_PARTS + 1)], np.int32)


# ---- cases -------------------------------------------------------------------
_context = None


def _ctx():
    """The program's context: one for its whole life."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        graphs = _split_mix(*_mix(case, seed))
        return {"op": op, "batch": _ctx().batch(graphs)}
    if op == "serve":
        graphs = _split_mix(*_mix(case, seed))
        for k in range(case["large"]):  # spread among the small ones
            big = Graph.from_csr(*_host(*_single("rmat", case["large_n"], case["large_edges"], seed, 2 + k)))
            graphs.insert((k + 1) * len(graphs) // (case["large"] + 1), big)
        server = Server(_ctx(), hbm_budget=4 << 30, host_staging=512 << 20)
        return {"op": op, "graphs": graphs, "server": server}
    rowptr, colidx = _host(*_single(case["kind"], case["n"], case["edges"], seed))
    if op == "count":
        return {"op": op, "graph": _ctx().upload_arrays(rowptr, colidx)}
    if op == "local":
        return {"op": op, "graph": _ctx().upload_arrays(rowptr, colidx), "edges": case["edge_counts"],
                "vertices": case["vertex_counts"], "bounds": _bounds(case["n"]) if case["part_counts"] else None}
    g = Graph.from_csr(rowptr, colidx)
    if op == "partition":
        part = PartitionedGraph(g, _PARTS, balance="partner").halo_partition(0)
        return {"op": "count", "graph": _ctx().upload_partition(part)}
    return {"op": op, "host": g, "context": _ctx() if case["context"] else None}


def run(state):
    op = state["op"]
    if op == "count":
        return _ctx().count(state["graph"])[0]
    if op == "solver":
        return TCSolver(state["host"], ctx=state["context"])
    if op == "local":
        total, out = _ctx().count_local(state["graph"], edges=state["edges"], vertices=state["vertices"],
                                        bounds=state["bounds"])
        # counts are far below the sign bit: signed views of the same memory
        views = {k: v.view(np.int32 if v.dtype.itemsize == 4 else np.int64)
                 for k, v in out.items() if isinstance(v, np.ndarray)}
        return {"total": total, **views}
    if op == "batch":
        return state["batch"].count()[0].view(np.int64)
    server, graphs = state["server"], state["graphs"]
    counts = np.full(len(graphs), -1, np.int64)
    for tag, g in enumerate(graphs):
        server.submit(g, tag)
    got = 0
    while got < len(graphs):
        for r in server.poll(timeout_ms=1000):
            counts[r["tag"]] = r["count"] if r["status"] == 0 else -2
            got += 1
    return counts


def work(case):
    """Each DAG read once (8 bytes a row, 4 an edge) and each output written
    once."""
    if case["op"] in ("batch", "serve"):
        low, high = case["n_low"], case["n_high"]
        mean_n = (high - low) / math.log(high / low)  # mean of a log-uniform size
        rows, edges = case["graphs"] * mean_n, case["graphs"] * mean_n * 17
        if case["op"] == "serve":
            rows += case["large"] * case["large_n"]
            edges += case["large"] * case["large_edges"]
        return {"bytes": 8 * rows + 4 * edges + 8 * case["graphs"], "flops": 0}
    rows, edges = case["n"], case["edges"]
    read = 8 * (rows + 1) + 4 * edges
    if case["op"] == "partition":  # a quarter of the streamed work: its rows and the lists they reach
        return {"bytes": read / 2, "flops": 0}
    wrote = 8
    if case["op"] == "local":
        wrote += 4 * edges * case["edge_counts"] + 8 * rows * case["vertex_counts"] + 8 * _PARTS * case["part_counts"]
    return {"bytes": read + wrote, "flops": 0}


# ---- the same counts in plain torch ------------------------------------------
def _hits(rowptr, colidx, vertices=False):
    """Common out-neighbours of each edge's ends, and with ``vertices`` the
    triangles at each vertex; None when there is too much to do here."""
    n, m = rowptr.numel() - 1, colidx.numel()
    degree = rowptr[1:] - rowptr[:-1]
    src = torch.repeat_interleave(torch.arange(n, device=colidx.device), degree)
    key = src * n + colidx
    short = torch.where(degree[src] < degree[colidx], src, colidx)
    other = src + colidx - short
    end = torch.cumsum(degree[short], 0)
    if m and int(end[-1]) > _EXACT_MOST:
        return None
    hits = torch.zeros(m, dtype=torch.int64, device=colidx.device)
    at = torch.zeros(n, dtype=torch.int64, device=colidx.device)
    e0 = 0
    while e0 < m:
        begun = int(end[e0 - 1]) if e0 else 0
        e1 = max(e0 + 1, int(torch.searchsorted(end, begun + _ELEMENTS, right=True)))
        size = degree[short[e0:e1]]
        edge = torch.repeat_interleave(torch.arange(e0, e1, device=colidx.device), size)
        place = torch.arange(begun, begun + edge.numel(), device=colidx.device) - (end - degree[short])[edge]
        w = colidx[rowptr[short[edge]] + place]
        want = other[edge] * n + w
        found = key[torch.searchsorted(key, want).clamp_(max=m - 1)] == want
        edge, w = edge[found], w[found]
        hits += torch.bincount(edge, minlength=m)
        if vertices:
            for corner in (src[edge], colidx[edge], w):
                at += torch.bincount(corner, minlength=n)
        e0 = e1
    return src, degree, hits, at


def exact(case, seed):
    op = case["op"]
    if op in ("batch", "serve"):
        rowptr, colidx, first = _mix(case, seed)
        got = _hits(rowptr, colidx)
        if got is None:
            return None
        cut = torch.cat([torch.zeros(1, dtype=torch.int64, device=colidx.device), torch.cumsum(got[2], 0)])
        ends = cut[rowptr[torch.from_numpy(first).to(colidx.device)]]
        counts = (ends[1:] - ends[:-1]).cpu().tolist()
        if op == "serve":
            for k in range(case["large"]):
                big = _hits(*_single("rmat", case["large_n"], case["large_edges"], seed, 2 + k))
                if big is None:
                    return None
                counts.insert((k + 1) * len(counts) // (case["large"] + 1), int(big[2].sum()))
        return np.array(counts, np.int64)
    if op == "partition":
        return None  # which rows the part owns is the partitioner's choice
    rowptr, colidx = _single(case["kind"], case["n"], case["edges"], seed)
    got = _hits(rowptr, colidx, vertices=op == "local" and case["vertex_counts"])
    if got is None:
        return None
    src, degree, hits, at = got
    total = int(hits.sum())
    if op != "local":
        return total
    out = {"total": total}
    if case["edge_counts"]:
        out["edge_counts"] = hits.to(torch.int32).cpu().numpy()
    if case["vertex_counts"]:
        out["vertex_counts"] = at.cpu().numpy()
    if case["part_counts"]:
        # the part that computes edge (u, v): u's, unless v is elsewhere with the longer list
        cuts = torch.from_numpy(_bounds(case["n"])[1:-1].astype(np.int64)).to(colidx.device)
        pu, pv = torch.bucketize(src, cuts, right=True), torch.bucketize(colidx, cuts, right=True)
        part = torch.where((pu != pv) & (degree[src] < degree[colidx]), pv, pu)
        sums = torch.zeros(_PARTS, dtype=torch.int64, device=colidx.device)
        out["part_counts"] = sums.scatter_add_(0, part, hits).cpu().numpy()
    return out
