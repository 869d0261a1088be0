"""The count's tile queues and the lists on cache lines against the CPU oracle:
grids around the 8 XCDs and around the number of tiles, single graphs and
batches; flat graphs whose lists are copied to lines, with owned-row masks,
partitions and the local rebuild."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import oracle  # noqa: E402

from hetegeneous_parallel_programming_amd import Graph  # noqa: E402
from hetegeneous_parallel_programming_amd.graph import PartitionedGraph  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from hetegeneous_parallel_programming_amd.solver import Context

    with Context(0) as c:
        yield c


def arrays(g):
    return g.out_rowptr(), g.out_colidx()


@pytest.mark.parametrize("grid", [1, 2, 7, 8, 9, 15, 16, 17, 63, 64, 65, 500, 4099])
def test_grids(ctx, grid):
    # bins of a few to a few thousand tiles: fewer tiles than workgroups, one
    # each, a few in turn, and queues that every XCD ends on another's eighth
    graphs = [Graph.rmat(n, 12, n).oriented() for n in (9, 300, 4000, 30011)] + [Graph.er(9000, 24, 1).oriented()]
    big = Graph.rmat(140_000, 8, 3).oriented()
    want = [oracle.tc_count(*arrays(g)) for g in graphs]
    uploads = [ctx.upload(g) for g in graphs] + [ctx.upload(big)]
    b = ctx.batch(graphs)
    default = ctx.tune
    try:
        for t in ({}, dict(t_g8=0, t_g16=40, t_g32=160, t_wave=640)):
            ctx.tune = dict(t, grid=grid)
            got = [[ctx.count_binned(u)[0] for u in uploads] for _ in range(2)]
            assert got == [want + [oracle.tc_count(*arrays(big))]] * 2
            assert [b.count()[0].tolist() for _ in range(2)] == [want] * 2
            assert ctx.count_local(uploads[-1])[0] == got[0][-1]
            ctx.tune = default
    finally:
        ctx.tune = default


def flat(n, lo, hi, seed):
    """A DAG of rows of lo..hi ids, each near above its row (so that lists
    meet)."""
    rng = np.random.default_rng(seed)
    length = rng.integers(lo, hi + 1, n)
    reach = max(hi + 1, n // 1000)
    offs = np.sort(rng.integers(1, reach, (n, hi)), axis=1)
    keep = (np.arange(hi) < length[:, None]) & (np.diff(offs, axis=1, prepend=0) > 0)
    ids = np.arange(n)[:, None] + offs
    keep &= ids < n
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(keep.sum(1), out=rp[1:])
    return rp, np.ascontiguousarray(ids[keep].astype(np.int32))


@pytest.mark.parametrize("n,lo,hi", [(66_000, 14, 30), (70_001, 0, 63), (300_000, 0, 12), (140_000, 8, 33)])
def test_lists_on_lines(ctx, n, lo, hi):
    rp, ci = flat(n, lo, hi, n)
    assert rp[-1] >= 1 << 20 and np.diff(rp).max() < 64  # such a graph's lists go to lines
    want = oracle.tc_count(rp, ci)
    dg = ctx.upload_arrays(rp, ci)
    assert [ctx.count_binned(dg)[0] for _ in range(2)] + [ctx.count_plain(dg)[0]] == [want] * 3
    total, out = ctx.count_local(dg, bounds=[0, n // 3, n])
    assert total == want and (out["vertex_counts"] == oracle.tc_per_vertex(rp, ci)).all()
    assert ctx.count_binned(dg)[0] == want  # after the local rebuild
    assert ctx.count_noalloc(dg)[0] == want


def test_lines_of_owned_rows_and_partitions(ctx):
    g = Graph.er(90_001, 30, 4).oriented()
    rp, ci = arrays(g)
    assert rp[-1] >= 1 << 20 and np.diff(rp).max() < 64
    owned = (np.arange(90_001) % 3 == 1).astype(np.uint8)
    dg = ctx.upload(g, owned=owned)
    want = oracle.tc_count_rows(rp, ci, np.flatnonzero(owned).astype(np.int32))
    assert ctx.count_binned(dg)[0] == want and ctx.count_binned(dg)[0] == want
    pg = PartitionedGraph(g, 2, balance="partner")
    parts = [ctx.count_binned(ctx.upload_partition(pg.halo_partition(i)))[0] for i in range(2)]
    assert sum(parts) == oracle.tc_count(rp, ci)


@pytest.mark.parametrize("m", [(1 << 21) - 1, 1 << 21, (1 << 21) + 1, (1 << 22) + 4099, (5 << 20) + 3])
def test_large_edge_counts_reach_the_host(ctx, m):
    # outputs around 8 MB and around the copies' chunks: triples of rows with
    # three edges, four in five of them a triangle (only its first edge's ends
    # share an out-neighbour), then one edge a row
    k = m // 3 - 1
    i = np.arange(k)
    tri = i % 5 != 0
    src = np.stack([3 * i, 3 * i, 3 * i + 1], 1)
    dst = np.stack([np.where(tri, 3 * i + 1, 3 * i + 2), np.where(tri, 3 * i + 2, 3 * i + 3), 3 * i + 2], 1)
    rest = m - 3 * k
    n = 3 * k + rest + 1
    src = np.concatenate([src.ravel(), 3 * k + np.arange(rest)])
    ci = np.concatenate([dst.ravel(), 3 * k + 1 + np.arange(rest)]).astype(np.int32)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src, minlength=n), out=rp[1:])
    want = np.zeros(m, np.uint32)
    want[3 * i[tri]] = 1
    dg = ctx.upload_arrays(rp, ci)
    for _ in range(2):
        total, out = ctx.count_local(dg, vertices=False)
        assert total == tri.sum() and (out["edge_counts"] == want).all()
