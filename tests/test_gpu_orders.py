"""Graphs past 65535 vertices that are counted with codes, whatever their rows'
order: the share of edges that the codes cover is computed here from the
degrees, and the upload's bytes say that it kept them (and, for flat graphs, the
lists on lines)."""
import numpy as np
import pytest

import oracle
from hetegeneous_parallel_programming_amd import Graph

pytestmark = pytest.mark.gpu

ONCE = 1 | 8  # TC_CHECK_SHAPE | TC_UPLOAD_ONCE: neither codes nor lines for graphs of this size
TUNES = [dict(t_g8=0, t_g16=0, t_g32=0, t_wave=0), dict(t_g8=0, t_g16=0, t_g32=0, t_wave=1 << 30), {}]


def coded_share(rp, ci):
    """Share of the edges whose head's ids all have codes: those of the at most
    65535 vertices of highest degree, none below 16."""
    n, out = rp.size - 1, np.diff(rp)
    degree = out + np.bincount(ci, minlength=n)
    reach = np.bincount(np.minimum(degree, 16384), minlength=16385)[::-1].cumsum()[::-1]
    coded = degree >= max(16, int(np.argmax(reach <= 65535)))
    open_ids = np.bincount(np.repeat(np.arange(n), out), weights=~coded[ci], minlength=n)
    return float((open_ids[ci] == 0).mean())


def uneven(n, m, seed):
    """Edges between a vertex drawn evenly and one drawn towards a few hubs of
    any id: every vertex has some degree, lists are uneven in every order."""
    rng = np.random.default_rng(seed)
    hubs = rng.permutation(n)[(n * rng.random(m) ** 2.4).astype(np.int64)]
    return Graph.from_pairs(n, rng.integers(0, n, m).astype(np.int32), hubs.astype(np.int32))


@pytest.mark.parametrize("order", ["degree up", "id", "reversed", "degree down", "symmetric"])
def test_codes_in_rows_of_any_order(ctx, order):
    sym = uneven(66_000, 1_500_000, 3)
    rp, ci = sym.out_rowptr(), sym.out_colidx()
    deg = np.diff(rp)
    src = np.repeat(np.arange(rp.size - 1), deg)
    higher = (deg[src] > deg[ci]) | ((deg[src] == deg[ci]) & (src > ci))
    keep = {"id": src < ci, "reversed": src > ci, "symmetric": np.ones(ci.size, bool), "degree down": higher,
            "degree up": ~higher}[order]
    n, ci = rp.size - 1, np.ascontiguousarray(ci[keep])
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src[keep], minlength=n), out=rp[1:])
    out = np.diff(rp)
    uneven_lists = (out.astype(float) ** 2).sum() * (out > 0).sum() >= 2.0 * float(ci.size) ** 2
    assert uneven_lists == (order != "degree up") and coded_share(rp, ci) > 0.5
    want = oracle.tc_count(rp, ci)
    dg = ctx.upload_arrays(rp, ci)
    spare = dg.info()["bytes"] - ctx.upload_arrays(rp, ci, check=ONCE).info()["bytes"]
    # codes, a mark a row and a part an id; or, lists being even, lists on lines
    assert spare == (2 * (2 * ci.size + 4096) + n + ci.size if uneven_lists else 4 * (2 * ci.size + 4))
    default = ctx.tune
    try:
        for t in TUNES:
            ctx.tune = t
            assert [ctx.count_binned(dg)[0] for _ in range(2)] == [want] * 2
            ctx.tune = default
    finally:
        ctx.tune = default
    total, res = ctx.count_local(dg, bounds=[0, n // 3, n])
    assert total == want and (res["vertex_counts"] == oracle.tc_per_vertex(rp, ci)).all()
    assert ctx.count_binned(dg)[0] == want  # after the local rebuild


def test_codes_of_few_edges_are_not_kept(ctx):
    # a symmetric R-MAT graph: one edge in eight leads to a list of codes only
    sym = Graph.rmat(80_000, 6, 7)
    rp, ci = sym.out_rowptr(), sym.out_colidx()
    assert coded_share(rp, ci) < 0.2
    dg = ctx.upload_arrays(rp, ci)
    assert dg.info()["bytes"] == ctx.upload_arrays(rp, ci, check=ONCE).info()["bytes"]
    want = oracle.tc_count(rp, ci)
    assert [ctx.count_binned(dg)[0] for _ in range(2)] == [want] * 2
    total, res = ctx.count_local(dg, vertices=False)
    assert total == want and ctx.count_binned(dg)[0] == want
    flat = Graph.er(100_003, 80, 5).oriented()  # lists of 64 ids and more, but even ones
    rp, ci = flat.out_rowptr(), flat.out_colidx()
    assert np.diff(rp).max() >= 64
    dg = ctx.upload(flat)
    assert dg.info()["bytes"] - ctx.upload(flat, check=ONCE).info()["bytes"] == 4 * (2 * ci.size + 4)
    want = oracle.tc_count(rp, ci)
    assert [ctx.count_binned(dg)[0] for _ in range(2)] == [want] * 2
    total, res = ctx.count_local(dg)
    assert total == want and (res["vertex_counts"] == oracle.tc_per_vertex(rp, ci)).all()
