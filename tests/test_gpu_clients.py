"""Several clients of one server submit requests around the sizes at which a
copy takes more threads; every count is the oracle's."""
import threading

import pytest

import oracle
from hetegeneous_parallel_programming_amd import Graph
from hetegeneous_parallel_programming_amd.solver import Server

pytestmark = pytest.mark.gpu


def test_counts_of_concurrent_requests(ctx):
    # 0.1 to 19 MB a request
    graphs = [Graph.rmat(n, ef, n + ef).oriented() for n, ef in
              ((2000, 8), (40_000, 6), (40_000, 14), (70_000, 24), (200_000, 10), (400_000, 12))]
    want = [oracle.tc_count(g.out_rowptr(), g.out_colidx()) for g in graphs]
    clients, errors = 6, []
    server = Server(ctx, hbm_budget=4 << 30, host_staging=64 << 20)
    try:
        def client(c):
            try:
                for i in range(2 * len(graphs)):
                    k = (c + i) % len(graphs)
                    server.submit(graphs[k], (c * 2 * len(graphs) + i) * len(graphs) + k)
            except Exception as e:  # noqa: BLE001
                errors.append(e)

        threads = [threading.Thread(target=client, args=(c,)) for c in range(clients)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
        assert not errors
        got = []
        while len(got) < clients * 2 * len(graphs):
            new = server.poll(timeout_ms=5000)
            assert new
            got += new
        assert all(r["status"] == 0 and r["count"] == want[r["tag"] % len(graphs)] for r in got)
    finally:
        server.close()
