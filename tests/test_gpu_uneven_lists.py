"""The search's adjacency scans at the lines of its degree classes among uneven
lists: above 128 entries a list is read by the whole wave, and no list is read by
one lane beyond 32 unless those beside it are as long."""

import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph
from scs_amd import scs
from tests.test_gpu_scan_edges import graph_with_degree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("no_bitmaps", [0, 1])
@pytest.mark.parametrize("d", [127, 128, 129, 130, 258, 384])
def test_uneven_lists_expand_the_oracles_nodes(d, no_bitmaps):
    g = graph_with_degree(d, d)
    assert g.degree[0] == d
    G, og = scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)
    qs = [(5, 9, 0, 0, 8), (6, 12, 5, 1, 4), (4, 10, 1, 0, 8),
          (5, 14, int(g.adj[g.off[0] + 20]), 0, 8)]
    for whole in (0, 2):
        print("degree", d, "no_bitmaps", no_bitmaps, "whole", whole, flush=True)
        E = scs.Engine(G, deterministic=1, node_budget=300, limit_queries=4, whole_graph=whole,
                       no_lds_bitmaps=no_bitmaps)
        for r, q in zip(E.run(qs), qs):
            o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=300)
            assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), (d, whole, q)
        E.close()
    G.close()
