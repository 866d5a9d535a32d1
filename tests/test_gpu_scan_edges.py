"""The search's adjacency scans at the edges of their degree classes, and the
removal of most of R at once: a single wave must expand the oracle's nodes on
graphs whose large vertices have exactly those degrees."""

import numpy as np
import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def graph_with_degree(d, seed):
    """A dense group of 24 vertices, whose vertex 0 is widened to degree d and
    whose vertex 1 to about d / 2, over a sparse background that the rules
    remove in large batches."""
    rng = np.random.default_rng(seed)
    n = max(700, d + 200)
    i, j = np.triu_indices(24, 1)
    pick = rng.random(i.size) < 0.7
    us, vs = [i[pick], rng.integers(24, n, n)], [j[pick], rng.integers(24, n, n)]
    have = int((np.r_[i[pick], j[pick]] == 0).sum())
    for h, want in ((0, d - have), (1, d // 2)):
        far = rng.choice(np.arange(24, n), max(0, want), replace=False)
        us.append(np.full(far.size, h))
        vs.append(far)
    return gg.csr_from_pairs(n, np.concatenate(us), np.concatenate(vs))


@pytest.mark.parametrize("no_bitmaps", [0, 1])
@pytest.mark.parametrize("d", [32, 33, 64, 256, 512, 513, 1025])
def test_degree_class_edges_expand_the_oracles_nodes(d, no_bitmaps):
    g = graph_with_degree(d, d)
    assert g.degree[0] == d
    G, og = scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)
    qs = [(5, 9, 0, 0, 8), (6, 12, 5, 1, 4), (4, 10, 1, 0, 8), (5, 14, int(g.adj[g.off[0] + 20]), 0, 8)]
    for whole in (0, 2):
        print("degree", d, "no_bitmaps", no_bitmaps, "whole", whole, flush=True)
        E = scs.Engine(G, deterministic=1, node_budget=300, limit_queries=4, whole_graph=whole,
                       no_lds_bitmaps=no_bitmaps)
        for r, q in zip(E.run(qs), qs):
            o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=300)
            assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), (d, whole, q)
        E.close()
    G.close()
