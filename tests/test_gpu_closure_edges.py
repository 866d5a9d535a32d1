"""The rule 1/2 closure where it looks at all of R instead of the removed
vertices' lists, in id order or in R's order, at the edges of its steps: a
single wave must expand the oracle's nodes."""

import numpy as np
import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def two_part_graph(n, dense, seed):
    """n vertices; a share `dense` of them has 24 neighbours of its own on
    average (R beside the removed lists is small), the rest two."""
    rng = np.random.default_rng(seed)
    k = max(20, int(n * dense))
    us = [rng.integers(0, k, 12 * k), rng.integers(0, n, 2 * n)]
    vs = [rng.integers(0, k, 12 * k), rng.integers(0, n, 2 * n)]
    u, v = np.concatenate(us), np.concatenate(vs)
    return gg.csr_from_pairs(n, u[u != v], v[u != v])


@pytest.mark.parametrize("dense", [0.2, 0.5, 1.0])
@pytest.mark.parametrize("n", [63, 511, 512, 513, 1025])
def test_closure_over_all_of_r_expands_the_oracles_nodes(n, dense):
    g = two_part_graph(n, dense, n)
    G, og = scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)
    qs = [(6, 12, 0, 0, 8), (4, 9, 1, 0, 8), (8, 20, 2, 1, 4)]
    for whole in (0, 2):
        print("n", n, "dense", dense, "whole", whole, flush=True)
        E = scs.Engine(G, deterministic=1, node_budget=200, limit_queries=4, whole_graph=whole)
        full = E.stats()["full_scans"]
        for r, q in zip(E.run(qs), qs):
            o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=200)
            assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), (n, dense, whole, q)
        assert E.stats()["full_scans"] > full
        E.close()
    G.close()
