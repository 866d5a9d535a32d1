"""The search's adjacency scans over lists of much the same length, which one
lane each reads, beside uneven ones: a single wave must expand the oracle's
nodes on near-regular graphs around the lengths where the classes meet."""

import numpy as np
import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def near_regular(n, d, wide, seed):
    """A circulant graph of degree d, a tenth of its edges moved, whose first
    `wide` vertices have three times the degree."""
    rng = np.random.default_rng(seed)
    u = np.repeat(np.arange(n), d // 2)
    v = (u + np.tile(np.arange(1, d // 2 + 1), n)) % n
    move = rng.random(u.size) < 0.1
    v[move] = rng.integers(0, n, move.sum())
    hu = np.repeat(np.arange(wide), 2 * d)
    hv = rng.integers(0, n, hu.size)
    u, v = np.concatenate([u, hu]), np.concatenate([v, hv])
    return gg.csr_from_pairs(n, u[u != v], v[u != v])


@pytest.mark.parametrize("no_bitmaps", [0, 1])
@pytest.mark.parametrize("wide", [0, 3])
@pytest.mark.parametrize("n,d", [(127, 34), (128, 40), (700, 100), (700, 128), (900, 256), (1100, 500), (1300, 520)])
def test_even_lists_expand_the_oracles_nodes(n, d, wide, no_bitmaps):
    g = near_regular(n, d, wide, d)
    G, og = scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)
    qs = [(6, 12, 5, 0, 8), (5, 10, 0, 0, 8), (8, 24, 70, 1, 4)]
    for whole in (0, 2):
        print("n", n, "d", d, "wide", wide, "no_bitmaps", no_bitmaps, "whole", whole, flush=True)
        E = scs.Engine(G, deterministic=1, node_budget=60, limit_queries=4, whole_graph=whole,
                       no_lds_bitmaps=no_bitmaps)
        for r, q in zip(E.run(qs), qs):
            o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=60)
            assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), (n, d, whole, q)
        E.close()
    G.close()
