"""The GPU heuristic where its forms change: members' bits in 1, 2, 4 and more
than 4 words (h up to 64, 128, 256 and above), a neighbourhood whose block keys
exceed the LDS (more than 4,096 members), and one engine's workspace used by
batches of different sizes."""

import numpy as np
import pytest

from oracle.oracle import OracleGraph
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    """7,000 vertices: 40,000 random edges, a hub of degree about 5,000 and a
    dense group of 400 in which the constructions can grow large."""
    rng = np.random.default_rng(11)
    n = 7000
    i, j = np.triu_indices(400, 1)
    pick = rng.random(i.size) < 0.3
    hub = rng.choice(np.arange(500, n), 5000, replace=False)
    g = gg.csr_from_pairs(n, np.concatenate([rng.integers(0, n, 40000), i[pick], np.full(5000, 450)]),
                          np.concatenate([rng.integers(0, n, 40000), j[pick], hub]))
    return scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj), g


@pytest.mark.parametrize("h", [1, 2, 63, 64, 65, 128, 129, 192, 256, 257, 400, 1000])
def test_sizes_of_h(graph, h):
    G, og, g = graph
    assert g.degree[450] > 4096
    qs = [(max(1, h // 2), h, q) for q in (0, 7, 399, 450, 6999)] + [(0, h, 5), (h, h, 3)]
    print("h", h, flush=True)
    for (l, hh, q), (kl, H) in zip(qs, scs.heuristic_gpu(G, qs)):
        ref_kl, ref_H = og.heuristic(0, l, hh, q)
        assert kl == ref_kl, (l, hh, q)
        if kl > 0:
            assert list(H) == list(ref_H)[:scs.MAX_H], (l, hh, q)


def test_one_workspace_for_batches_of_different_h(graph):
    G, og, _ = graph
    E = scs.Engine(G, deterministic=1, node_budget=1, limit_queries=8, gpu_heuristic=1)
    for h in (20, 300, 40, 130, 20):
        qs = [(max(2, h // 2), h, q, 1, 8) for q in (1, 450, 6000)]
        for r in E.run(qs):
            assert r.heu_kl == og.heuristic(0, r.l, r.h, r.q)[0], (h, r.q)
    E.close()
