"""Compacted batches of which some queries go back to the queue after their
degrees were counted, because the arena does not hold every local adjacency:
the others' rows of local ids keep the columns of the whole batch, in both forms
of the adjacency pass (up to 16 queries, and more)."""

import numpy as np
import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph, ubd_host
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def granule(b):
    return max(256, (b + 255) // 256 * 256)


@pytest.mark.parametrize("share", [0.35, 0.8])
@pytest.mark.parametrize("cnt", [9, 16, 24, 60])
def test_queries_sent_back_between_the_passes(cnt, share):
    rng = np.random.default_rng(cnt)
    n = 3000
    hub = rng.choice(np.arange(1, n), 700, replace=False)
    g = gg.csr_from_pairs(n, np.r_[rng.integers(0, n, 12000), np.zeros(700, np.int64)],
                          np.r_[rng.integers(0, n, 12000), hub])
    G, og = scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)
    qs, a_sum, b_len = [], 0, []
    core = og.core()
    for v in rng.choice(np.flatnonzero(core > 3), cnt, replace=False):
        h = int(rng.integers(6, 12))
        p = og.preprocess(int(v), 0, ubd_host(0, h))
        qs.append((4, h, int(v), 0, 8))
        a_sum += granule(4 * (4 * p["K"] + 1))
        b_len.append(granule(4 * max(1, p["adj"].size)))
    # every query's first block fits, and a share of the adjacencies
    budget = a_sum + int(share * sum(b_len)) // 256 * 256
    assert min(b_len) <= budget - a_sum < sum(b_len)
    print("batch of", cnt, "arena", budget, "blocks", a_sum, sum(b_len), flush=True)
    E = scs.Engine(G, deterministic=1, node_budget=15, limit_queries=64, mem_budget=budget,
                   whole_graph=0)
    res = E.run(qs)
    assert E.stats()["prep_batches"] >= 2  # some came a second time
    for r, q in zip(res, qs):
        o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=15)
        assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), q
    E.close()
    G.close()
