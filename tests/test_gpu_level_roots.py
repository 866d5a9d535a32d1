"""A level's root grown from the one before it: queries whose search descends
through many levels, with the status in LDS bitmaps and in device memory, on
local graphs and the resident one, in time slices so short that levels change
across epochs (a wave's root bound is then read back from its saved state)."""

import numpy as np
import pytest

from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL, OracleGraph
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def nested_cores(seed):
    """Groups of 24 to 60 vertices of rising density that share vertices, over a
    sparse background: core numbers from 2 to about 20, so that a level's bound
    lets a few dozen vertices join."""
    rng = np.random.default_rng(seed)
    n, us, vs, at = 900, [rng.integers(0, 900, 2500)], [rng.integers(0, 900, 2500)], 0
    for size, p in ((60, 0.18), (50, 0.3), (40, 0.45), (32, 0.6), (24, 0.85)):
        i, j = np.triu_indices(size, 1)
        pick = rng.random(i.size) < p
        us.append(at + i[pick])
        vs.append(at + j[pick])
        at += size - 12
    u, v = np.concatenate(us), np.concatenate(vs)
    return gg.csr_from_pairs(n, u[u != v], v[u != v])


@pytest.fixture(scope="module")
def graph():
    g = nested_cores(1)
    return scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj)


def _queries(og):
    core = og.core()
    by = np.argsort(-core.astype(np.int64), kind="stable")
    # far above what a set of h vertices around q can reach: the first levels fail
    return [(3, 8, int(by[0]), 0, 8), (4, 12, int(by[30]), 0, 8), (5, 14, int(by[60]), 0, 4),
            (3, 10, int(by[120]), 0, 8), (2, 6, int(by[400]), 0, 8)]


@pytest.mark.parametrize("slice_us", [200_000, 300])
@pytest.mark.parametrize("whole", [0, 2])
@pytest.mark.parametrize("no_bitmaps", [0, 1])
def test_descending_levels_expand_the_oracles_nodes(graph, no_bitmaps, whole, slice_us):
    G, og = graph
    qs = _queries(og)
    want = [og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=400) for q in qs]
    # levels descend one by one from min(core, h - 1)
    core = og.core()
    assert sum(min(int(core[q[2]]), q[1] - 1) - o["kl"] for q, o in zip(qs, want)) >= 10
    print("no_bitmaps", no_bitmaps, "whole", whole, "slice", slice_us, flush=True)
    E = scs.Engine(G, deterministic=1, node_budget=400, limit_queries=8, whole_graph=whole,
                   no_lds_bitmaps=no_bitmaps, time_slice_us=slice_us)
    res = E.run(qs)
    if slice_us < 1000:
        # several epochs per query, so some of its levels began in another one
        assert E.stats()["epochs"] > 4 * len(qs)
    E.close()
    for r, o, q in zip(res, want, qs):
        assert (r.kl, r.status, r.nodes) == (o["kl"], o["status"], o["nodes"]), q


@pytest.mark.parametrize("slice_us", [200_000, 300])
def test_descending_levels_with_many_waves(graph, slice_us):
    """The wave that ends a level need not be the one that built its root."""
    G, og = graph
    qs = _queries(og)
    E = scs.Engine(G, limit_queries=8, time_slice_us=slice_us)
    res = E.run(qs)
    E.close()
    for r, q in zip(res, qs):
        o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=2_000_000)
        assert r.kl == o["kl"] and r.status == o["status"], q
