"""Core numbers from the persistent peeling kernel against a host peeling, at
the forms where a level, a cascade or the block's queue can go wrong."""

import numpy as np
import pytest

from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def _pairs(form):
    a = np.arange
    if form == "single":
        return 1, a(0), a(0)
    if form == "no_edges":
        return 257, a(0), a(0)
    if form == "path":  # one cascade through every vertex
        return 3000, a(2999), a(1, 3000)
    if form == "star":  # a hub of many steps of a wave
        return 5001, np.zeros(5000, np.int64), a(1, 5001)
    if form == "clique_gap":  # levels 1 and 299: the levels between are jumped
        i, j = np.triu_indices(300, 1)
        return 600, np.r_[i, a(299, 599)], np.r_[j, a(300, 600)]
    if form == "bipartite":  # equal hubs that leave together
        i, j = np.meshgrid(a(40), a(40, 2040))
        return 2040, i.ravel(), j.ravel()
    if form == "cycle_overflow":  # more vertices at one level than the queues hold
        return 1_300_000, a(1_300_000), (a(1_300_000) + 1) % 1_300_000
    g = gg.rmat(13, 8, 0.57, 0.19, 0.19, 5)
    src = np.repeat(np.arange(g.n), np.diff(g.off))
    return g.n, src, g.adj.astype(np.int64)


@pytest.mark.parametrize("form", ["single", "no_edges", "path", "star", "clique_gap", "bipartite",
                                  "cycle_overflow", "rmat"])
def test_core_numbers_match_host_peeling(form):
    n, u, v = _pairs(form)
    g = gg.csr_from_pairs(n, u, v)
    print("core numbers,", form, "n =", n, flush=True)
    G = scs.Graph.from_csr(g.off, g.adj)
    got = G.core()
    G.close()
    want = np.full(n, 2) if form == "cycle_overflow" else gg.core_numbers(g)
    assert np.array_equal(got, want)
