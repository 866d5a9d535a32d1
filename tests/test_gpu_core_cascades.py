"""Core numbers where a cascade overflows the blocks' queues: vertices that one
block's cascade queues beyond its 4,096 entries go through the list in device
memory to whichever block shares it out next, and may overflow there again."""

import numpy as np
import pytest

from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def _pairs(form):
    a = np.arange
    if form == "path":
        # peeled from both ends, one vertex after another: 25,000 steps each,
        # so each end's cascade outgrows a queue six times in a row
        return 50_000, a(49_999), a(1, 50_000)
    if form == "paths_on_a_clique":
        # 40 paths of 5,000 that hang on a clique of 41: one end each, level 1
        # takes them all and level 40 the clique
        i, j = np.triu_indices(41, 1)
        chain = 41 + a(200_000).reshape(40, 5000)
        return (200_041, np.r_[i, chain[:, :-1].ravel(), chain[:, -1]],
                np.r_[j, chain[:, 1:].ravel(), a(40)])
    # a hub's 20,000 leaves each carry a leaf of their own: the leaves' leaves go
    # first, then all of the hub's leaves, from many blocks, and the hub
    return (40_001, np.r_[np.zeros(20_000, np.int64), a(1, 20_001)],
            np.r_[a(1, 20_001), a(20_001, 40_001)])


@pytest.mark.parametrize("form", ["path", "paths_on_a_clique", "two_layer_star"])
def test_cascades_beyond_the_queues(form):
    n, u, v = _pairs(form)
    g = gg.csr_from_pairs(n, u, v)
    print("core numbers,", form, "n =", n, flush=True)
    G = scs.Graph.from_csr(g.off, g.adj)
    got = G.core()
    G.close()
    want = np.ones(n, np.uint32)
    if form == "paths_on_a_clique":
        want[:41] = 40
    assert np.array_equal(got, want)
