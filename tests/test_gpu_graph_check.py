"""scs_graph_create's device validation: one defect of each kind, in a short
row, in a hub's row, in the first and in the last entry, is SCS_EINVAL, and the
sound graph is accepted with its offsets, ids and core numbers."""

import numpy as np
import pytest

from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


def _graph():
    rng = np.random.default_rng(2)
    n = 3000
    hub = rng.choice(np.arange(1, n), 900, replace=False)
    return gg.csr_from_pairs(n, np.r_[rng.integers(0, n, 9000), np.zeros(900, np.int64)],
                             np.r_[rng.integers(0, n, 9000), hub])


def test_sound_graph_is_accepted():
    g = _graph()
    G = scs.Graph.from_csr(g.off, g.adj)
    off, adj = G.csr()
    assert np.array_equal(off, g.off) and np.array_equal(adj, g.adj)
    assert G.dmax == g.degree.max() and np.array_equal(G.core(), gg.core_numbers(g))
    G.close()


@pytest.mark.parametrize("row", ["hub", "short", "last"])
@pytest.mark.parametrize("kind", ["above_n", "negative", "self_loop", "duplicate", "unsorted",
                                  "one_way", "both_one_way"])
def test_one_defect_is_refused(kind, row):
    g = _graph()
    adj, deg = g.adj.copy(), g.degree
    v = {"hub": 0, "short": int(np.flatnonzero(deg == 4)[7]),
         "last": int(np.flatnonzero(deg >= 3)[-1])}[row]
    b, e = int(g.off[v]), int(g.off[v + 1])
    row_ids = set(adj[b:e].tolist())
    if kind == "above_n":
        adj[e - 1] = g.n
    elif kind == "negative":
        adj[b] = -1
    elif kind == "self_loop":
        adj[b] = v
    elif kind == "duplicate":
        adj[b + 1] = adj[b]
    elif kind == "unsorted":
        adj[b], adj[b + 1] = adj[b + 1], adj[b]
    else:
        # another neighbour in the same place of the order: the old one's entry
        # is left without its mirror, and the new one has none
        for j in range(b, e):
            lo = int(adj[j - 1]) + 1 if j > b else 0
            hi = int(adj[j + 1]) if j + 1 < e else g.n
            new = [x for x in range(lo, hi) if x != v and x not in row_ids]
            if new:
                adj[j] = new[0]
                if kind == "one_way":
                    break
    with pytest.raises(scs.SCSError) as err:
        scs.Graph.from_csr(g.off, adj)
    assert err.value.code == -1
