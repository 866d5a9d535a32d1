"""Batched preprocessing at the edges of its passes: adjacency units of exactly
256 entries and hubs of several, batches on both sides of the few-query form of
the adjacency pass, queries sent back for want of arena between the passes, and
whole-graph and compacted queries in one batch."""

import ctypes as C

import numpy as np
import pytest

from oracle.oracle import OracleGraph, ubd_host
from scs_amd import graphgen as gg, scs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(3)
    n = 9000  # more units than one generation of waves
    us, vs = [rng.integers(4, n, 40000)], [rng.integers(4, n, 40000)]
    for h, d in ((0, 256), (1, 257), (2, 1024), (3, 5000)):
        us.append(np.full(d, h))
        vs.append(rng.choice(np.arange(4, n), d, replace=False))
    g = gg.csr_from_pairs(n, np.concatenate(us), np.concatenate(vs))
    return scs.Graph.from_csr(g.off, g.adj), OracleGraph.from_csr(g.n, g.off, g.adj), g


def _queries(og, cnt, seed):
    core = og.core()
    rng = np.random.default_rng(seed)
    q = rng.integers(0, og.n, cnt).astype(np.uint32)
    q[:min(cnt, 4)] = np.arange(min(cnt, 4))
    kl0 = np.array([int(rng.integers(0, max(1, int(core[v])))) for v in q], np.uint32)
    ubd = np.array([ubd_host(int(k), int(rng.integers(2, 40))) for k in kl0], np.uint32)
    return q, kl0, ubd


@pytest.mark.parametrize("cnt", [1, 7, 8, 9, 16, 17, 40, 64])
def test_local_graphs_of_batches(graph, cnt):
    G, og, g = graph
    assert list(g.degree[:3]) == [256, 257, 1024]
    E = scs.Engine(G, limit_queries=64, waves_per_cu=1)
    q, kl0, ubd = _queries(og, cnt, cnt)
    n, cap = og.n, int(g.off[-1])
    K, nnz = np.zeros(cnt, np.uint32), np.zeros(cnt, np.uint64)
    kept, dist = np.zeros((cnt, n), np.uint32), np.zeros((cnt, n), np.uint32)
    loff, ladj = np.zeros((cnt, n + 1), np.uint32), np.zeros((cnt, cap), np.uint32)
    f = scs.lib().scs_prep_probe_many
    f.argtypes = [C.c_void_p, C.c_uint32] + [C.c_void_p] * 8 + [C.c_uint32, C.c_void_p, C.c_uint64]
    print("batch of", cnt, flush=True)
    p = [a.ctypes.data for a in (q, kl0, ubd, K, nnz, kept, loff, dist)]
    assert f(E._h, cnt, *p, n, ladj.ctypes.data, cap) == 0
    E.close()
    for i in range(cnt):
        ref = og.preprocess(int(q[i]), int(kl0[i]), int(ubd[i]))
        k, z = int(K[i]), int(nnz[i])
        assert k == ref["K"] and z == ref["adj"].size, i
        assert np.array_equal(kept[i, :k], ref["kept"]) and np.array_equal(dist[i, :k], ref["dist"])
        assert np.array_equal(loff[i, :k + 1], ref["off"]) and np.array_equal(ladj[i, :z], ref["adj"])


@pytest.mark.parametrize("mem", [2 << 20, 64 << 20])
def test_mixed_batch_expands_the_oracles_nodes(graph, mem):
    """whole_graph=1 sends some queries of the batch to the resident graph and
    compacts the others; in 2 MB of arena not all fit at once, so some go back
    to the queue after their degrees were counted."""
    from oracle.oracle import FLAG_LEVELS, FLAG_PAIR, FLAGS_ALL
    G, og, _ = graph
    rng = np.random.default_rng(5)
    core = og.core()
    qs = []
    for v in rng.integers(0, og.n, 24):
        l = int(rng.integers(2, 6))
        qs.append((l, l + int(rng.integers(1, 6)), int(v), int(core[v] > 4), 8))
    E = scs.Engine(G, deterministic=1, node_budget=20, limit_queries=32, mem_budget=mem)
    for r, q in zip(E.run(qs), qs):
        o = og.solve(*q, flags=FLAGS_ALL | FLAG_LEVELS | FLAG_PAIR, node_cap=20)
        assert r.kl == o["kl"] and r.nodes == o["nodes"], q
    E.close()
