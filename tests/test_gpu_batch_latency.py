"""Small queries in a batch that fills the chip: their tasks must not wait in the
pool behind tasks of long searches that no wave is free to take."""

import json
import os

import pytest

from scs_amd import configs, scs

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_small_queries_of_a_full_batch_end_early():
    """100 queries, most of them with hundreds of thousands of nodes: those the
    oracle proves within 300 nodes are through in 10 time slices of 50 ms (some
    250 nodes of one wave; 7 or 8 measured, 21 when the pool may fill up)."""
    rows = json.load(open(os.path.join(ROOT, "tests", "golden", "golden.json")))["C1"]
    small = [i for i, r in enumerate(rows) if r["status"] != "CAPPED" and r["nodes"] <= 300]
    assert len(small) >= 10
    g = configs.graph("C1")
    G = scs.Graph.from_csr(g.off, g.adj)
    E = scs.Engine(G, waves_per_cu=4, limit_queries=256, time_slice_us=50_000, copy_limit=0.5,
                   admit_per_step=256, node_budget=500_000)
    E.set_model(scs.Model.load(os.path.join(ROOT, "models", "branching_c1.npz")), True)
    for i, r in enumerate(rows):
        E.submit(*r["query"], tag=i)
    kl = {}
    while E.stats()["epochs"] < 10:
        E.step()
        for r in E.poll():
            kl[r.tag] = r.kl
    E.close()
    G.close()
    print("done in 10 epochs:", len(kl), flush=True)
    assert [i for i in small if i not in kl] == []
    assert all(kl[i] == rows[i]["kl"] for i in small)
