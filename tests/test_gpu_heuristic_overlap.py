"""An engine that admits through the GPU heuristic computes the bounds beside its
search epoch, not after it."""

import numpy as np
import pytest

from scs_amd import configs, scs

pytestmark = pytest.mark.gpu

SLICE_US = 200_000


def test_bounds_come_while_the_epoch_runs():
    g = configs.graph("C1")
    G = scs.Graph.from_csr(g.off, g.adj)
    by_core = [int(v) for v in np.argsort(-G.core().astype(np.int64), kind="stable")]
    E = scs.Engine(G, limit_queries=128, waves_per_cu=4, gpu_heuristic=1, time_slice_us=SLICE_US)
    for v in by_core[:60]:  # large h: none of these ends in a few slices
        E.submit(20, 60, v)
    E.step()
    E.step()
    took = []
    for k in range(3):
        for v in by_core[60 + 4 * k:64 + 4 * k]:
            E.submit(20, 60, v)
        h0, e0 = E.stats()["heu_us"], E.stats()["engine_us"]
        E.step()
        s = E.stats()
        assert s["engine_us"] - e0 > 0.9 * SLICE_US  # an epoch ran all along
        took.append(s["heu_us"] - h0)
    print("heuristic beside an epoch, us:", took, flush=True)
    E.close()
    G.close()
    assert max(took) < SLICE_US / 2
