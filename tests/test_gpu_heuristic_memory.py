"""The GPU heuristic where its workspace (some 200 bytes per vertex and query at
the largest h) is not there for a whole call: the call goes in parts, with the
same bounds."""

import ctypes as C

import numpy as np
import pytest

from scs_amd import graphgen as gg, scs
from tests.test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def test_a_call_beside_a_full_device():
    g = gg.chung_lu(200_000, 400_000, 2.5, 500, 4)
    G = scs.Graph.from_csr(g.off, g.adj)
    by_deg = np.argsort(-g.degree, kind="stable")
    qs = [(3, 1000 if i == 5 else 12, int(by_deg[7 * i])) for i in range(64)]
    want = scs.heuristic_gpu(G, qs)
    hip = _hip()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    # 64 queries want 2.6 GB
    rest = 1500 << 20
    assert free.value > rest
    held = C.c_void_p()
    print("heuristic with 1.5 GB free", flush=True)
    assert hip.hipMalloc(C.byref(held), free.value - rest) == 0
    try:
        got = scs.heuristic_gpu(G, qs)
    finally:
        hip.hipFree(held)
    G.close()
    for (kl, H), (kl2, H2) in zip(want, got):
        assert kl == kl2 and list(H) == list(H2)
