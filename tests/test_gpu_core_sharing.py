"""Core numbers on a GPU that is not the call's alone: more blocks than find room
(those that come late take no part)."""

import ctypes as C

import numpy as np
import pytest

from scs_amd import graphgen as gg, scs
from tests.test_zz_no_alloc import DevBuf, _hip

pytestmark = pytest.mark.gpu


class Peel:
    """The library's core_peel on a device-resident graph with its own working
    memory."""

    def __init__(self, hip, n, avg, seed):
        g = gg.chung_lu(n, n * avg // 2, 2.5, 400, seed)
        self.hip, self.n, self.want = hip, g.n, gg.core_numbers(g)
        off, adj = np.ascontiguousarray(g.off, np.int64), np.ascontiguousarray(g.adj, np.int32)
        self.off, self.adj = DevBuf(hip, off.nbytes), DevBuf(hip, adj.nbytes)
        self.off.put(off)
        self.adj.put(adj)
        words = scs.lib().scs_core_words
        words.argtypes, words.restype = [C.c_uint32], C.c_uint64
        self.core, self.tmp = DevBuf(hip, 4 * g.n), DevBuf(hip, 4 * words(g.n))
        self.fn = scs.lib().scs_core_run
        self.fn.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.c_void_p,
                            C.c_void_p, C.c_uint32]

    def run(self, stream=None, blocks=0):
        assert self.fn(self.off.p, self.adj.p, self.n, self.core.p, self.tmp.p, stream, blocks) == 0

    def check(self):
        got = self.core.get(np.zeros(self.n, np.uint32))
        assert np.array_equal(got, self.want)

    def close(self):
        for b in (self.off, self.adj, self.core, self.tmp):
            b.free()


@pytest.mark.parametrize("blocks", [1, 2, 9, 300, 4096])
def test_any_number_of_blocks(blocks):
    """4,096 blocks of 512 threads are more than the GPU holds at once (at most
    2,048 threads a CU): those left over come when the others have ended."""
    hip = _hip()
    p = Peel(hip, 20000, 12, 3)
    print("core numbers with", blocks, "blocks", flush=True)
    for _ in range(2):
        p.run(blocks=blocks)
        p.check()
    p.close()
