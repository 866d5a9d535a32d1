"""Core numbers on a GPU that is not the call's alone: more blocks than find room
(those that come late take no part), and calls that do not wait for each other
where they share nothing."""

import ctypes as C
import threading

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


def _stream(hip):
    s = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # not blocked by the default stream
    return s


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


def test_peels_of_several_streams_at_once():
    hip = _hip()
    peels = [Peel(hip, 30000, 10 + i, i) for i in range(4)]
    streams = [_stream(hip) for _ in peels]
    print("4 peels at once", flush=True)
    errors = []

    def work(p, s):
        try:
            for _ in range(3):
                p.run(s)
        except AssertionError as e:
            errors.append(e)

    ts = [threading.Thread(target=work, args=a) for a in zip(peels, streams)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    for p, s in zip(peels, streams):
        p.check()
        hip.hipStreamDestroy(s)
        p.close()


def test_a_call_does_not_wait_for_another_stream():
    """A call whose stream still waits for the host holds up no call on another
    stream."""
    hip = _hip()
    a, b = Peel(hip, 5000, 8, 1), Peel(hip, 5000, 8, 2)
    sa, sb = _stream(hip), _stream(hip)
    go = threading.Event()
    done_a, done_b = threading.Event(), threading.Event()
    wait = C.CFUNCTYPE(None, C.c_void_p)(lambda _: go.wait(20))
    assert hip.hipLaunchHostFunc(sa, wait, None) == 0
    ta = threading.Thread(target=lambda: (a.run(sa), done_a.set()))
    tb = threading.Thread(target=lambda: (b.run(sb), done_b.set()))
    ta.start()
    tb.start()
    print("one stream held by the host", flush=True)
    free = done_b.wait(5) and not done_a.is_set()
    go.set()
    ta.join()
    tb.join()
    assert free
    a.check()
    b.check()
    for s in (sa, sb):
        hip.hipStreamDestroy(s)
    a.close()
    b.close()
