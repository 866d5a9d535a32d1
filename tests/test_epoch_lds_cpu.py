"""LDS of the search waves: every wave of an epoch is resident, engines without
the GPU heuristic give none of it away, and those with it leave a block of the
heuristic its piece."""

import ctypes as C

import pytest

from scs_amd import scs

PIECE, PIECES = 1280, 128  # the granule in which a CU hands out its 160 KB


def _fns():
    b, s = scs.lib().scs_epoch_lds_bytes, scs.lib().scs_epoch_lds_spare
    b.argtypes, s.argtypes = [C.c_uint32, C.c_uint32], [C.c_uint32, C.c_uint32]
    b.restype = s.restype = C.c_uint32
    return b, s


def _bitmap_capacity(nbytes):
    return nbytes // 8 * 32  # two bits per vertex, in words


@pytest.mark.parametrize("spare", [0, 1])
@pytest.mark.parametrize("wpc", range(1, 9))
def test_all_waves_of_a_cu_fit(wpc, spare):
    lds, _ = _fns()
    static = PIECES // 4 * PIECE - lds(4, 0)  # a wave's struct, to the next 8 bytes
    pieces = -(-(static + lds(wpc, spare)) // PIECE)
    assert 8000 < static < 9000 and pieces * wpc <= PIECES - spare


def test_bitmaps_without_the_gpu_heuristic():
    lds, _ = _fns()
    # 32,256 bytes at four waves per CU and 11,776 at eight: what they had
    # before any piece was left free
    assert _bitmap_capacity(lds(4, 0)) >= 129_024
    assert _bitmap_capacity(lds(8, 0)) >= 47_104
    assert lds(1, 0) == lds(2, 0) == 48 * 1024


def test_pieces_left_for_the_heuristic():
    lds, spare = _fns()
    lo, hi = _bitmap_capacity(lds(4, 1)), _bitmap_capacity(lds(4, 0))
    assert lo < hi
    assert spare(4, 4000) == spare(4, lo) == 1
    assert spare(4, lo + 32) == spare(4, hi) == 0
    assert spare(4, hi + 32) == spare(4, 500_000) == 1
    assert [spare(w, 4000) for w in (5, 8)] == [0, 0]
