"""What an engine sets aside for its preprocessing buffers before it sizes the
search state is what those buffers take."""

import ctypes as C

import pytest

from scs_amd import scs


@pytest.mark.parametrize("n", [1, 64, 65, 4000, 100_000, 4_194_304])
def test_reserve_covers_the_buffers(n):
    f = scs.lib().scs_prep_buffer_bytes
    f.argtypes, f.restype = [C.c_uint32], C.c_uint64
    groups = -(-n // 64)
    masks = 5 * 8 * n            # elig, vis and three frontiers
    rows = 64 * (2 + 4) * n      # distances and local ids of 64 queries
    counts = 64 * 4 * groups     # per 64 vertices
    chunks = f(n) - masks - rows - counts
    # one row of 64 words per chunk, at most 256 chunks
    assert 0 < chunks <= 256 * 64 * 4 and chunks % 256 == 0
