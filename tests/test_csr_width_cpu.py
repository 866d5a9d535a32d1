"""Which graphs are read through 32-bit offsets: those whose rows end far enough
below 2^32 that a loop's step past a row's end does not wrap."""

import ctypes as C
import os
import re

import pytest

from scs_amd import build, scs

TOP = 1 << 32


@pytest.mark.parametrize("nnz,fits", [(0, 1), (6_000_000, 1), (TOP - 4097, 1), (TOP - 4096, 0),
                                      (TOP - 2, 0), (TOP - 1, 0), (TOP, 0), (TOP + 10, 0)])
def test_entries_that_fit(nnz, fits):
    f = scs.lib().scs_csr_fits32
    f.argtypes, f.restype = [C.c_uint64], C.c_int
    assert f(nnz) == fits


def test_the_margin_covers_the_longest_step():
    """Steps of the heuristic's loops over a row: 4 x HEU_T entries."""
    src = open(os.path.join(build.CSRC, "scs_heu.hip")).read()
    threads = int(re.search(r"#define HEU_T (\d+)", src).group(1))
    assert "j0 += 4 * HEU_T" in src and 2 * 4 * threads <= 4096
