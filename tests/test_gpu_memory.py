"""Paths chosen by a size, on both sides of its line.  Exact."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


def test_text_on_both_sides_of_the_unpacking_rule(g):
    codes = np.random.default_rng(4).integers(0, 4, 600_001, dtype=np.uint8)
    with g.Index(codes=codes, sa_intv=7) as X:
        X.set_direct(True)
        for first in (0, 3, 17, 300_000):
            for count in (1, 15, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, 300_001):
                if first + count > len(codes):
                    continue
                say("first=%d count=%d" % (first, count))
                assert np.array_equal(X.read_text(first, count), codes[first:first + count])
        assert np.array_equal(X.read_text(0, len(codes)), codes)


@pytest.mark.parametrize("shift", [1, 2_500_000, -2_500_000])
def test_locate_where_rows_and_positions_overlap(g, shift):
    import ctypes as C
    codes = np.random.default_rng(4).integers(0, 4, 600_001, dtype=np.uint8)
    n = 7_000_003
    both = np.random.default_rng(5).integers(0, len(codes) + 3, n + abs(shift), dtype=np.uint32)
    rows, out = both[max(0, -shift):][:n], both[max(0, shift):][:n]
    with g.Index(codes=codes, sa_intv=7) as X:
        want = X.locate(rows.copy())
        say("shift=%d" % shift)
        u32 = C.POINTER(C.c_uint32)
        assert g.lib().gs_index_locate(X.h, rows.ctypes.data_as(u32), n, out.ctypes.data_as(u32)) == g.GS_OK
    assert np.array_equal(out, want)
