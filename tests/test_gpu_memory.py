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
