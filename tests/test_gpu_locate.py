"""gs_index_locate over its pinned chunks (8 MB, two in turn): sizes around
one, two and three of them, rows without a position, the caller's rows
overwritten in place, and two threads at once.  Exact, against the oracle."""
import ctypes as C
import random
import threading

import numpy as np
import pytest

from conftest import build_index, random_text

pytestmark = pytest.mark.gpu

CHUNK = (8 << 20) // 4


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def case(g, tmp_path_factory):
    import oracle_bind as ob
    text = random_text(random.Random(8), 5000)
    prefix = build_index(tmp_path_factory.mktemp("locate"), text, 5)
    ox = ob.Index(prefix)
    want = np.array([ox.locate(r) for r in range(len(text) + 1)], dtype=np.uint64).astype(np.uint32)
    ox.close()
    return dict(prefix=prefix, want=np.concatenate([want, np.full(3, 0xFFFFFFFF, np.uint32)]))


@pytest.mark.parametrize("n", [1, 63, 64, 65, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK, 2 * CHUNK + 3, 3 * CHUNK + 1])
@pytest.mark.parametrize("direct", [False, True])
def test_locate_sizes(g, case, n, direct):
    rng = np.random.default_rng(n)
    with g.Index(case["prefix"]) as X:
        X.set_direct(direct)
        for _ in range(2):
            rows = rng.integers(1, len(case["want"]), n, dtype=np.uint32)
            assert np.array_equal(X.locate(rows), case["want"][rows])
        both = rows.copy()
        p = both.ctypes.data_as(C.POINTER(C.c_uint32))
        assert g.lib().gs_index_locate(X.h, p, n, p) == g.GS_OK
        assert np.array_equal(both, case["want"][rows])


def test_locate_from_two_threads(g, case):
    with g.Index(case["prefix"]) as X:
        bad = []

        def work(seed):
            rng = np.random.default_rng(seed)
            for n in (1000, CHUNK + 77, 5):
                rows = rng.integers(1, len(case["want"]), n, dtype=np.uint32)
                if not np.array_equal(X.locate(rows), case["want"][rows]):
                    bad.append((seed, n))

        threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
        [t.start() for t in threads]
        [t.join() for t in threads]
        assert not bad
