"""Calls around the sizes where the plan's and the counts' scans take fewer
items per thread (256, 1024 reads), with long reads whose items and codes
several waves write, and seeds around the 16 rows from which a wave writes
them.  Exact, against the oracle."""
import random

import numpy as np
import pytest

from conftest import build_index, random_text, repetitive_text, sample_reads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def case(g, tmp_path_factory):
    rng = random.Random(256)
    # units of 14 to 18 copies: seeds of 15, 16 and 17 rows among others
    text = repetitive_text(rng, 30000, n_units=8, unit_len=250, copies=10, div=0.03, tandem=5)
    for copies in (14, 15, 16, 17, 18, 70):
        unit = random_text(rng, 60)
        text += "".join(unit + random_text(rng, 20) for _ in range(copies))
    prefix = build_index(tmp_path_factory.mktemp("small"), text, 7)
    short = sample_reads(rng, text, 900, 0, 160, sub=0.01, indel=0.002, n_frac=0.05)
    longer = sample_reads(rng, text, 20, 161, 5000, sub=0.02, indel=0.005, n_frac=0.1)
    return dict(prefix=prefix, pool=short + longer, n_short=len(short))


@pytest.mark.parametrize("n", [1, 8, 9, 255, 256, 257, 1023, 1024, 1025])
@pytest.mark.parametrize("smem,k", [(True, 19), (False, 16)])
def test_small_calls_against_the_oracle(g, case, n, smem, k):
    import oracle_bind as ob
    rng = np.random.default_rng(n)
    pick = rng.integers(0, case["n_short"], n)
    pick[:: 37] = rng.integers(case["n_short"], len(case["pool"]), len(pick[:: 37]))
    reads = [case["pool"][i] for i in pick]
    ox = ob.Index(case["prefix"])
    with g.Index(case["prefix"]) as X:
        for max_occ in (0, 16):
            want, _ = ob.seed(ox, reads, k, smem=smem, prune=1, max_occ=max_occ)
            want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
            for kernel in (3, 0):
                assert g.seed(X, reads, k=k, smem=smem, kernel=kernel, max_occ=max_occ).as_lists() == want, kernel
            arrays = g.pack_reads(reads)
            assert g.seed_noalloc(X, arrays, k=k, smem=smem, kernel=3, max_occ=max_occ).as_lists() == want
    ox.close()
