"""Backward steps at the left edge of the codes and size records that a lane
holds (160 positions, on multiples of 32), where the next position's code and
the record are no longer the ones read ahead: reads that match far to the
left of it, with and without codes above 3 there.  Exact, against the oracle."""
import random

import pytest

from conftest import build_index, repetitive_text

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def case(g, tmp_path_factory):
    rng = random.Random(160)
    text = repetitive_text(rng, 40000, n_units=12, unit_len=600, copies=6, div=0.01, tandem=4)
    prefix = build_index(tmp_path_factory.mktemp("steps"), text, 7)
    reads = []
    for length in (159, 160, 161, 191, 192, 193, 223, 257, 320, 321, 400, 777):
        for at in (None, 0, 1, 31, 32, 33, 63, 64, 95, 96, 97, 127, 128, 130):
            p = rng.randint(0, len(text) - length)
            r = bytearray(text[p:p + length].encode())
            if at is not None and at < length:
                r[length - 1 - at if rng.random() < 0.5 else at] = ord("N")
            reads.append(bytes(r))
    return dict(prefix=prefix, reads=reads)


@pytest.mark.parametrize("seg_tasks", [1, 31, 33, 64, 112])
@pytest.mark.parametrize("smem,k", [(True, 19), (False, 15)])
def test_steps_past_the_window(g, case, seg_tasks, smem, k):
    import oracle_bind as ob
    ox = ob.Index(case["prefix"])
    want, _ = ob.seed(ox, case["reads"], k, smem=smem, prune=1)
    ox.close()
    want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
    with g.Index(case["prefix"]) as X:
        for direct in (False, True):
            X.set_direct(direct)
            for kernel in (0, 1, 2, 3):
                got = g.seed(X, case["reads"], k=k, smem=smem, kernel=kernel, seg_tasks=seg_tasks).as_lists()
                assert got == want, (direct, kernel)
