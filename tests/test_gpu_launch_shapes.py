"""Launches around the number of items from which waves take them from the
queue (a lane per item of a full grid), and the sizes at which half, three
quarters and all of the grid's waves start: batched and plain kernels, short
reads and segments, the same seeds as an index without splitting gives with
the other kernel, and as the oracle gives for a sample of them."""
import random

import numpy as np
import pytest

from conftest import build_index, repetitive_text, sample_reads

pytestmark = pytest.mark.gpu

LANES = 256 * 16 * 64  # of a grid that fills the chip with 4-bit size records


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def case(g, tmp_path_factory):
    rng = random.Random(262)
    text = repetitive_text(rng, 60000, n_units=10, unit_len=300, copies=8, div=0.02, tandem=4)
    prefix = build_index(tmp_path_factory.mktemp("shapes"), text, 7)
    short = sample_reads(rng, text, 700, 20, 70, sub=0.01, indel=0.002, n_frac=0.05)
    longer = sample_reads(rng, text, 12, 200, 3000, sub=0.02, indel=0.005, n_frac=0.1)
    return dict(prefix=prefix, pool=short + longer, n_short=len(short))


# items (two per short read) at the edges of each rule
@pytest.mark.parametrize("items", [LANES - 2, LANES, LANES + 2, 2 * LANES - 2, 2 * LANES, 6 * LANES - 2, 6 * LANES + 2])
@pytest.mark.parametrize("n_long", [0, 5])
def test_launches_at_the_edges_of_their_rules(g, case, items, n_long):
    import oracle_bind as ob
    rng = np.random.default_rng(items + n_long)
    n = items // 2
    pick = rng.integers(0, case["n_short"], n)
    if n_long:
        pick[rng.choice(n, n_long, replace=False)] = case["n_short"] + rng.integers(0, 12, n_long)
    buf, offs, lens = g.pack_reads(case["pool"])
    arrays = (buf, offs[pick], lens[pick])
    head = 400
    ox = ob.Index(case["prefix"])
    want, _ = ob.seed(ox, [case["pool"][i] for i in pick[:head]], 19, smem=True, prune=1)
    ox.close()
    want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
    with g.Index(case["prefix"]) as X:
        outs = [g.seed(X, arrays=arrays, k=19, smem=True, kernel=kernel, split_tasks=split)
                for kernel, split in ((3, 0), (0, 0), (1, 0xFFFF))]
        for out in outs[1:]:
            for a in ("read_nseeds", "read_npos", "read_seed_off", "read_pos_off", "seeds", "pos"):
                assert np.array_equal(getattr(outs[0], a), getattr(out, a)), a
        few = g.seed(X, arrays=(buf, offs[pick[:head]], lens[pick[:head]]), k=19, smem=True, kernel=3)
        assert few.as_lists() == want
        ns = int(outs[0].read_seed_off[head])
        assert np.array_equal(outs[0].seeds[:ns], few.seeds)
