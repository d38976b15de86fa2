"""The batch plan computed on the device and the paired scans of counts, at
the edges of their tiles (2048 reads): task and code offsets, work items,
long reads among short ones, reference batches listed in the launch (up to 16
cuts) and in memory, reads that are not in order or overlap in the buffer.
Exact, against the oracle (whose plan is a loop) and the plain kernel."""
import random
import sys

import numpy as np
import pytest

from conftest import build_index, repetitive_text, sample_reads

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def case(g, tmp_path_factory):
    rng = random.Random(88)
    text = repetitive_text(rng, 40000, n_units=10, unit_len=250, copies=10, div=0.03, tandem=5)
    prefix = build_index(tmp_path_factory.mktemp("plan"), text, 7)
    short = sample_reads(rng, text, 2000, 0, 160, sub=0.01, indel=0.002, n_frac=0.05)
    longer = sample_reads(rng, text, 30, 161, 3000, sub=0.02, indel=0.005, n_frac=0.1)
    return dict(prefix=prefix, short=short, longer=longer)


def arrays_of(g, case, n, n_long, seed):
    rng = np.random.default_rng(seed)
    pool = case["short"] + case["longer"]
    pick = rng.integers(0, len(case["short"]), n)
    if n_long:
        pick[rng.choice(n, min(n, n_long), replace=False)] = len(case["short"]) + rng.integers(0, len(case["longer"]),
                                                                                                min(n, n_long))
    base = g.pack_reads(pool)
    return base[0], base[1][pick], base[2][pick]  # picked anywhere in the buffer, some twice


def same(a, b):
    return (np.array_equal(a.seeds, b.seeds) and np.array_equal(a.pos, b.pos) and
            np.array_equal(a.read_seed_off, b.read_seed_off) and np.array_equal(a.read_pos_off, b.read_pos_off) and
            np.array_equal(a.read_nseeds, b.read_nseeds) and np.array_equal(a.read_npos, b.read_npos))


@pytest.mark.parametrize("n", [1, 7, 2047, 2048, 2049, 4097])
@pytest.mark.parametrize("n_long", [0, 1, 90])
def test_plan_at_the_edges_of_tiles(g, case, n, n_long):
    import oracle_bind as ob
    ox = ob.Index(case["prefix"])
    arrays = arrays_of(g, case, n, n_long, 10 * n + n_long)
    reads = [arrays[0][int(o):int(o) + int(l)].tobytes() for o, l in zip(arrays[1], arrays[2])]
    with g.Index(case["prefix"]) as X:
        for smem, k in ((True, 19), (False, 20)):
            want, _ = ob.seed(ox, reads, k, smem=smem, prune=1)
            want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
            for kernel in (3, 0):
                say("n=%d n_long=%d smem=%d kernel=%d" % (n, n_long, smem, kernel))
                assert g.seed(X, arrays=arrays, k=k, smem=smem, kernel=kernel).as_lists() == want
            assert g.seed_noalloc(X, arrays, k=k, smem=smem, kernel=3).as_lists() == want
    ox.close()


@pytest.mark.parametrize("n_batches", [1, 2, 16, 17, 18, 200])
def test_reference_batches(g, case, n_batches):
    """MEM rows depend on where reference batches close; a call cut at the same
    reads, batch by batch, gives the same seeds."""
    n = 4 * n_batches + 3
    arrays = arrays_of(g, case, n, n // 10, n_batches)
    lens = arrays[2].astype(np.int64)
    bb = max(1, int(lens.sum()) // n_batches)
    cuts, acc = [0], 0
    for i, l in enumerate(lens):
        acc += int(l)
        if acc >= bb:
            cuts.append(i + 1)
            acc = 0
    if cuts[-1] != n:
        cuts.append(n)
    say("batches", len(cuts) - 1)
    with g.Index(case["prefix"]) as X:
        parts = []
        for a, z in zip(cuts, cuts[1:]):
            parts += g.seed(X, arrays=(arrays[0], arrays[1][a:z], arrays[2][a:z]), k=15, smem=False, kernel=0).as_lists()
        got = g.seed(X, arrays=arrays, k=15, smem=False, kernel=3, batch_bases=bb)
        assert got.as_lists() == parts
        assert same(g.seed_noalloc(X, arrays, k=15, smem=False, kernel=3, batch_bases=bb), got)
