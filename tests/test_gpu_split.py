"""Work splitting within a wave (the batched kernels' take_pieces): launches
of one item per wave, of fewer and of more items than lanes, and gs_seed_noalloc,
whose pieces lie where its outputs go later.  Seeds are whole numbers, so
every comparison is exact: against the oracle, and at sizes the oracle is slow
for against the same launch without splitting."""
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
    rng = random.Random(411)
    text = repetitive_text(rng, 60000, n_units=12, unit_len=300, copies=12, div=0.03, tandem=8)
    prefix = build_index(tmp_path_factory.mktemp("split"), text, 7)
    short = sample_reads(rng, text, 3000, 20, 160, sub=0.02, indel=0.002, n_frac=0.1)
    longer = sample_reads(rng, text, 40, 161, 2500, sub=0.03, indel=0.01, n_frac=0.2)
    return dict(prefix=prefix, short=short, longer=longer)


def same(a, b):
    return (np.array_equal(a.seeds, b.seeds) and np.array_equal(a.pos, b.pos) and
            np.array_equal(a.read_seed_off, b.read_seed_off) and np.array_equal(a.read_pos_off, b.read_pos_off))


@pytest.mark.parametrize("tables", [False, True])
@pytest.mark.parametrize("smem,k", [(True, 19), (False, 16)])
def test_small_launches_equal_the_oracle(g, case, smem, k, tables):
    """1 read to a few more items than waves (2048 reads: one item for each of
    4096 waves), every record width, with and without long reads."""
    import oracle_bind as ob
    ox = ob.Index(case["prefix"])
    with g.Index(case["prefix"]) as X:
        if tables:
            X.set_kmer_len(14)
            X.set_direct(True)
        for kernel, n, nl in ((3, 1, 0), (3, 33, 1), (1, 65, 2), (2, 130, 40), (3, 2047, 0), (3, 2049, 3)):
            reads = case["longer"][:nl] + case["short"][:n]
            want, _ = ob.seed(ox, reads, k, smem=smem, prune=1)
            want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
            for kw in (dict(), dict(split_tasks=1), dict(wg=64), dict(split_tasks=1, split_work=1, wg=256)):
                say("smem=%d tables=%d kernel=%d reads=%d+%d %s" % (smem, tables, kernel, nl, n, kw))
                got = g.seed(X, reads, k=k, smem=smem, kernel=kernel, **kw).as_lists()
                assert got == want, (kernel, n, nl, kw)
    ox.close()


@pytest.mark.parametrize("n", [131071, 131073, 150000])
def test_launches_around_the_lanes_of_the_grid(g, case, n):
    """262,144 lanes (4-bit records on 256 CUs): launches of just fewer and
    just more items than that take their items in different ways."""
    rng = np.random.default_rng(n)
    base = g.pack_reads(case["short"])
    pick = rng.integers(0, len(base[2]), n)
    arrays = (base[0], base[1][pick], base[2][pick])
    with g.Index(case["prefix"]) as X:
        want = g.seed(X, arrays=arrays, k=19, smem=True, kernel=3, split_tasks=g.NO_SPLIT)
        for kw in (dict(), dict(split_tasks=1), dict(split_tasks=1, split_work=1)):
            say("reads=%d %s" % (n, kw))
            assert same(g.seed(X, arrays=arrays, k=19, smem=True, kernel=3, **kw), want), kw


@pytest.mark.parametrize("smem", [True, False])
def test_noalloc_splits_like_gs_seed(g, case, smem):
    with g.Index(case["prefix"]) as X:
        for n in (1, 64, 3000):
            arrays = g.pack_reads(case["short"][:n])
            want = g.seed(X, arrays=arrays, k=19, smem=smem, kernel=3, split_tasks=g.NO_SPLIT)
            for kw in (dict(), dict(split_tasks=1), dict(split_tasks=g.NO_SPLIT)):
                say("noalloc smem=%d reads=%d %s" % (smem, n, kw))
                assert same(g.seed_noalloc(X, arrays, k=19, smem=smem, kernel=3, **kw), want), (n, kw)


@pytest.mark.parametrize("n", [8192, 8193])
def test_joins_on_both_sides_of_the_wave_per_stream_rule(g, case, n):
    """16,384 streams and two more."""
    base = g.pack_reads(case["short"])
    pick = np.random.default_rng(n).integers(0, len(base[2]), n)
    arrays = (base[0], base[1][pick], base[2][pick])
    with g.Index(case["prefix"]) as X:
        for smem in (True, False):
            want = g.seed(X, arrays=arrays, k=17, smem=smem, kernel=3, split_tasks=g.NO_SPLIT)
            assert same(g.seed(X, arrays=arrays, k=17, smem=smem, kernel=3, split_tasks=1), want), smem


@pytest.mark.parametrize("seg_tasks", [1, 2, 40, 112])
def test_joins_of_segments_and_their_pieces(g, case, seg_tasks):
    """Reads of 63, 64, 65 and 129 segments (one lane each, 64 at a time), and
    of many short ones; every segment split as far as it goes, so that 64
    chains do not fit the join's list at once."""
    import oracle_bind as ob
    rng = random.Random(seg_tasks)
    k = 15
    text = "".join(case["longer"][i].decode() for i in range(40)).replace("N", "A")
    reads = []
    for nseg in (63, 64, 65, 129):
        L = min(nseg * seg_tasks + k - 1, len(text) - 1)
        p = rng.randrange(0, len(text) - L)
        reads.append(text[p:p + L].encode())
    reads += case["longer"][:8]
    ox = ob.Index(case["prefix"])
    with g.Index(case["prefix"]) as X:
        for smem in (True, False):
            want, _ = ob.seed(ox, reads, k, smem=smem, prune=1)
            want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
            for kw in (dict(split_tasks=1), dict(split_tasks=g.NO_SPLIT), dict(kernel=0, split_tasks=1)):
                kw.setdefault("kernel", 3)
                say("seg_tasks=%d smem=%d %s" % (seg_tasks, smem, kw))
                assert g.seed(X, reads, k=k, smem=smem, seg_tasks=seg_tasks, **kw).as_lists() == want, kw
    ox.close()
