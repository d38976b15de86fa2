"""The plain kernel (kernel 0) as one work item per lane: reads cut into
segments, launches of fewer and of more items than lanes, and gs_seed_noalloc
with long reads, at the sizes where its array holds the pieces of work
splitting, only the work items, or neither (then seed_streams runs).  All
comparisons are exact."""
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
    rng = random.Random(733)
    text = repetitive_text(rng, 60000, n_units=12, unit_len=300, copies=12, div=0.03, tandem=8)
    prefix = build_index(tmp_path_factory.mktemp("plain"), text, 7)
    reads = (sample_reads(rng, text, 300, 10, 160, sub=0.02, indel=0.002, n_frac=0.2) +
             sample_reads(rng, text, 60, 161, 400, sub=0.02, indel=0.005, n_frac=0.3) +
             sample_reads(rng, text, 6, 4000, 9000, sub=0.05, indel=0.02, n_frac=0.5))
    rng.shuffle(reads)
    return dict(prefix=prefix, reads=reads)


def same(a, b):
    return (np.array_equal(a.seeds, b.seeds) and np.array_equal(a.pos, b.pos) and
            np.array_equal(a.read_seed_off, b.read_seed_off) and np.array_equal(a.read_pos_off, b.read_pos_off))


@pytest.mark.parametrize("smem,k", [(True, 19), (True, 14), (False, 16)])
def test_plain_kernel_on_long_reads_equals_the_oracle(g, case, smem, k):
    import oracle_bind as ob
    ox = ob.Index(case["prefix"])
    want, _ = ob.seed(ox, case["reads"], k, smem=smem, prune=1)
    want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
    with g.Index(case["prefix"]) as X:
        for tables in (False, True):
            if tables:
                X.set_kmer_len(16)
            for kw in (dict(), dict(seg_tasks=1), dict(seg_tasks=112), dict(split_tasks=g.NO_SPLIT)):
                say("smem=%d k=%d tables=%d %s" % (smem, k, tables, kw))
                assert g.seed(X, case["reads"], k=k, smem=smem, kernel=0, **kw).as_lists() == want, kw
    ox.close()


def test_plain_kernel_around_the_lanes_of_the_grid(g, case):
    short = [r for r in case["reads"] if len(r) <= 160]
    base = g.pack_reads(short)
    with g.Index(case["prefix"]) as X:
        for n in (131071, 131073, 200001):
            pick = np.random.default_rng(n).integers(0, len(short), n)
            arrays = (base[0], base[1][pick], base[2][pick])
            say("reads=%d" % n)
            want = g.seed(X, arrays=arrays, k=19, smem=True, kernel=3, split_tasks=g.NO_SPLIT)
            assert same(g.seed(X, arrays=arrays, k=19, smem=True, kernel=0), want)


@pytest.mark.parametrize("smem", [True, False])
@pytest.mark.parametrize("kernel", [0, 1, 3])
def test_noalloc_with_long_reads_equals_gs_seed(g, case, smem, kernel):
    reads = case["reads"]
    sets = [reads, reads[:1], [r for r in reads if len(r) <= 250], [r for r in reads if len(r) > 160]]
    with g.Index(case["prefix"]) as X:
        for rs in sets:
            for kw in (dict(), dict(seg_tasks=5), dict(split_tasks=1)):
                say("noalloc smem=%d kernel=%d reads=%d %s" % (smem, kernel, len(rs), kw))
                arrays = g.pack_reads(rs)
                want = g.seed(X, arrays=arrays, k=17, smem=smem, kernel=kernel, **kw)
                assert same(g.seed_noalloc(X, arrays, k=17, smem=smem, kernel=kernel, **kw), want)


# 150 bp reads take 4,438 bytes each in the plain layout of the 2^28-byte
# array and 16 more for their work items: 59,000 hold the work items and not
# the pieces, 60,450 neither, 60,500 do not fit at all
@pytest.mark.parametrize("n,fits", [(59000, True), (60450, True), (60500, False)])
def test_noalloc_at_the_array_s_limits(g, case, n, fits):
    rng = np.random.default_rng(5)
    letters = np.frombuffer(b"ACGT", np.uint8)
    buf = letters[rng.integers(0, 4, 150 * n)]  # random reads: few seeds, so that the outputs fit too
    short = next(r for r in case["reads"] if len(r) >= 150)
    for i in range(0, 64):  # and some with seeds, all over the call
        at = (i * (n // 64)) * 150
        buf[at:at + 150] = np.frombuffer(short[:150], np.uint8)
    arrays = (buf, np.arange(n, dtype=np.uint64) * 150, np.full(n, 150, np.uint32))
    with g.Index(case["prefix"]) as X:
        say("noalloc reads=%d" % n)
        if not fits:
            with pytest.raises(g.GsError) as ei:
                g.seed_noalloc(X, arrays, k=19, smem=True, kernel=0, max_occ=4)
            assert ei.value.rc == g.GS_ERANGE
            return
        want = g.seed(X, arrays=arrays, k=19, smem=True, kernel=3, max_occ=4)
        assert len(want.seeds) > 0
        assert same(g.seed_noalloc(X, arrays, k=19, smem=True, kernel=0, max_occ=4), want)
