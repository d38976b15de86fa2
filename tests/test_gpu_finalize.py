"""Merging, counting and writing of seeds and rows at the sizes where the
kernels' ways part: reads with fewer and more merged entries than a lane takes
alone (16), seeds with more rows than a wave writes at once (64) and than it
takes per turn (65,536), the MEM row skip inside and across reads, capped
occurrences.  Exact, against the oracle."""
import random
import sys

import pytest

from conftest import build_index, random_text, repetitive_text, sample_reads

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.mark.parametrize("max_occ", [0, 1, 63, 65])
@pytest.mark.parametrize("smem,k", [(True, 14), (False, 14), (False, 20)])
def test_entries_and_rows_against_the_oracle(g, tmp_path, smem, k, max_occ):
    import oracle_bind as ob
    rng = random.Random(17 * k + max_occ)
    # 150 copies of a unit (intervals above and below 64 rows) and repeats of
    # several depths, so that MEM reads have from 0 to far more than 16 entries
    unit = random_text(rng, 80)
    text = repetitive_text(rng, 30000, n_units=6, unit_len=200, copies=9, div=0.04, tandem=4)
    text += "".join(unit[: rng.randint(30, 80)] + random_text(rng, rng.randint(1, 9)) for _ in range(150))
    prefix = build_index(tmp_path, text, 7)
    reads = sample_reads(rng, text, 500, 14, 160, sub=0.01, indel=0.002, n_frac=0.1)
    reads += sample_reads(rng, text, 30, 161, 700, sub=0.02, indel=0.004, n_frac=0.1)
    rng.shuffle(reads)
    ox = ob.Index(prefix)
    want, _ = ob.seed(ox, reads, k, smem=smem, prune=1, max_occ=max_occ)
    want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
    counts = [len(r) for r in want]
    say("entries per read: max %d, reads over 16: %d" % (max(counts), sum(c > 16 for c in counts)))
    with g.Index(prefix) as X:
        for direct in (False, True):
            X.set_direct(direct)
            for n in (len(reads), 1, 65):
                got = g.seed(X, reads[:n], k=k, smem=smem, kernel=3, max_occ=max_occ).as_lists()
                if n == len(reads) or smem:  # MEM rows depend on the reads that follow
                    assert got == want[:n], (direct, n)
    ox.close()


@pytest.mark.parametrize("smem", [True, False])
def test_intervals_of_more_rows_than_a_turn(g, tmp_path, smem):
    """A base repeated 70,000 times: intervals of 64 to 70,000 rows, every row
    located, against the oracle (in MEM mode the batch-wide row skip, which
    reaches the next read's entries, takes part)."""
    import oracle_bind as ob
    rng = random.Random(3)
    text = random_text(rng, 3000) + "A" * 70000 + random_text(rng, 1000)
    prefix = build_index(tmp_path, text, 7)
    reads = [b"A" * 14, b"A" * 40 + b"C", b"A" * 100, b"ACGT" * 10]
    ox = ob.Index(prefix)
    want, _ = ob.seed(ox, reads, 14, smem=smem, prune=1)
    want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
    ox.close()
    assert max(len(p) for r in want for (_, _, _, _, p) in r) > 65536
    with g.Index(prefix) as X:
        for kernel in (3, 0):
            got = g.seed(X, reads, k=14, smem=smem, kernel=kernel).as_lists()
            say([(x, y, u - l + 1, len(p)) for x, y, l, u, p in got[0]])
            assert got == want, kernel
