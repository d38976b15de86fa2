"""Results on their way to the caller: gathered by one launch into pinned
chunks and copied out from there (gs_batch_fetch, small calls of
gs_seed_noalloc), against the copies of each array that a captured replay and
a large gs_seed_noalloc call make."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ARRAYS = ("read_nseeds", "read_npos", "read_seed_off", "read_pos_off", "seeds", "pos")


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def index(g):
    rp, _ = g.preset(1)
    rp.length = 400_000
    codes = g.synth_reference(rp)
    with g.Index(codes=codes, sa_intv=7) as X:
        yield codes, X


# reads, and the bytes of results that they must give: below a lane's 16
# bytes, within one chunk, past the megabyte that leaves gs_seed_noalloc
# through pinned memory, past two chunks of 8 MB (the last one partial)
@pytest.mark.parametrize("n,least", [(0, 0), (1, 0), (3, 0), (511, 0), (20_001, 1 << 20), (300_003, 17 << 20)])
def test_results_arrive_whole(g, index, n, least):
    codes, X = index
    _, qp = g.preset(1)
    qp.n_reads = n
    qp.seed = 77
    reads = g.synth_reads(codes, qp)[:3] if n else (np.zeros(1, np.uint8), np.zeros(0, np.uint64),
                                                    np.zeros(0, np.uint32))
    o = g.make_opts(k=16, smem=False, max_occ=50, kernel=3)
    batch = g.Batch(X, reads, opts=o)
    batch.run()
    eager = batch.fetch()
    batch.capture()
    batch.replay()
    replayed = batch.fetch()
    batch.close()
    assert sum(getattr(eager, a).nbytes for a in ARRAYS) >= least
    for a in ARRAYS:
        assert np.array_equal(getattr(eager, a), getattr(replayed, a)), a
    once = g.seed(X, arrays=reads, opts=o)
    for a in ARRAYS:
        assert np.array_equal(getattr(eager, a), getattr(once, a)), a
    if n <= 20_001:
        whole = g.seed_noalloc(X, reads, opts=o)
        for a in ARRAYS:
            assert np.array_equal(getattr(eager, a), getattr(whole, a)), a
