"""Served rounds and large launches against the oracle, on samples: every
kernel shares the slots, segments, splitting and joins of one template, so that
their agreement alone says little.  SMEM seeds depend on a read only, so reads
are picked from where launches end and where reads are cut into segments; MEM
requests are compared whole."""
import random
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


@pytest.fixture(scope="module")
def world(g, tmp_path_factory):
    """A 3 Mbp reference with the repeats of the 3.1 Gbp preset and uneven reads (100 bp to 20 kbp)."""
    import oracle_bind as ob
    rp, qp = g.preset(4)
    rp.length = 3_000_000
    qp.n_reads = 30_000
    ref = g.synth_reference(rp)
    buf, offs, lens = g.synth_reads(ref, qp)[:3]
    prefix = str(tmp_path_factory.mktemp("samples") / "idx")
    g.build_index_host(ref, 7, prefix)
    ox = ob.Index(prefix)
    yield dict(prefix=prefix, ox=ox, buf=buf, offs=offs, lens=lens)
    ox.close()


def oracle(world, arrays, picked, **kw):
    """Per-read lists of the picked reads, seeded as one input."""
    import oracle_bind as ob
    buf, offs, lens = arrays
    reads = [buf[int(offs[i]):int(offs[i]) + int(lens[i])].tobytes() for i in picked]
    out, _ = ob.seed(world["ox"], reads, 19, prune=1, threads=8, **kw)
    return [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in out]


def sample(rng, lens):
    """The last reads, some with segments, some others."""
    n = len(lens)
    cut = [i for i in range(n) if lens[i] > 160]
    picked = set(range(max(0, n - 16), n)) | set(rng.sample(range(n), min(n, 24)))
    return sorted(picked | set(rng.sample(cut, min(len(cut), 8))))


def request(world, first, n):
    offs, lens = world["offs"][first:first + n], world["lens"][first:first + n]
    lo, hi = int(offs[0]), int(offs[-1]) + int(lens[-1])
    return world["buf"][lo:hi].copy(), (offs - np.uint64(lo)).copy(), lens.copy()


@pytest.mark.parametrize("seg_tasks", [0, 7])
@pytest.mark.parametrize("smem", [True, False])
def test_served_requests(g, world, smem, seg_tasks):
    rng = random.Random(seg_tasks + smem)
    sizes = [1, 2, 3, 17, 64, 200, 900] + ([4000, 4000] if smem else [1100])
    requests = [request(world, rng.randrange(0, len(world["lens"]) - n), n) for n in sizes]
    with g.Index(world["prefix"]) as X:
        # small rounds: requests share some and are spread over others
        with g.Server(X, round_bases=400_000, round_growth=1, k=19, smem=smem, kernel=3, seg_tasks=seg_tasks,
                      max_occ=50) as S:
            tickets = [S.submit(r) for r in requests]
            for r, t in zip(requests, tickets):
                res, info = S.wait(t)
                n = len(r[2])
                say("smem=%d seg_tasks=%d reads=%d rounds=%d" % (smem, seg_tasks, n, info.n_rounds))
                picked = sample(rng, r[2]) if smem else list(range(n))
                assert [res.read(i) for i in picked] == oracle(world, r, picked, smem=smem, max_occ=50)


# items per lane of the launch: less than one, from one to two, up to six, more
@pytest.mark.parametrize("kind,n", [("short", 60_000), ("short", 200_000), ("short", 500_000), ("short", 1_000_000),
                                    ("uneven", 1000), ("uneven", 8000), ("uneven", 30_000)])
def test_ends_of_launches(g, world, kind, n):
    rng = random.Random(n)
    if kind == "short":
        held = [i for i in range(len(world["lens"])) if world["lens"][i] <= 160]
        pick = np.array(held)[np.random.default_rng(n).integers(0, len(held), n)]
    else:
        pick = np.arange(n)
    arrays = (world["buf"], world["offs"][pick].copy(), world["lens"][pick].copy())
    picked = sample(rng, arrays[2])
    want = oracle(world, arrays, picked, smem=True, max_occ=50)
    with g.Index(world["prefix"]) as X:
        b = g.Batch(X, arrays, k=19, smem=True, max_occ=50)
        for kernel in (0, 1, 2, 3):
            say("%s n=%d kernel=%d" % (kind, n, kernel))
            b.run(kernel)
            out = b.fetch()
            assert [out.read(i) for i in picked] == want, kernel
        b.close()
