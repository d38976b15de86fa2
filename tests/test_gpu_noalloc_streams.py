"""gs_seed_noalloc where its array holds the call but not the work items of
the kernel that gs_seed would run: seed_streams, in the forms for reads of up
to 160 bases, up to 256, and longer ones with their size records in the array.
Exact, against gs_seed and, for a sample, the oracle."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ARRAY = 256 << 20
LETTERS = np.frombuffer(b"ACGT", np.uint8)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


def layout(n, length, k, kernel, seg_tasks):
    """Bytes of the array that n reads of one length need before their results
    (the call is refused beyond the array), and with the work items (above the
    array: seed_streams runs)."""
    nr1, span, task = n + 1, n * length, length - k + 1
    chunks = 2 * n * ((length + 31) // 32)
    nseg = 1 if length <= 160 else -(-task // seg_tasks)
    n_items, n_long = 2 * n * nseg, n if length > 160 else 0

    def total(*slices):
        return sum((s + 255) & ~255 for s in slices)

    common = total(span + 32, 8 * nr1, 4 * nr1, 8 * nr1, 4 * nr1, 16 * (2 * n * task + 1), *[4 * nr1] * 4,
                   8 * nr1, 8 * nr1, 8 * (nr1 // 2048 + 2), 16, 16, 288)
    short = kernel != 0 and length <= 160
    least = common + total(8 * nr1, 4 * (span + 16) if not short and length > 256 else 0,
                           *([16 * n + 8, 16 * (chunks + 1)] if short else []))
    items = common + total(4 * (n_long + 1), 8 * nr1, 8 * (n_items + 1), 16 * (chunks + 1) if kernel else 0,
                           40 * (-(-n // 2048) + 1), 8 * (n_long + 1), 16 * n_items if n_long else 0)
    return least, items


@pytest.mark.parametrize("length,seg_tasks,kernel,smem", [
    (150, 64, 0, True),   # codes in LDS, 160 bases
    (161, 64, 0, True),   # 256 bases
    (250, 64, 0, False),
    (256, 64, 3, True),
    (257, 1, 0, True),    # size records in the array
    (700, 1, 3, False),
    (3000, 1, 0, True),
])
def test_streams_equal_gs_seed(g, length, seg_tasks, kernel, smem, tmp_path):
    import oracle_bind as ob
    k = 19
    n = next(n for n in range(100, 70000, 50) if layout(n, length, k, kernel, seg_tasks)[1] > ARRAY)
    least, items = layout(n, length, k, kernel, seg_tasks)
    assert items > ARRAY and least + (1 << 19) < ARRAY  # room for the results
    say("reads=%d of %d seg_tasks=%d kernel=%d smem=%d: %d, %d bytes" % (n, length, seg_tasks, kernel, smem, least, items))
    rng = np.random.default_rng(length)
    text = rng.integers(0, 4, 60_000, dtype=np.uint8)
    for p in range(0, 60_000 - 400, 1500):
        text[p:p + 400] = text[:400]  # 40 copies
    buf = LETTERS[rng.integers(0, 4, n * length)]  # random reads: few seeds, so that the results fit
    taken = [i * (n // 40) for i in range(40)] + [n - 1]
    for i in taken:  # and some with seeds, all over the call
        at = int(rng.integers(0, len(text) - length))
        read = LETTERS[text[at:at + length]]
        read[rng.random(length) < 0.02] = ord("N")
        buf[i * length:(i + 1) * length] = read
    arrays = (buf, np.arange(n, dtype=np.uint64) * length, np.full(n, length, np.uint32))
    prefix = str(tmp_path / "idx")
    g.build_index_host(text, 7, prefix)
    kw = dict(k=k, smem=smem, max_occ=4, seg_tasks=seg_tasks)
    with g.Index(prefix) as X:
        want = g.seed(X, arrays=arrays, kernel=3, **kw)
        got = g.seed_noalloc(X, arrays, kernel=kernel, **kw)
    for name in ("seeds", "pos", "read_nseeds", "read_npos", "read_seed_off", "read_pos_off"):
        assert np.array_equal(getattr(got, name), getattr(want, name)), name
    if smem:  # MEM's row skip looks at the reads around
        ox = ob.Index(prefix)
        exact, _ = ob.seed(ox, [buf[i * length:(i + 1) * length].tobytes() for i in taken], k, smem=True, max_occ=4,
                           prune=1)
        ox.close()
        lists = got.as_lists()
        assert [lists[i] for i in taken] == [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in exact]
