"""The plain kernel on reads from many exact copies: its intervals keep their
size there, so that only size records wide enough to hold it end a task early.
Its kernel time is held against that of the batched kernel with 16-bit records
(the same procedure with shortcuts besides), its results against the oracle's."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LETTERS = np.frombuffer(b"ACGT", np.uint8)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


def text_of(rng, copies, unit_len, n):
    text = rng.integers(0, 4, n, dtype=np.uint8)
    unit = rng.integers(0, 4, unit_len, dtype=np.uint8)
    for p in rng.permutation(n // unit_len - 1)[:copies] * unit_len:
        text[p:p + unit_len] = unit
    return text, unit


def reads_of(rng, unit, n, length):
    bases = np.tile(unit, length // len(unit) + 2)
    buf = np.empty(n * length, np.uint8)
    for i in range(n):
        at = rng.integers(0, len(unit))
        read = bases[at:at + length].copy()
        wrong = rng.random(length) < 0.01
        read[wrong] = rng.integers(0, 4, wrong.sum())
        buf[i * length:(i + 1) * length] = LETTERS[read]
    return buf, np.arange(n, dtype=np.uint64) * length, np.full(n, length, np.uint32)


# sizes that 4 bits cannot hold, and that 8 cannot; reads held whole and in
# segments.  With 4-bit records the plain kernel took 2.4 to 2.8 times as long as the other.
@pytest.mark.parametrize("copies", [30, 600])
@pytest.mark.parametrize("n,length", [(50000, 150), (300, 2000)])
def test_plain_kernel_prunes_in_repeats(g, copies, n, length):
    rng = np.random.default_rng(copies)
    text, unit = text_of(rng, copies, 2000, 3_000_000)
    arrays = reads_of(rng, unit, n, length)
    with g.Index(codes=text, sa_intv=7) as X:
        b = g.Batch(X, arrays, k=19, smem=False, max_occ=20)
        t = {}
        for kernel in (0, 2):
            b.run(kernel)
            t[kernel] = min(b.run(kernel).t_kernel for _ in range(5))
        b.close()
    say("copies=%d reads=%d of %d: plain %.0f us, 16-bit batched %.0f us" % (copies, n, length, 1e6 * t[0], 1e6 * t[2]))
    assert t[0] < 1.8 * t[2]


@pytest.mark.parametrize("smem", [True, False])
def test_plain_kernel_in_repeats_equals_the_oracle(g, smem, tmp_path):
    import oracle_bind as ob
    rng = np.random.default_rng(11)
    text, unit = text_of(rng, 300, 400, 200_000)
    prefix = str(tmp_path / "rep")
    g.build_index_host(text, 7, prefix)
    ox = ob.Index(prefix)
    with g.Index(prefix) as X:
        for n, length in ((200, 150), (20, 161), (6, 1500)):
            buf, offs, lens = reads_of(rng, unit, n, length)
            reads = [buf[int(o):int(o) + int(l)].tobytes() for o, l in zip(offs, lens)]
            want, _ = ob.seed(ox, reads, 19, smem=smem, prune=1)
            want = [[(x, y, l, u, list(p)) for (x, y, l, u, p) in r] for r in want]
            say("smem=%d reads=%d of %d" % (smem, n, length))
            assert g.seed(X, reads, k=19, smem=smem, kernel=0).as_lists() == want
    ox.close()
