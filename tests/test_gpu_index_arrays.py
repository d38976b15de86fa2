"""What the builder makes on the device, against plain loops: the text read
back from any offset, interval tables at the edges of their launches, and
codes above 3, which it refuses wherever they lie."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g(built):
    import gpuseed_amd
    return gpuseed_amd


@pytest.fixture(scope="module")
def codes():
    rng = np.random.default_rng(96)
    return np.tile(rng.integers(0, 4, 2500, dtype=np.uint8), 4)[:9973]


def test_text_from_any_offset(g, codes):
    n = len(codes)
    with g.Index(codes=codes, sa_intv=7) as X:
        X.set_direct(True)
        for first in (0, 1, 15, 16, 17, 63, 64, n - 5):
            for count in (0, 1, 2, 3, 4, 5, 63, 64, 1025):
                count = min(count, n - first)
                assert np.array_equal(X.read_text(first, count), codes[first:first + count]), (first, count)
        assert np.array_equal(X.read_text(0, n), codes)


@pytest.mark.parametrize("chunk", [0, 1000, 4096])
def test_tables_against_counting(g, codes, chunk):
    text = codes.tobytes()
    g.lib().gs_set_launch_chunk(chunk)
    try:
        with g.Index(codes=codes, sa_intv=7) as X:
            table = X.read_kmer(0, 1 << 26)
    finally:
        g.lib().gs_set_launch_chunk(0)
    # occurring 13-mers: their interval holds as many rows as they have occurrences
    seen = {}
    for i in range(len(codes) - 12):
        seen[text[i:i + 13]] = seen.get(text[i:i + 13], 0) + 1
    index = [sum(int(c) << (2 * (12 - j)) for j, c in enumerate(w)) for w in seen]
    t = np.asarray(table).reshape(-1, 2).astype(np.int64)
    sizes = t[:, 1] - t[:, 0] + 1
    assert [int(sizes[i]) for i in index] == list(seen.values())
    assert int((sizes > 0).sum()) == len(seen)


@pytest.mark.parametrize("at", [0, 1, 255, 256, 9972])
@pytest.mark.parametrize("code", [4, 7, 255])
def test_codes_above_3_are_refused(g, codes, at, code):
    bad = codes.copy()
    bad[at] = code
    with pytest.raises(g.GsError) as e:
        g.Index(codes=bad, sa_intv=7)
    assert e.value.rc == g.GS_EINVAL
