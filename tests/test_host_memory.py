"""What the library does where memory is short or refused, and what it
allocates where it says it allocates nothing.  CPU only: the library runs in a
child process on a stand-in for the HIP runtime (fake_hip.c) whose kernels do
nothing, so that calls end without results and only their allocations, copies
and return codes are looked at."""
import os
import shutil
import subprocess
import sys
import textwrap

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.join(HERE, "..")
pytestmark = pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not found")

PRELUDE = """
import ctypes as C, sys
F = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
F.fake_held.restype = F.fake_calls.restype = C.c_uint64
F.fake_limit.argtypes = [C.c_int, C.c_uint64, C.c_uint64]
F.fake_chain_rows.argtypes = [C.c_uint64]
DEVICE, PINNED, ANY = 0, 1, 2**64 - 1
sys.path.insert(0, sys.argv[2])
import numpy as np
import gpuseed_amd as g
TEXT = 600_000

def index():
    return g.Index(sys.argv[3])

def reads(n, length):
    return (np.frombuffer(b"ACGT", np.uint8)[np.random.default_rng(n).integers(0, 4, n * length)].copy(),
            np.arange(n, dtype=np.uint64) * length, np.full(n, length, np.uint32))

def rc_of(f, *a, **kw):
    try:
        f(*a, **kw)
        return 0
    except g.GsError as e:
        return e.rc
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    """Runs a program on the stand-in; its output."""
    d = tmp_path_factory.mktemp("fake")
    shim = str(d / "libfake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-pthread", "-I/opt/rocm/include", "-o", shim,
                    os.path.join(HERE, "fake_hip.c")], check=True, stdout=subprocess.PIPE, stderr=subprocess.PIPE)
    import gpuseed_amd
    prefix = str(d / "idx")
    gpuseed_amd.build_index_host(np.random.default_rng(1).integers(0, 4, 600_000, dtype=np.uint8), 7, prefix)

    def run(program):
        p = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(program), shim, ROOT, prefix],
                           stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=300)
        assert p.returncode == 0, p.stderr.decode()[-3000:]
        return p.stdout.decode().split()

    return run


def test_reading_text_needs_no_device_memory(child):
    """Short ranges allocate nothing; long ones do without where there is none."""
    out = child("""
        X = index()
        F.fake_chain_rows(TEXT + 1)
        X.set_direct(True)
        before = F.fake_calls(DEVICE)
        X.read_text(5, 1000)
        X.read_direct(0, 100)
        print(F.fake_calls(DEVICE) - before)
        F.fake_limit(DEVICE, F.fake_held(DEVICE), ANY)
        print(rc_of(X.read_text, 0, TEXT), rc_of(X.read_direct, 3, TEXT - 3))
        print(rc_of(X.set_kmer_len, 13))
    """)
    assert out == ["0", "0", "0", "0"]


def test_noalloc_does_without_pinned_memory(child):
    """Its pinned megabyte is refused when the index is opened, then to be had."""
    out = child("""
        small, large = reads(20, 150), reads(20000, 150)
        F.fake_limit(PINNED, ANY, 4096)
        X = index()
        for r in (small, large):
            print(rc_of(g.seed_noalloc, X, r, 100, 100, k=19, smem=True, kernel=3))
        held = F.fake_held(PINNED)
        F.fake_limit(PINNED, ANY, ANY)
        with index() as Y:
            print(F.fake_held(PINNED) - held >= 1 << 20, rc_of(g.seed_noalloc, X, small, 100, 100, k=19, kernel=0))
    """)
    assert out == ["0", "0", "True", "0"]


def test_batches_do_without_pinned_memory(child):
    """Calls, batches and servers, of one chunk and of several."""
    out = child("""
        F.fake_limit(PINNED, ANY, 4096)
        X = index()
        for r in (reads(1, 150), reads(20, 150), reads(100_000, 150)):
            print(rc_of(g.seed, X, arrays=r, k=19, smem=True, kernel=3))
            b = g.Batch(X, r, k=19, smem=False, batch_bases=1000)
            b.run()
            print(len(b.fetch().pos))
            b.close()
        g.Server(X, k=19, round_bases=100_000).close()
        print(F.fake_held(PINNED) < 8192)
    """)
    assert out == ["0"] * 6 + ["True"]


def test_locate_does_without_pinned_memory(child):
    out = child("""
        F.fake_limit(PINNED, ANY, 1024)
        X = index()
        for n in (1, 1000, 5_000_000):
            rows = np.arange(n, dtype=np.uint32)
            print(rc_of(X.locate, rows))
        print(np.array_equal(X.locate(rows), rows))
    """)
    assert out == ["0", "0", "0", "True"]


@pytest.mark.parametrize("shift", [1, 2_097_152, 3_000_000, 5_000_000, -1, -3_000_000])
def test_locate_where_rows_and_positions_overlap(child, shift):
    """The stand-in's walks leave the rows as they are."""
    out = child("""
        shift, n = %d, 9_000_000
        X = index()
        both = np.arange(n + abs(shift), dtype=np.uint32)
        rows, at = both[max(0, -shift):][:n], both[max(0, shift):][:n]
        want = rows.copy()
        u32 = C.POINTER(C.c_uint32)
        print(g.lib().gs_index_locate(X.h, rows.ctypes.data_as(u32), n, at.ctypes.data_as(u32)))
        print(np.array_equal(at, want))
    """ % shift)
    assert out == ["0", "True"]


def test_build_takes_its_sort_arrays_in_pieces(child):
    """No block of the sort's 37 bytes per base can be had, but smaller ones
    can.  The stand-in sorts nothing, so the build fails later on, with an
    index that does not fit its text."""
    out = child("""
        codes = np.zeros(1_000_000, np.uint8)
        print(rc_of(g.Index, codes=codes) == g.GS_EINVAL)
        F.fake_limit(DEVICE, ANY, 20_000_000)
        print(rc_of(g.Index, codes=codes) == g.GS_EINVAL)
        F.fake_limit(DEVICE, 20_000_000, ANY)
        print(rc_of(g.Index, codes=codes) == -2, F.fake_held(DEVICE))
    """)
    assert out == ["True", "True", "True", "0"]


def test_batches_do_without_room_for_split_off_pieces(child):
    """No room for the pieces when the batch is made, or for its results
    beside them."""
    out = child("""
        X = index()
        r = reads(50_000, 150)
        start = F.fake_held(DEVICE)
        def made(limit, **kw):
            F.fake_limit(DEVICE, limit, ANY)
            rc, held = 0, 0
            try:
                b = g.Batch(X, r, k=19, **kw)
                held = F.fake_held(DEVICE) - start
                b.run()
                b.run()
                b.fetch()
                b.close()
            except g.GsError as e:
                rc = e.rc
            return rc, held
        rc, bare = made(ANY, split_tasks=g.NO_SPLIT)
        rc2, full = made(ANY)
        print(rc, rc2, full > bare + 2_000_000)
        room = 2048  # for the results, which are empty here
        for limit in (bare + room, bare + 1_000_000, (bare + full) // 2, full - 1, full):
            rc, held = made(start + limit)
            print(rc, held <= limit)
        rc, _ = made(start + bare // 2)
        print(rc)
    """)
    assert out == ["0", "0", "True"] + ["0", "True"] * 5 + ["-2"]


def test_served_mem_rounds_allocate_no_more_than_smem_rounds(child):
    """More reference batches than the plan's launch holds: their list has its
    room from the start, as everything else but the results."""
    out = child("""
        X = index()
        r = reads(2000, 150)
        for smem in (True, False):
            with g.Server(X, k=19, smem=smem, batch_bases=1000, round_bases=1_000_000, workers=1) as S:
                before = F.fake_calls(DEVICE)
                for _ in range(3):
                    S.wait(S.submit(r))
                print(F.fake_calls(DEVICE) - before)
    """)
    assert out == ["2", "2"]  # seed records and rows


@pytest.mark.parametrize("opts", ["seg_tasks=64", "seg_tasks=1", "seg_tasks=64, smem=False, batch_bases=2000",
                                  "seg_tasks=5, split_tasks=g.NO_SPLIT"])
@pytest.mark.parametrize("n,length", [(20_000, 150), (300, 4000)])
def test_a_round_s_device_bytes_are_those_it_allocates(child, opts, n, length):
    """peak_round_bytes against the buffers of a batch of the same reads (each
    allocated with a quarter and 256 bytes of headroom)."""
    out = child("""
        X = index()
        r = reads(%d, %d)
        kw = dict(dict(k=19, smem=True, kernel=3), **dict(%s))
        before = F.fake_held(DEVICE)
        b = g.Batch(X, r, **kw)
        held = F.fake_held(DEVICE) - before
        b.close()
        with g.Server(X, workers=1, round_bases=10_000_000, **kw) as S:
            S.wait(S.submit(r))
            peak = S.stats().peak_round_bytes
        print(0 <= held - 1.25 * peak <= 40 * 256, held, peak)
    """ % (n, length, opts))
    assert out[0] == "True", out


@pytest.mark.parametrize("seg_tasks", [1, 3, 64])
def test_rounds_stay_within_their_budget(child, seg_tasks):
    out = child("""
        X = index()
        with g.Server(X, budget_bytes=16_000_000, workers=1, round_bases=1_000_000, k=19, smem=True, batch_bases=5000,
                      seg_tasks=%d) as S:
            rs = [reads(5, 2000 + i) for i in range(100)] + [reads(1000, 100 + i) for i in range(5)]
            for t in [S.submit(r) for r in rs]:
                S.wait(t)
            st = S.stats()
            print(st.peak_round_bytes <= 8_000_000, st.peak_round_bytes > 4_000_000, st.peak_round_bytes, st.n_rounds)
    """ % seg_tasks)
    assert out[:2] == ["True", "True"], out
