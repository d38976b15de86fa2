"""Calls on a device whose host refuses pinned memory beyond a page: they
copy from and to the caller's arrays instead; and a build that gets no block
for all of its sort's arrays.  Exact, against the same calls in a process that
has the memory."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.join(HERE, "..")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not found")]

PROGRAM = """
import ctypes as C, sys
shim, root, prefix, what, out = sys.argv[1:]
if shim:
    F = C.CDLL(shim, mode=C.RTLD_GLOBAL)
    F.no_pinned_limit.argtypes = [C.c_size_t]
    F.no_device_between.argtypes = [C.c_size_t, C.c_size_t]
    F.no_pinned_limit(4096 if what != "build" else 1 << 40)
    if what == "build":
        F.no_device_between(5_000_000, 15_000_000)  # the sort's arrays together: 11.1 MB, the largest 2.4
sys.path.insert(0, root)
import numpy as np
import gpuseed_amd as g
codes = np.random.default_rng(1).integers(0, 4, 300_000, dtype=np.uint8)
rng = np.random.default_rng(2)
res = {}
def keep(name, r):
    res.update({name + k: getattr(r, k) for k in ("read_nseeds", "read_npos", "read_seed_off", "read_pos_off", "pos")})
    res[name + "seeds"] = r.seeds.view(np.uint32)
if what == "build":
    X = g.Index(codes=np.concatenate([codes[:150_000], codes[:150_000]]), sa_intv=7)
    X.set_direct(True)
    res["occ"] = X.read_occ(0, X.info().n_blocks)
    res["sa"], res["isa"], res["pos"] = X.read_direct(0, 300_000)
else:
    X = g.Index(prefix)
for n, length in ((1, 150), (300, 150), (60, 700), (20000, 150)):
    at = rng.integers(0, len(codes) - length, n)
    buf = np.frombuffer(b"ACGT", np.uint8)[codes[at[:, None] + np.arange(length)]].reshape(-1).copy()
    buf[rng.random(len(buf)) < 0.02] = ord("A")
    reads = (buf, np.arange(n, dtype=np.uint64) * length, np.full(n, length, np.uint32))
    for smem in (True, False):
        kw = dict(k=15, smem=smem, kernel=3, batch_bases=2000)
        name = "%d-%d-%d-" % (n, length, smem)
        if what == "noalloc":
            keep(name, g.seed_noalloc(X, reads, **kw))
        elif what == "locate":
            res[name + "pos"] = X.locate(rng.integers(0, len(codes) + 3, n * length, dtype=np.uint32))
        elif what == "seed":
            keep(name, g.seed(X, arrays=reads, **kw))
        elif what == "batch":
            b = g.Batch(X, reads, **kw)
            b.run()
            keep(name, b.fetch())
            b.close()
print("refused", F.no_pinned_refused() if shim else 0, flush=True)
np.savez(out, **res)
X.close()
"""


@pytest.fixture(scope="module")
def setting(tmp_path_factory):
    import gpuseed_amd
    d = tmp_path_factory.mktemp("pinned")
    shim = str(d / "libno_pinned.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", shim, os.path.join(HERE, "no_pinned.c"),
                    "-L/opt/rocm/lib", "-lamdhip64", "-ldl"], check=True, stdout=subprocess.PIPE,
                   stderr=subprocess.PIPE)
    prefix = str(d / "idx")
    codes = np.random.default_rng(1).integers(0, 4, 300_000, dtype=np.uint8)
    gpuseed_amd.build_index_host(codes, 7, prefix)
    return d, shim, prefix


def run(setting, what, shim):
    d, _, prefix = setting
    out = str(d / (what + ("-without" if shim else "-with") + ".npz"))
    p = subprocess.run([sys.executable, "-c", PROGRAM, shim, ROOT, prefix, what, out], stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, timeout=100)
    assert p.returncode == 0, p.stderr.decode()[-3000:]
    refused = int(p.stdout.decode().split("refused")[1].split()[0])
    return np.load(out), refused


@pytest.mark.parametrize("what", ["noalloc", "seed", "batch", "locate", "build"])
def test_without_pinned_memory(setting, what):
    want, _ = run(setting, what, "")
    got, refused = run(setting, what, setting[1])
    assert refused > 0
    assert sum(a.size for k, a in want.items() if k.endswith("pos")) > 0
    assert sorted(got) == sorted(want)
    for key in want:
        assert np.array_equal(got[key], want[key]), key
