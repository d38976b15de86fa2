"""Performance cases of the seeder: what a user's program has it do, through
the package's public entry points, from a call of a few reads to the
human-scale workloads of the benchmark.

The references and reads are the benchmark configurations' (gs_synth_preset):
a 1 Mbp reference with 300 bp repeats, a 100 Mbp one with interspersed and
tandem repeats, a 3.1 Gbp human-scale one.  An index belongs to its reference
and is what a program keeps between calls, so it is made once per process and
shared by the states that use it; every state has reads (or rows, or a
reference to index) of its own, made from its seed.

Every output is a whole number (intervals, positions, offsets, counts, index
structures), so there is nothing to compute in 64 bits: exact() has no values.
"""
import ctypes as C
import gc
import math
import random

import numpy as np

import gpuseed_amd as gs

# gs_synth_preset numbers: reference genome and reads of the configurations
SMALL, MEDIUM, HUMAN = 1, 2, 3
UNEVEN = 4  # the read mix: 70 % 100-250 bp, 25 % 1-5 kbp, 5 % 5-20 kbp

# Index shapes: "reference" is what the reference program keeps (13-mer table
# and sampled suffix array); "full" adds everything a batched user adds (16-mer
# table, direct-extension structures, pair table).
PLAIN_SHAPE, FULL_SHAPE = "reference", "full"


def listed():
    return [
        # A request of 64 reads on a resident index: launches, waits and the
        # slowest read decide, not throughput.  The entry point without
        # allocation is the one meant for it.
        {"name": "tiny-request", "what": "noalloc", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "reads": "short", "n": 64, "read_len": 150, "read_min": 150, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 3},
        # 1000 reads of an uneven mix with the command line's defaults (batched
        # kernel, 13-mer table): a small interactive call.
        {"name": "small-uneven", "what": "seed", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "reads": "uneven", "n": 1000, "read_len": 0, "read_min": 0, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 3},
        # gs_seed with its default kernel (the plain one) on 100,000 SMEM reads.
        {"name": "plain-smem", "what": "seed", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "reads": "short", "n": 100_000, "read_len": 150, "read_min": 150, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 0},
        # The default kernel again, on reads of uneven lengths up to 20 kbp.
        {"name": "plain-uneven", "what": "seed", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "reads": "uneven", "n": 3000, "read_len": 0, "read_min": 0, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 0},
        # The command line's defaults in MEM mode, whose outputs are many more
        # than SMEM's, on trimmed reads of 36 to 101 bases.
        {"name": "batched-mem", "what": "seed", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "reads": "short", "n": 300_007, "read_len": 101, "read_min": 36, "k": 20, "smem": False, "max_occ": 500,
         "kernel": 3},
        # Suffix-array rows to text positions by themselves (the reference's
        # walk over the sampled suffix array).
        {"name": "locate-rows", "what": "locate", "preset": MEDIUM, "length": 100_000_000, "shape": PLAIN_SHAPE,
         "n": 5_000_003},
        # The reference's own small case: 1 Mbp, MEM, 10,000 x 100 bp with Ns,
        # every row located, all defaults.
        {"name": "small-mem", "what": "seed", "preset": SMALL, "length": 1_000_000, "shape": PLAIN_SHAPE,
         "reads": "short", "n": 10_000, "read_len": 100, "read_min": 100, "k": 20, "smem": False, "max_occ": 0,
         "kernel": 0},
        # Making an index on the device (a program's start): suffix sorting,
        # occurrence blocks, 13-mer and tandem tables, the direct structures.
        {"name": "build-index", "what": "build", "preset": MEDIUM, "length": 5_000_011, "sa_intv": 7},
        # 300,000 short reads against a 100 Mbp reference with every table.
        {"name": "batched-smem", "what": "seed", "preset": MEDIUM, "length": 100_000_000, "shape": FULL_SHAPE,
         "reads": "short", "n": 300_000, "read_len": 150, "read_min": 150, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 3},
        # Human scale, reads resident on the device: the headline workload in a
        # batch of 1,000,000 reads, results fetched.
        {"name": "human-batch", "what": "batch", "preset": HUMAN, "length": 3_100_000_000, "shape": FULL_SHAPE,
         "reads": "short", "n": 1_000_000, "read_len": 150, "read_min": 150, "k": 19, "smem": True, "max_occ": 500,
         "kernel": 3},
        # Human scale, uneven lengths, the pipeline as a captured graph from
        # host memory to host memory.
        {"name": "human-uneven-graph", "what": "graph", "preset": HUMAN, "length": 3_100_000_000,
         "shape": FULL_SHAPE, "reads": "uneven", "n": 60_000, "read_len": 0, "read_min": 0, "k": 19, "smem": True,
         "max_occ": 500, "kernel": 3},
        # Human scale, served: 24 requests of 1 to 20,000 uneven reads arrive
        # together and are all waited for.
        {"name": "human-served", "what": "serve", "preset": HUMAN, "length": 3_100_000_000, "shape": FULL_SHAPE,
         "reads": "uneven", "n": 20_000, "requests": 24, "read_len": 0, "read_min": 0, "k": 19, "smem": True,
         "max_occ": 500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["noalloc", "seed", "seed", "seed", "batch", "graph", "serve", "locate", "build"])
    if what == "build":
        return {"what": "build", "preset": MEDIUM, "length": _log(rng, 300_000, 5_000_000),
                "sa_intv": rng.choice([4, 7, 16, 32])}
    preset = rng.choice([SMALL, MEDIUM, MEDIUM, MEDIUM])
    length = _log(rng, 300_000, 3_000_000) if preset == SMALL else _log(rng, 5_000_000, 150_000_000)
    shape = rng.choice([PLAIN_SHAPE, PLAIN_SHAPE, FULL_SHAPE])
    if rng.random() < 0.1:
        preset, length, shape = HUMAN, 3_100_000_000, FULL_SHAPE
    case = {"what": what, "preset": preset, "length": length, "shape": shape}
    if what == "locate":
        return {**case, "n": _log(rng, 1000, 5_000_000)}
    reads = "short" if what == "noalloc" else rng.choice(["short", "short", "uneven"])
    kernel = rng.choice([0, 3, 3, 3, 1])
    # reads by the bases that they hold (about 1500 a read in the uneven mix);
    # fewer where the plain kernel runs, and where nothing is allocated
    bases = _log(rng, 3_000, 2_000_000 if what == "noalloc" else 80_000_000 if kernel and what != "serve"
                 else 40_000_000 if what == "serve" else 15_000_000 if reads == "short" else 3_000_000)
    read_len = rng.choice([51, 76, 100, 101, 125, 150, 150, 160, 250]) if reads == "short" else 0
    n = max(1, bases // (read_len or 1500))
    # the shortest length that seldom occurs by chance, or some more
    k = max(14, math.ceil(math.log(length, 4)) + 3) + rng.choice([0, 0, 0, 1, 3, 8])
    case.update(reads=reads, n=n, read_len=read_len, read_min=rng.choice([read_len, read_len, min(36, read_len)]),
                k=k, smem=rng.random() < 0.7, max_occ=rng.choice([50, 500, 500]))
    if what == "serve":
        requests = rng.randint(2, 30)
        return {**case, "n": max(1, n // requests), "requests": requests}
    return {**case, "kernel": kernel}


# ---- the index of a process ---------------------------------------------------

_kept = {}  # key -> (reference codes, Index): the last one used


def _index(case):
    key = (case["preset"], case["length"], case["shape"])
    if key not in _kept:
        _kept.clear()  # a human-scale index takes more than half of the card
        gc.collect()
        codes = _reference(case["preset"], case["length"], None)
        index = gs.Index(codes=codes, sa_intv=7)
        if case["shape"] == FULL_SHAPE:
            index.set_kmer_len(16)
            index.set_direct(True)
            index.set_pairs(True)
        _kept[key] = (codes, index)
    return _kept[key]


def _reference(preset, length, seed):
    params, _ = gs.preset(preset)
    params.length = length
    if seed is not None:
        params.seed = 1 + seed
    return gs.synth_reference(params)


def _reads(codes, case, n, seed):
    _, q = gs.preset(UNEVEN if case["reads"] == "uneven" else case["preset"])
    if case["reads"] == "short":
        q.classes[0].len_min, q.classes[0].len_max = case["read_min"], case["read_len"]
    q.n_reads = n
    q.seed = 1000 + seed
    return gs.synth_reads(codes, q)[:3]


def _opts(case):
    return gs.make_opts(k=case["k"], smem=case["smem"], max_occ=case["max_occ"], kernel=case.get("kernel", 3))


# ---- results --------------------------------------------------------------------
# A program reads a call's results into arrays that it keeps for the next
# call; these hold the results of one call, zeros behind them.


class Kept:
    """Result arrays for reads of `bases` bases in all."""

    def __init__(self, case, n, bases):
        per_seed, per_pos = (0.06, 0.1) if case["smem"] else (0.3, 0.6)
        self.nseeds = np.zeros(n, np.uint32)
        self.npos = np.zeros(n, np.uint32)
        self.seed_off = np.zeros(n + 1, np.uint64)
        self.pos_off = np.zeros(n + 1, np.uint64)
        self.seeds = np.zeros((int(per_seed * bases) + 4096, 6), np.uint32)
        self.pos = np.zeros(int(per_pos * bases) + 65536, np.uint32)

    def buffers(self):
        """For the entry point that writes into the caller's arrays."""
        u32, u64 = C.POINTER(C.c_uint32), C.POINTER(C.c_uint64)
        return gs.ResultBuffers(
            self.nseeds.ctypes.data_as(u32), self.npos.ctypes.data_as(u32), self.seed_off.ctypes.data_as(u64),
            self.pos_off.ctypes.data_as(u64), self.seeds.ctypes.data_as(C.POINTER(gs.SeedRec)),
            self.pos.ctypes.data_as(u32), len(self.seeds), len(self.pos), 0, 0)

    def take(self, res):
        """Copies a gs_result in and frees it."""
        n, ns, np_ = res.n_reads, res.n_seeds, res.n_pos
        if ns > len(self.seeds) or np_ > len(self.pos):  # more than reads usually give: larger arrays
            self.seeds = np.zeros((max(2 * len(self.seeds), ns), 6), np.uint32)
            self.pos = np.zeros(max(2 * len(self.pos), np_), np.uint32)
        C.memmove(self.nseeds.ctypes.data, res.read_nseeds, 4 * n)
        C.memmove(self.npos.ctypes.data, res.read_npos, 4 * n)
        C.memmove(self.seed_off.ctypes.data, res.read_seed_off, 8 * (n + 1))
        C.memmove(self.pos_off.ctypes.data, res.read_pos_off, 8 * (n + 1))
        C.memmove(self.seeds.ctypes.data, res.seeds, C.sizeof(gs.SeedRec) * ns)
        C.memmove(self.pos.ctypes.data, res.pos, 4 * np_)
        gs.lib().gs_result_free(C.byref(res))

    def arrays(self):
        """Unsigned numbers seen as signed ones of their size."""
        return {"nseeds": self.nseeds.view(np.int32), "npos": self.npos.view(np.int32),
                "seed_off": self.seed_off.view(np.int64), "pos_off": self.pos_off.view(np.int64),
                "seeds": self.seeds.view(np.int32), "pos": self.pos.view(np.int32)}


def _reads_args(reads):
    buf, offs, lens = reads
    return (C.cast(buf.ctypes.data, C.c_char_p), offs.ctypes.data_as(C.POINTER(C.c_uint64)),
            lens.ctypes.data_as(C.POINTER(C.c_uint32)), len(lens))


def _done(rc, what):
    if rc != gs.GS_OK:
        raise gs.GsError(what, rc)


def prepare(case, seed):
    what = case["what"]
    if what == "build":
        return {"case": case, "codes": _reference(case["preset"], case["length"], seed)}
    codes, index = _index(case)
    state = {"case": case, "index": index}
    if what == "locate":
        rng = np.random.default_rng(seed)
        state["rows"] = rng.integers(0, case["length"] + 1, case["n"], dtype=np.uint32)
        return state
    state["opts"] = _opts(case)
    if what == "serve":
        rng = random.Random(case["requests"])  # sizes belong to the case, reads to the seed
        sizes = [_log(rng, 1, case["n"]) for _ in range(case["requests"])]
        state["requests"] = [_reads(codes, case, n, 64 * seed + i) for i, n in enumerate(sizes)]
        state["kept"] = [Kept(case, n, n * (case["read_len"] or 1500)) for n in sizes]
        state["server"] = gs.Server(index, opts=state["opts"])
        return state
    state["reads"] = _reads(codes, case, case["n"], seed)
    state["kept"] = Kept(case, case["n"], case["n"] * (case["read_len"] or 1500))
    if what in ("batch", "graph"):
        state["batch"] = gs.Batch(index, state["reads"], opts=state["opts"])
    if what == "graph":
        state["batch"].run()
        state["batch"].capture()
    return state


def run(state):
    case = state["case"]
    what = case["what"]
    L = gs.lib()
    if what == "seed":
        res = gs.Result()
        _done(L.gs_seed(state["index"].h, *_reads_args(state["reads"]), C.byref(state["opts"]), C.byref(res)),
              "gs_seed")
        state["kept"].take(res)
        return state["kept"].arrays()
    if what == "noalloc":
        out = state["kept"].buffers()
        _done(L.gs_seed_noalloc(state["index"].h, *_reads_args(state["reads"]), C.byref(state["opts"]),
                                C.byref(out)), "gs_seed_noalloc")
        return state["kept"].arrays()
    if what in ("batch", "graph"):
        if what == "batch":
            state["batch"].run()
        else:
            state["batch"].replay()
        res = gs.Result()
        _done(L.gs_batch_fetch(state["batch"].h, C.byref(res)), "gs_batch_fetch")
        state["kept"].take(res)
        return state["kept"].arrays()
    if what == "serve":
        server = state["server"]
        tickets = [server.submit(r) for r in state["requests"]]
        for ticket, kept in zip(tickets, state["kept"]):
            res, info = gs.Result(), gs.RequestInfo()
            _done(L.gs_server_wait(server.h, ticket, C.byref(res), C.byref(info)), "gs_server_wait")
            kept.take(res)
        # two arrays a request, those that tell all
        return [{k: v for k, v in kept.arrays().items() if k in ("seeds", "pos")} for kept in state["kept"]]
    if what == "locate":
        return state["index"].locate(state["rows"]).view(np.int32)
    with gs.Index(codes=state["codes"], sa_intv=case["sa_intv"]) as index:
        index.set_direct(True)
        info = index.info()
        rows, inverse, text = index.read_direct(0, info.seq_len)
        return {"primary": int(info.primary), "occ": index.read_occ(0, info.n_blocks).view(np.int32),
                "sa": rows.view(np.int32), "isa": inverse.view(np.int32), "text": text}


def exact(case, seed):
    """No value: every output is a whole number, equal or wrong."""
    return None


def work(case):
    """Reads (or rows, or the reference) in, results out, and of the index one
    16-byte entry per strand and k bases: less cannot tell what occurs."""
    if case["what"] == "locate":
        return {"bytes": 4 * case["n"] + 4 * case["n"] + 4 * case["n"], "flops": 0}
    if case["what"] == "build":
        n = case["length"]
        return {"bytes": n + n // 6 + 9 * n, "flops": 0}
    n = case["n"]
    if case["what"] == "serve":  # log-uniform sizes: their mean
        n = case["requests"] * n / max(1.0, math.log(max(2, n)))
    bases = n * (case["read_len"] if case["reads"] == "short" else 1500)
    seeds = 0.025 * bases
    return {"bytes": bases + 12 * n + 24 * n + 28 * seeds + 2 * 16 * bases / case["k"], "flops": 0}
