// Seeding kernels: backward extension, SMEM/MEM finalisation, SA walk.
//
// Reference path replaced (seed_gen.cu): find_seed_intervals_gpu (2087-2413),
// DeviceSelect/DeviceScan/DeviceReduce and sum_arrays (3383-3430),
// filter/count kernels and the device-side segmented sort (865-1251),
// seeds_to_threads(_mem) and locate_seeds_gpu (555-724).
//
// Design (one read = two extension streams, forward and reverse):
//  * A lane owns one stream.  Streams are written in a common "virtual" form:
//    the forward stream reads the forward codes left-to-right, the reverse
//    stream reads the reverse-complement codes of the reversed read, and both
//    run the reference's forward-task procedure (2132-2264) on task ends
//    e = L, L-1, ..., k.  A virtual candidate [b, e) of the reverse stream is
//    the reference's reverse seed (L-e, L-b) (2272-2404).
//  * Tasks of a stream run one after another in the same lane, so pruning is
//    exact distance-1 pruning: task e stops at left end x as soon as its
//    interval size equals the size the previous tasks recorded for x (then
//    every occurrence of read[x,e) continues with read[e], so the task's seed
//    has the same left end as a longer one).  The reference approximates this
//    with 30-lane shuffles (2192-2212); its output does not depend on which
//    candidates are pruned, and neither does this one.
//  * Every loop iteration issues at most one memory operation per lane: a
//    13-mer table read or one occ entry (two when l-1 and u fall in different
//    96-base blocks).  The loop stays converged on the loads; all pointer
//    chasing between loads is LDS-only work on the staged read bytes and the
//    per-position size record.
//  * SMEM filtering happens in the lane: tasks finish in decreasing end order
//    and left ends never increase, so a task is a survivor exactly when its
//    left end is smaller than the previous finished task's (991-1018).  For
//    the same reason an SMEM stream ends when a task reaches the read start:
//    every later task would end there too and be filtered out.
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <mutex>
#include <thread>
#include <vector>

#include "gs_internal.h"

using gs::DevIndex;

namespace {

struct SeedParams {
  DevIndex X;
  const uint8_t* bases;     // batch bytes, padded by 16
  const uint64_t* offs;     // per read
  const uint32_t* lens;     // per read
  const uint64_t* task_off; // per read: sum of tasks of earlier reads
  uint32_t n_reads, k, smem, pad;
  uint4* cand;              // per read: 2*task_off .. : forward region then reverse region
  uint32_t* nF;
  uint32_t* nR;
  void* scratch;            // size records of reads longer than the LDS slots
};

template <typename AT>
struct SatMax {
  static constexpr uint32_t value = (uint32_t)(AT)(~(AT)0);
};

constexpr int kSeedBlock = 128;

template <typename AT, int LMAX>
struct Slot {
  static constexpr int bytes = ((LMAX + 2 * LMAX * (int)sizeof(AT)) + 15) & ~15;
};

template <typename AT, int LMAX>
__global__ void __launch_bounds__(kSeedBlock) seed_streams(SeedParams P) {
  constexpr int PAIR = Slot<AT, LMAX>::bytes;
  constexpr uint32_t SAT = SatMax<AT>::value;
  __shared__ __align__(16) uint8_t lds[(kSeedBlock / 2) * PAIR];
  const uint32_t gid = blockIdx.x * kSeedBlock + threadIdx.x;
  const uint32_t r = gid >> 1;
  const uint32_t strand = gid & 1;
  uint8_t* slot = lds + (threadIdx.x >> 1) * PAIR;
  const bool live = r < P.n_reads;
  const uint32_t L = live ? P.lens[r] : 0;
  const uint64_t off = live ? P.offs[r] : 0;
  const bool in_lds = L <= (uint32_t)LMAX;

  // stage the read bytes: the two lanes of a pair take alternate aligned 16-byte chunks
  if (live && in_lds && L) {
    const uint64_t c0 = off >> 4, c1 = (off + L - 1) >> 4;
    for (uint64_t ch = c0 + strand; ch <= c1; ch += 2) {
      const uint4 v = reinterpret_cast<const uint4*>(P.bases)[ch];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      for (int q = 0; q < 16; ++q) {
        const uint64_t pos = ch * 16 + q;
        if (pos >= off && pos < off + L) slot[pos - off] = (uint8_t)(w[q >> 2] >> ((q & 3) * 8));
      }
    }
  }
  __syncthreads();

  const uint8_t* src = in_lds ? slot : P.bases + off;
  AT* A = in_lds ? reinterpret_cast<AT*>(slot + LMAX) + strand * LMAX
                 : reinterpret_cast<AT*>(P.scratch) + 2 * off + strand * L;
  auto V = [&](int32_t i) -> uint32_t {
    return strand == 0 ? gs::code_fwd(src[i]) : gs::code_rev(src[L - 1 - i]);
  };

  const uint32_t k = P.k;
  const uint32_t ntask = L >= k ? L - k + 1 : 0;
  bool done = !live || L < k;
  for (uint32_t q = 0; !done && q < L; ++q) A[q] = 0;

  int32_t e = (int32_t)L;
  uint32_t p = 0, nbad = 0;
  if (!done)
    for (int j = 0; j < gs::kPrecalc; ++j) {
      const uint32_t c = V((int32_t)L - 1 - j);
      nbad += c > 3;
      p |= (c & 3u) << (2 * j);
    }
  int phase = 0;  // 0: task e waits for its table lookup; 1: task e is extending
  bool ext_miss = false;  // the task's extended-table pattern is absent: use the 13-mer path
  int32_t x = 0;
  uint32_t l = 0, u = 0, b = 0, s = 0, last_b = 0xFFFFFFFFu, nout = 0;
  uint4* outF = P.cand + (live ? 2 * P.task_off[r] : 0);

  auto next_task = [&]() -> bool {
    ext_miss = false;
    if ((uint32_t)(e - 1) < k) return false;
    const uint32_t cn = V(e - 14), co = V(e - 1);
    nbad = nbad + (cn > 3 ? 1u : 0u) - (co > 3 ? 1u : 0u);
    p = (p >> 2) | ((cn & 3u) << 24);
    --e;
    return true;
  };
  // size record at x: prune if the previous tasks recorded the same size there
  auto prune_at = [&](int32_t pos, uint32_t size) -> bool {
    const uint32_t sv = size >= SAT ? SAT : size;
    if (size < SAT && (uint32_t)A[pos] == sv) return true;
    A[pos] = (AT)sv;
    return false;
  };
  auto finish = [&]() {
    if ((uint32_t)e - b >= k && (!P.smem || b < last_b)) {
      if (strand == 0) {
        outF[ntask - 1 - nout] = make_uint4(b, (uint32_t)e, l, u);
      } else {
        outF[ntask + nout] = make_uint4((L - (uint32_t)e) | 0x80000000u, (L - b) | 0x80000000u, l, u);
      }
      ++nout;
    }
    last_b = b;
  };

  while (true) {
    int op = 0;
    uint32_t c = 0;
    while (!done) {
      if (phase == 0) {
        if (nbad == 0) {
          op = 1;
          break;
        }
        if (!next_task()) done = true;
        continue;
      }
      if (x < 0) {
        finish();
        // SMEM: once a task reaches the read start, every later task does too
        // (its pattern is a substring of this one's), so none can pass the
        // filter b < last_b = 0: the stream is done
        phase = 0;
        if (P.smem || !next_task()) done = true;
        continue;
      }
      c = V(x);
      if (c <= 3) {
        op = 2;
        break;
      }
      b = (uint32_t)x;  // code > 3 after the window: interval kept, position consumed
      if (prune_at(x, s)) {
        phase = 0;
        if (!next_task()) done = true;
        continue;
      }
      --x;
    }
    if (__ballot(op != 0) == 0) break;

    // one memory operation per lane
    const uint4* a1 = nullptr;
    const uint4* a2 = nullptr;
    uint32_t i1 = 0, i2 = 0, b1 = 0, b2 = 0;
    bool have1 = false;
    uint32_t tlen = gs::kPrecalc, tidx = p;  // table lookup: pattern length and entry
    uint32_t pbit = 64;  // presence bit of the clean 3 bases left of an extended window (64: none)
    if (op == 1) {
      a1 = reinterpret_cast<const uint4*>(P.X.kmer) + (p >> 1);  // two 8-byte entries per load
      if (P.X.ext_len && !ext_miss && e >= (int32_t)P.X.ext_len) {
        uint32_t q = p, ok = 1;
        for (uint32_t j = gs::kPrecalc; j < P.X.ext_len; ++j) {
          const uint32_t cj = V(e - 1 - (int32_t)j);
          ok &= cj <= 3 ? 1u : 0u;
          q |= (cj & 3u) << (2 * j);
        }
        if (ok) {
          tlen = P.X.ext_len;
          tidx = q;
          a1 = P.X.kext + q;
          if (k >= tlen + 3 && e >= (int32_t)tlen + 3) {
            const uint32_t c1 = V(e - (int32_t)tlen - 1), c2 = V(e - (int32_t)tlen - 2),
                           c3 = V(e - (int32_t)tlen - 3);
            if ((c1 | c2 | c3) <= 3) pbit = c1 + 4 * c2 + 16 * c3;
          }
        }
      }
    } else if (op == 2) {
      const uint32_t r1 = l - 1u;
      have1 = r1 != 0xFFFFFFFFu;
      i2 = gs::row_to_idx(u, P.X.primary);
      b2 = gs::div96(i2);
      i1 = have1 ? gs::row_to_idx(r1, P.X.primary) : 0u;
      b1 = gs::div96(i1);
      a1 = P.X.occ + (size_t)b2 * 4 + c;
      if (have1 && b1 != b2) a2 = P.X.occ + (size_t)b1 * 4 + c;
    }
    uint4 d1 = make_uint4(0, 0, 0, 0), d2;
    if (a1) d1 = *a1;
    d2 = d1;
    if (a2) d2 = *a2;

    if (op == 1) {
      const bool ext = tlen > gs::kPrecalc;
      const uint32_t il = ext ? d1.x : ((tidx & 1) ? d1.z : d1.x), iu = ext ? d1.y : ((tidx & 1) ? d1.w : d1.y);
      const bool absent = pbit < 64 && !(((pbit < 32 ? d1.z : d1.w) >> (pbit & 31)) & 1u);
      if (il > iu) {
        // absent clean tlen-base window: with k >= tlen the task can emit
        // nothing and ends (as in seed_persistent); else the 13-mer path decides
        if (ext && P.k < tlen)
          ext_miss = true;
        else if (!next_task())
          done = true;
      } else if (absent) {  // absent clean (tlen + 3)-base window, k >= tlen + 3: ends likewise
        if (!next_task()) done = true;
      } else {
        l = il;
        u = iu;
        s = u - l + 1;
        b = (uint32_t)e - tlen;
        if (prune_at((int32_t)b, s)) {
          if (!next_task()) done = true;
        } else {
          x = (int32_t)b - 1;
          phase = 1;
        }
      }
    } else if (op == 2) {
      const uint32_t o2 = gs::rank_in_entry(d1, i2 - b2 * gs::kBlockBases);
      const uint32_t o1 = have1 ? gs::rank_in_entry(d2, i1 - b1 * gs::kBlockBases) : 0u;
      const uint32_t base = P.X.L2[c];
      const uint32_t l2 = base + o1 + 1u, u2 = base + o2;
      if (l2 > u2) {
        finish();
        phase = 0;
        if (!next_task()) done = true;
      } else {
        l = l2;
        u = u2;
        s = u - l + 1;
        b = (uint32_t)x;
        if (prune_at(x, s)) {
          phase = 0;
          if (!next_task()) done = true;
        } else {
          --x;
        }
      }
    }
  }
  if (live) (strand == 0 ? P.nF : P.nR)[r] = nout;
}

// ---- finalisation ---------------------------------------------------------

struct PostParams {
  const uint4* cand;
  const uint32_t* nF;
  const uint32_t* nR;
  const uint64_t* task_off;
  const uint32_t* lens;
  const uint32_t* batch;  // reference batch of each read
  uint32_t n_reads, k, smem, max_occ;
  uint32_t* nseeds;       // count pass
  uint32_t* npos;
  const uint64_t* seed_off;  // write pass
  const uint64_t* pos_off;
  gs_seed_rec* seeds;
  uint32_t* rows;
  uint32_t per_wave;          // reads of a wave of finalize_reads
  uint32_t long_min;          // reads longer than this go to finalize_long
  uint32_t n_long;
  const uint32_t* long_reads;
};

struct ReadLists {
  const uint4* F;  // increasing qend
  const uint4* R;  // increasing qbeg
  uint32_t nF, nR;
};

__device__ __forceinline__ ReadLists lists_of(const PostParams& P, uint32_t r) {
  ReadLists Ls;
  const uint32_t L = P.lens[r];
  const uint32_t ntask = L >= P.k ? L - P.k + 1 : 0;
  const uint4* base = P.cand + 2 * P.task_off[r];
  Ls.nF = P.nF[r];
  Ls.nR = P.nR[r];
  Ls.F = base + ntask - Ls.nF;
  Ls.R = base + ntask;
  return Ls;
}

__device__ __forceinline__ uint32_t isize(uint4 c) { return c.w - c.z + 1u; }

// MEM filter (filter_seed_intervals_gpu_mem, 1103-1139): an entry is dropped
// when its neighbour towards the longer seed has the same qbeg/qend and size.
__device__ __forceinline__ bool mem_killed(const ReadLists& Ls, int rev, uint32_t i) {
  if (!rev) {
    const uint4 a = Ls.F[i];
    if (i + 1 >= Ls.nF) return false;
    const uint4 n = Ls.F[i + 1];
    return n.x == a.x && isize(n) == isize(a);
  }
  if (i == 0) return false;
  const uint4 a = Ls.R[i], pv = Ls.R[i - 1];
  return pv.y == a.y && isize(pv) == isize(a);
}

// rows an entry contributes (count_seed_intervals_gpu_mem, 927-989; in-read)
__device__ uint32_t mem_count(const ReadLists& Ls, int rev, uint32_t i) {
  if (mem_killed(Ls, rev, i)) return 0;
  const uint4 a = rev ? Ls.R[i] : Ls.F[i];
  const uint32_t sz = isize(a);
  if (!rev) {
    for (uint32_t j = i + 1; j < Ls.nF && Ls.F[j].x == a.x; ++j)
      if (!mem_killed(Ls, 0, j)) return sz - isize(Ls.F[j]);
  } else {
    for (uint32_t j = i; j-- > 0 && Ls.R[j].y == a.y;)
      if (!mem_killed(Ls, 1, j)) return sz - isize(Ls.R[j]);
  }
  return sz;
}

// interval whose rows an entry skips (seeds_to_threads_mem, 624-667): the next
// non-empty entry with the same qbeg (forward, scanning on) or qend (reverse,
// scanning back) anywhere in the same reference batch; (1, 0) if none.
__device__ uint2 mem_skip(const PostParams& P, uint32_t r, int rev, uint32_t i) {
  const ReadLists L0 = lists_of(P, r);
  const uint4 a = rev ? L0.R[i] : L0.F[i];
  uint2 skip = make_uint2(1, 0);
  const uint32_t bid = P.batch[r];
  if (!rev) {
    uint32_t rr = r;
    int part = 0;  // 0: F, 1: R
    uint32_t j = i + 1;
    while (rr < P.n_reads && P.batch[rr] == bid) {
      const ReadLists Ls = lists_of(P, rr);
      const uint32_t n = part == 0 ? Ls.nF : Ls.nR;
      if (j < n) {
        const uint4 en = part == 0 ? Ls.F[j] : Ls.R[j];
        if (en.x != a.x) break;
        if (!mem_killed(Ls, part, j)) {
          skip = make_uint2(en.z, en.w);
          break;
        }
        ++j;
        continue;
      }
      j = 0;
      if (part == 0) {
        part = 1;
      } else {
        part = 0;
        ++rr;
      }
    }
  } else {
    int64_t rr = r;
    int part = 1;
    int64_t j = (int64_t)i - 1;
    while (rr >= 0 && P.batch[rr] == bid) {
      const ReadLists Ls = lists_of(P, (uint32_t)rr);
      if (j >= 0) {
        const uint4 en = part == 0 ? Ls.F[j] : Ls.R[j];
        if (en.y != a.y) break;
        if (!mem_killed(Ls, part, (uint32_t)j)) {
          skip = make_uint2(en.z, en.w);
          break;
        }
        --j;
        continue;
      }
      if (part == 1) {
        part = 0;
        j = (int64_t)Ls.nF - 1;
      } else {
        --rr;
        if (rr < 0 || P.batch[rr] != bid) break;
        part = 1;
        j = (int64_t)lists_of(P, (uint32_t)rr).nR - 1;
      }
    }
  }
  return skip;
}

// the next entry of the merge: forward entries first on ties of qbeg (the
// stable segmented sort at 1233 and 3570)
__device__ __forceinline__ bool take_forward(const ReadLists& Ls, uint32_t a, uint32_t z) {
  return z >= Ls.nR || (a < Ls.nF && Ls.F[a].x <= (Ls.R[z].x & 0x7FFFFFFFu));
}

// A lane's part of the merged entries of read r: `left` of them, from forward
// entry a and reverse entry z on.
struct Part {
  ReadLists Ls;
  uint32_t r, a, z, left;
};

// The entry at the part's front: its list and index, its interval, and the
// rows it reports (none for an entry that is no seed, `seed` false; none for
// a seed over max_occ).
struct Entry {
  uint4 en;
  uint32_t i, cnt;
  int rev;
  bool seed;
};

__device__ __forceinline__ Entry take_entry(const PostParams& P, Part& p) {
  Entry e;
  e.rev = take_forward(p.Ls, p.a, p.z) ? 0 : 1;
  e.i = e.rev ? p.z++ : p.a++;
  --p.left;
  e.en = e.rev ? p.Ls.R[e.i] : p.Ls.F[e.i];
  const uint32_t sz = isize(e.en);
  e.cnt = P.smem ? sz : mem_count(p.Ls, e.rev, e.i);
  e.seed = e.cnt != 0;
  if (P.max_occ && sz > P.max_occ) e.cnt = 0;
  return e;
}

// Row i of the rows from z on that are not in [skip.x, skip.y].
__device__ __forceinline__ uint32_t nth_row(uint32_t z, uint2 skip, uint32_t i) {
  if (skip.x > skip.y || z > skip.y) return z + i;
  const uint32_t before = skip.x > z ? skip.x - z : 0u;
  return i < before ? z + i : skip.y + 1u + (i - before);
}

// seeds and positions of the part's entries
__device__ __forceinline__ void count_part(const PostParams& P, Part p, uint32_t& ns, uint32_t& np) {
  ns = np = 0;
  while (p.left) {
    const Entry e = take_entry(P, p);
    ns += e.seed ? 1u : 0u;
    np += e.cnt;
  }
}

// Entries with at least this many rows have them written by the whole wave.
constexpr uint32_t kWaveRows = 16;

// Writes the seed records of the lanes' parts from so on, and their rows from
// po on.  The lanes take an entry each per turn and write up to kWaveRows - 1
// rows of it themselves; the rows of an entry with more (as many as max_occ
// allows, or the whole of a repeat) are written by the wave, 64 at a time,
// one such entry after another: a lane that wrote them alone kept its wave
// waiting (300,007 MEM reads of up to 101 bases on a 100 Mbp index, max_occ
// 500: 2.09 ms), and finding the entry of each row among all lanes' takes 19
// shuffles per 64 rows (the same reads 0.17 ms, 0.16 with this; 1000 uneven
// reads 41 -> 17 us, 10,000 MEM reads with every row 82 -> 49 us).
// Reading the full suffix array here in place of locate_rows' pass was slower
// (1,000,000 reads on the 3.1 Gbp index 0.30 ms against 0.25, 60,000 uneven
// reads 0.40 against 0.29): its loads wait a turn each.
// Every lane of the wave takes part.
__device__ void write_parts(const PostParams& P, Part p, uint64_t so, uint64_t po) {
  const uint32_t lane = threadIdx.x & 63;
  while (__ballot(p.left != 0)) {
    uint32_t cnt = 0, z = 0;
    uint2 skip = make_uint2(1, 0);
    uint64_t dst = po;
    if (p.left) {
      const Entry e = take_entry(P, p);
      if (e.seed) {
        gs_seed_rec rec;
        rec.qbeg = e.en.x;
        rec.qend = e.en.y;
        rec.l = e.en.z;
        rec.u = e.en.w;
        rec.n_pos = e.cnt;
        rec.pad = 0;
        P.seeds[so++] = rec;
        cnt = e.cnt;
        z = e.en.z;
        po += cnt;
        if (cnt && !P.smem) skip = mem_skip(P, p.r, e.rev, e.i);
      }
    }
    if (cnt < kWaveRows)
      for (uint32_t i = 0; i < cnt; ++i) P.rows[dst + i] = nth_row(z, skip, i);
    for (uint64_t m = __ballot(cnt >= kWaveRows); m; m &= m - 1) {
      const int q = __ffsll((unsigned long long)m) - 1;
      const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cnt, q);
      const uint32_t zq = (uint32_t)__builtin_amdgcn_readlane((int)z, q);
      const uint2 sk = make_uint2((uint32_t)__builtin_amdgcn_readlane((int)skip.x, q),
                                  (uint32_t)__builtin_amdgcn_readlane((int)skip.y, q));
      const uint64_t at = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)dst, q) |
                          ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(dst >> 32), q) << 32);
      for (uint64_t i = lane; i < c; i += 64) P.rows[at + i] = nth_row(zq, sk, (uint32_t)i);
    }
  }
}

// Lane l's part of read r when the wave shares it: positions
// [l*T/64, (l+1)*T/64) of the merged order of the T = nF + nR entries; its
// starting split between the two lists is found by binary search on the merge
// path (the number a of forward entries among the first d merged is the
// smallest a at which forward entry a does not come before reverse entry
// d-a-1).
__device__ __forceinline__ Part shared_part(const PostParams& P, uint32_t r) {
  const uint32_t lane = threadIdx.x & 63;
  Part p;
  p.r = r;
  p.Ls = lists_of(P, r);
  const uint32_t T = p.Ls.nF + p.Ls.nR;
  const uint32_t d0 = (uint32_t)((uint64_t)T * lane / 64), d1 = (uint32_t)((uint64_t)T * (lane + 1) / 64);
  uint32_t lo = d0 > p.Ls.nR ? d0 - p.Ls.nR : 0, hi = d0 < p.Ls.nF ? d0 : p.Ls.nF;
  while (lo < hi) {
    const uint32_t a = (lo + hi) >> 1, b = d0 - a;
    if (b > 0 && p.Ls.F[a].x <= (p.Ls.R[b - 1].x & 0x7FFFFFFFu))
      lo = a + 1;  // forward entry a is merged before reverse entry b-1
    else
      hi = a;
  }
  p.a = lo;
  p.z = d0 - lo;
  p.left = d1 - d0;
  return p;
}

// One read by the whole wave: its counts (WRITE false), or its records and
// rows, each lane's from the scanned counts of the lanes before it.
template <bool WRITE>
__device__ __forceinline__ void finalize_shared(const PostParams& P, uint32_t r) {
  const uint32_t lane = threadIdx.x & 63;
  const Part p = shared_part(P, r);
  uint32_t ns, np;
  count_part(P, p, ns, np);
  // inclusive scans over the lanes (64-bit positions: a read's rows can
  // exceed 2^32 only through pathological counts, so sum in 64 bits)
  uint64_t sn = ns, sp = np;
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t tn = __shfl_up(sn, o, 64), tp = __shfl_up(sp, o, 64);
    if ((int)lane >= o) {
      sn += tn;
      sp += tp;
    }
  }
  if (!WRITE) {
    if (lane == 63) {
      P.nseeds[r] = (uint32_t)sn;
      P.npos[r] = (uint32_t)sp;
    }
  } else {
    write_parts(P, p, P.seed_off[r] + (sn - ns), P.pos_off[r] + (sp - np));
  }
}

// Reads with more merged entries than this are shared by the wave's lanes
// (MEM reads in repeats have up to two entries per base; counts and records
// of 200,000 MEM reads on the 3.1 Gbp index with 8, 16, 24 and 48: 0.68, 0.68,
// 0.71, 0.84 ms; 1,000,000 SMEM reads with 4, 16: 0.75, 0.43 ms).
constexpr uint32_t kSharedEntries = 16;

// Reads of a wave: fewer than 64 in small calls, whose few waves otherwise take
// their reads of many entries one after another (10,000 MEM reads: 157 waves;
// counts 30 -> 21 us, records with kWaveRows above 82 -> 49 us).
inline uint32_t reads_per_wave(uint64_t n) {
  return (uint32_t)std::min<uint64_t>(64, std::max<uint64_t>(8, (n + 4095) / 4096));
}

// A lane per read, then the wave together for each of its reads with many
// entries.  Count pass (WRITE false): seeds and positions per read.  Write
// pass: seed records and suffix-array rows at the scanned offsets.
template <bool WRITE>
__global__ void __launch_bounds__(256) finalize_reads(PostParams P) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t r = (blockIdx.x * 4 + (threadIdx.x >> 6)) * P.per_wave + lane;
  const bool mine = lane < P.per_wave && r < P.n_reads && !(P.lens[r] > P.long_min && P.lens[r] >= P.k);  // else finalize_long's
  Part p;
  p.r = r;
  p.a = p.z = p.left = 0;
  if (mine) {
    p.Ls = lists_of(P, r);
    p.left = p.Ls.nF + p.Ls.nR;
  }
  const uint64_t many = __ballot(p.left > kSharedEntries);
  const bool own = mine && p.left <= kSharedEntries;
  if (!own) p.left = 0;
  if (!WRITE) {
    uint32_t ns, np;
    count_part(P, p, ns, np);
    if (own) {
      P.nseeds[r] = ns;
      P.npos[r] = np;
    }
  } else {
    write_parts(P, p, own ? P.seed_off[r] : 0, own ? P.pos_off[r] : 0);
  }
  for (uint64_t m = many; m; m &= m - 1) {
    const uint32_t lead = (uint32_t)(__ffsll((unsigned long long)m) - 1);
    finalize_shared<WRITE>(P, (uint32_t)__builtin_amdgcn_readlane((int)r, (int)lead));
  }
}

// Reads longer than long_min bases (thousands of entries each): one wave per
// read.
template <bool WRITE>
__global__ void __launch_bounds__(256) finalize_long(PostParams P) {
  const uint32_t w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= P.n_long) return;
  finalize_shared<WRITE>(P, P.long_reads[w]);
}

// ---- exclusive scans of per-read counts into 64-bit offsets --------------
// Seeds and positions are scanned together, as are the five counts of a
// batch's plan (below), each in three launches: per-workgroup totals, a
// single-workgroup scan of those totals, then per-workgroup local scans offset
// by the scanned totals; in the last one alone where one workgroup holds all
// the reads.  (One scan of three launches per count made 24 of the 40 launches
// of a call of 1000 reads.)  Waves scan with shuffles; the workgroup combines
// its four wave totals in LDS.

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;  // per thread, fewer where one workgroup holds all the reads (ONE_TILE)
constexpr uint32_t kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ uint64_t wave_incl_scan(uint64_t v) {
  const int lane = threadIdx.x & 63;
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  return v;
}

// exclusive scan of v across the workgroup; returns the workgroup total in *tot
__device__ __forceinline__ uint64_t block_excl_scan(uint64_t v, uint64_t* tot) {
  __shared__ uint64_t wsum[kScanBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t inc = wave_incl_scan(v);
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  uint64_t before = 0, all = 0;
  for (int w = 0; w < kScanBlock / 64; ++w) {
    if (w < wid) before += wsum[w];
    all += wsum[w];
  }
  __syncthreads();
  *tot = all;
  return before + inc - v;
}

// NQ rows of ntiles totals, each scanned exclusively in place; row q's total
// to total[q] (total may be null)
template <int NQ>
__global__ void __launch_bounds__(kScanBlock) scan_tiles(uint64_t* __restrict__ tiles, uint64_t ntiles,
                                                         uint64_t* __restrict__ total) {
  for (int q = 0; q < NQ; ++q) {
    uint64_t* const row = tiles + q * ntiles;
    uint64_t carry = 0;
    for (uint64_t base = 0; base < ntiles; base += kScanBlock) {
      const uint64_t i = base + threadIdx.x;
      const uint64_t v = i < ntiles ? row[i] : 0;
      uint64_t tot;
      const uint64_t ex = block_excl_scan(v, &tot);
      if (i < ntiles) row[i] = carry + ex;
      carry += tot;
    }
    if (total && threadIdx.x == 0) total[q] = carry;
  }
}

// seeds and positions per read, scanned into their offsets
struct PairScan {
  const uint32_t* in[2];
  uint64_t* out[2];  // n + 1 entries each
  uint64_t n, ntiles;
  uint64_t* tiles;  // [2][ntiles]
  uint64_t* total;  // [2], pinned host memory
};

// the thread's ITEMS counts from `base` on (sum returned, each in v)
template <int ITEMS>
__device__ __forceinline__ uint64_t load_counts(const uint32_t* __restrict__ in, uint64_t n, uint64_t base,
                                                uint32_t* v) {
  uint64_t s = 0;
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    v[q] = base + q < n ? in[base + q] : 0u;
    s += v[q];
  }
  return s;
}

__global__ void __launch_bounds__(kScanBlock) pair_totals(PairScan S) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint32_t v[kScanItems];
    uint64_t tot;
    block_excl_scan(load_counts<kScanItems>(S.in[h], S.n, base, v), &tot);
    if (threadIdx.x == 0) S.tiles[h * S.ntiles + blockIdx.x] = tot;
  }
}

template <int ITEMS>
__global__ void __launch_bounds__(kScanBlock) pair_apply(PairScan S) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanBlock * ITEMS + threadIdx.x * ITEMS;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint32_t v[ITEMS];
    uint64_t tot;
    uint64_t run = block_excl_scan(load_counts<ITEMS>(S.in[h], S.n, base, v), &tot);
    if (S.ntiles == 1) {
      if (threadIdx.x == 0) S.total[h] = tot;
    } else {
      run += S.tiles[h * S.ntiles + blockIdx.x];
    }
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
      if (base + q < S.n) S.out[h][base + q] = run;
      run += v[q];
    }
    if (base + ITEMS >= S.n && base < S.n) S.out[h][S.n] = run;  // the thread holding the last item
  }
}

// ---- suffix-array walk (locate_seeds_gpu, 668-684) -------------------------
// R rows per thread, walked together so that their dependent lookups overlap;
// the rows of a thread are R grid-strides apart, so every load of a round is
// coalesced across the wave.
template <int R>
__global__ void __launch_bounds__(256) locate_rows(const DevIndex X, uint32_t* __restrict__ rows,
                                                   uint64_t n) {
  const uint64_t T = (uint64_t)gridDim.x * 256;
  const uint64_t t = blockIdx.x * 256ull + threadIdx.x;
  if (X.locate_direct) {
    // one load from the full suffix array per row; the rows whose reference
    // walk detours through row primary+1 report what that walk reports
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const uint64_t i = t + j * T;
      if (i >= n) continue;
      const uint32_t r = rows[i];
      uint32_t pos = 0xFFFFFFFFu;  // rows past the last one (MEM row skip) and row 0 ($) have none
      if (r != 0 && r <= X.seq_len) {
        pos = X.sa_full[r];
        for (uint32_t q = 0; q < X.n_quirk; ++q)
          if (X.quirk[q].x == r) pos = X.quirk[q].y;
      }
      rows[i] = pos;
    }
    return;
  }
  // A position is kept until the wave's last walk ends and then written with
  // the others': rows may lie in host memory, where a store per walk would
  // cross the link 4 bytes at a time.
  uint32_t row[R], itr[R], pos[R];
  uint32_t live = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint64_t i = t + j * T;
    row[j] = 0;
    itr[j] = 0;
    pos[j] = 0xFFFFFFFFu;
    if (i >= n) continue;
    row[j] = rows[i];
    // Rows past the last one come only from the reference's batch-wide MEM
    // row skip (seed_gen.cu:637/645) and have no position.
    if (row[j] <= X.seq_len) live |= 1u << j;
  }
  while (live) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (!(live & (1u << j))) continue;
      const uint32_t q = gs::div_sa(X, row[j]);
      if (row[j] == q * X.sa_intv) {
        pos[j] = X.sa[q] + itr[j];
        live &= ~(1u << j);
      } else if (itr[j] > X.seq_len) {  // a walk on a consistent index ends within seq_len + 1 steps
        live &= ~(1u << j);
      } else {
        ++itr[j];
        row[j] = gs::lf_walk(X, row[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (t + j * T < n) rows[t + j * T] = pos[j];
}

inline unsigned grid_for(uint64_t n, unsigned bs) { return (unsigned)((n + bs - 1) / bs); }

__global__ void zero_bytes(uint8_t* __restrict__ p, uint32_t n) {
  if (threadIdx.x < n) p[threadIdx.x] = 0;
}

// ---- work items of the persistent kernel, written at load time ---------------
// Whole-read streams (reads held whole in the LDS window) come first, two
// items per read (forward, reverse) in read order; then every read cut into
// segments, segment-major: items (read | seg << 33) and (read | 1 << 32 |
// seg << 33) for seg = 0..nseg-1, with the read in long_reads and its first
// item in item0.  A whole-read stream holds up to ~150 task ends and a
// segment at most seg_tasks, so the last items a persistent kernel hands
// out are the small ones.

// The rest of a batch's plan, from the reads' lengths: task and code-chunk
// offsets, the reads' offsets rebased onto the uploaded bytes, the
// reference-batch ids that MEM's row skip needs, and the work items (null
// code_off, items: not needed).
constexpr uint32_t kInlineCuts = 16;
struct PlanParams {
  uint64_t* offs;
  const uint32_t* lens;
  uint64_t n, lo;      // lo: subtracted from the offsets
  uint64_t n_whole;    // items of reads held whole
  uint32_t k, seg_tasks;
  // first reads of the second reference batch and of those after it: in `cut`
  // (at most kInlineCuts), or at `cuts`; batch null: not needed
  uint32_t* batch;
  const uint32_t* cuts;
  uint32_t n_cuts;
  uint32_t cut[kInlineCuts];
  uint64_t* toff;      // n + 1 entries, as code_off
  uint64_t* code_off;
  uint64_t* items;
  uint32_t* long_reads;
  uint64_t* item0;
  uint64_t* tiles;     // [kPlanSums][ntiles]
  uint64_t ntiles;
};
constexpr int kPlanSums = 5;

// a read's tasks, code chunks, items as a whole-read stream, items as
// segments, and 1 if it is segmented (0s past the last read)
__device__ __forceinline__ bool plan_counts(const PlanParams& P, uint64_t i, uint32_t& L, uint32_t* c) {
#pragma unroll
  for (int q = 0; q < kPlanSums; ++q) c[q] = 0;
  L = 0;
  if (i >= P.n) return false;
  L = P.lens[i];
  const uint32_t nseg = gs::n_segments(L, P.k, P.seg_tasks);
  const bool lng = gs::read_is_long(L, P.k, nseg);
  c[0] = L >= P.k ? L - P.k + 1 : 0u;
  c[1] = 2u * (L / 32u + (L % 32u ? 1u : 0u));
  c[lng ? 3 : 2] = 2u * nseg;
  c[4] = lng ? 1u : 0u;
  return lng;
}

__global__ void __launch_bounds__(kScanBlock) plan_totals(PlanParams P) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint64_t s[kPlanSums] = {0, 0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    uint32_t L, c[kPlanSums];
    plan_counts(P, base + j, L, c);
#pragma unroll
    for (int q = 0; q < kPlanSums; ++q) s[q] += c[q];
  }
#pragma unroll
  for (int q = 0; q < kPlanSums; ++q) {
    uint64_t tot;
    block_excl_scan(s[q], &tot);
    if (threadIdx.x == 0) P.tiles[q * P.ntiles + blockIdx.x] = tot;
  }
}

template <int ITEMS>
__global__ void __launch_bounds__(kScanBlock) plan_apply(PlanParams P) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanBlock * ITEMS + threadIdx.x * ITEMS;
  uint64_t s[kPlanSums] = {0, 0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    uint32_t L, c[kPlanSums];
    plan_counts(P, base + j, L, c);
#pragma unroll
    for (int q = 0; q < kPlanSums; ++q) s[q] += c[q];
  }
#pragma unroll
  for (int q = 0; q < kPlanSums; ++q) {
    uint64_t tot;
    s[q] = block_excl_scan(s[q], &tot) + (P.ntiles == 1 ? 0 : P.tiles[q * P.ntiles + blockIdx.x]);
  }
  for (int j = 0; j < ITEMS; ++j) {
    const uint64_t i = base + j;
    uint32_t L, c[kPlanSums];
    const bool lng = plan_counts(P, i, L, c);
    const uint64_t first = P.n_whole + s[3];
    if (i < P.n) {
      P.toff[i] = s[0];
      P.offs[i] -= P.lo;
      if (i + 1 == P.n) P.toff[P.n] = s[0] + c[0];
      if (P.code_off) {
        P.code_off[i] = s[1];
        if (i + 1 == P.n) P.code_off[P.n] = s[1] + c[1];
      }
      if (P.batch) {
        uint32_t id = 0;  // reference batches that start at or before read i
        if (P.cuts) {
          uint32_t hi = P.n_cuts;
          while (id < hi) {
            const uint32_t mid = (id + hi) >> 1;
            if (P.cuts[mid] <= i)
              id = mid + 1;
            else
              hi = mid;
          }
        } else {
          for (uint32_t q = 0; q < kInlineCuts; ++q) id += q < P.n_cuts && P.cut[q] <= i ? 1u : 0u;
        }
        P.batch[i] = id;
      }
      if (P.items) {
        if (!lng) {
          P.items[s[2]] = i;
          P.items[s[2] + 1] = i | (1ull << 32);
        } else {
          P.long_reads[s[4]] = (uint32_t)i;
          P.item0[s[4]] = first;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kPlanSums; ++q) s[q] += c[q];
  }
}

// A long read's items, a wave each (in plan_apply, whose one workgroup holds
// the reads of a small call, its waves wrote them one read after another: 60
// of 68 us for 1000 uneven reads).
__global__ void __launch_bounds__(256) plan_long_items(PlanParams P, uint32_t n_long) {
  const uint32_t w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= n_long) return;
  const uint32_t r = P.long_reads[w];
  const uint32_t n = 2u * gs::n_segments(P.lens[r], P.k, P.seg_tasks);
  uint64_t* const out = P.items + P.item0[w];
  for (uint32_t g = threadIdx.x & 63; g < n; g += 64)
    out[g] = (uint64_t)r | ((uint64_t)(g & 1u) << 32) | ((uint64_t)(g >> 1) << 33);
}

// ---- device buffers of one gs_seed call -------------------------------------
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  bool own = true;  // false: a view into memory this buffer must not free or replace
  void view(void* q, size_t bytes) {
    p = q;
    cap = bytes;
    own = false;
  }
  int ensure(size_t bytes) {
    if (bytes <= cap) return GS_OK;
    if (!own) return GS_ENOMEM;
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    size_t want = bytes + (bytes / 4 < (256u << 20) ? bytes / 4 : (256u << 20)) + 256;  // headroom for reuse
    if (hipMalloc(&p, want) != hipSuccess) return GS_ENOMEM;
    cap = want;
    return GS_OK;
  }
  template <typename T>
  T* as() const {
    return reinterpret_cast<T*>(p);
  }
  void release() {
    if (p && own) (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
  ~DevBuf() { release(); }
};

inline uint64_t scan_ntiles(uint64_t n) { return (n + kScanTile - 1) / kScanTile; }

// bytes of the tile totals of either scan over n reads
inline uint64_t scan_tile_bytes(uint64_t n) { return 8 * kPlanSums * (scan_ntiles(n) + 1); }

// The last launch of a scan: with as few items per thread as hold n reads in
// one workgroup (the threads' serial parts decide there: the plan of 64 reads
// 9.2 -> 3.3 us, of 1000 13 -> 7.8).
#define GS_ONE_TILE(kernel, n, tiles, st, ...)                                                   \
  do {                                                                                           \
    if ((n) <= kScanBlock)                                                                       \
      hipLaunchKernelGGL(kernel<1>, dim3(1), dim3(kScanBlock), 0, st, __VA_ARGS__);              \
    else if ((n) <= 4 * kScanBlock)                                                              \
      hipLaunchKernelGGL(kernel<4>, dim3(1), dim3(kScanBlock), 0, st, __VA_ARGS__);              \
    else                                                                                         \
      hipLaunchKernelGGL(kernel<kScanItems>, dim3((unsigned)(tiles)), dim3(kScanBlock), 0, st,   \
                         __VA_ARGS__);                                                           \
  } while (0)

void launch_pair_scan(PairScan S, hipStream_t st) {
  S.ntiles = scan_ntiles(S.n);
  if (!S.ntiles) return;
  if (S.ntiles > 1) {
    hipLaunchKernelGGL(pair_totals, dim3((unsigned)S.ntiles), dim3(kScanBlock), 0, st, S);
    hipLaunchKernelGGL(scan_tiles<2>, dim3(1), dim3(kScanBlock), 0, st, S.tiles, S.ntiles, S.total);
  }
  GS_ONE_TILE(pair_apply, S.n, S.ntiles, st, S);
}

void launch_plan(PlanParams P, uint32_t n_long, hipStream_t st) {
  P.ntiles = scan_ntiles(P.n);
  if (!P.ntiles) return;
  if (P.ntiles > 1) {
    hipLaunchKernelGGL(plan_totals, dim3((unsigned)P.ntiles), dim3(kScanBlock), 0, st, P);
    hipLaunchKernelGGL(scan_tiles<kPlanSums>, dim3(1), dim3(kScanBlock), 0, st, P.tiles, P.ntiles,
                       (uint64_t*)nullptr);
  }
  GS_ONE_TILE(plan_apply, P.n, P.ntiles, st, P);
  if (n_long && P.items) hipLaunchKernelGGL(plan_long_items, dim3((n_long + 3) / 4), dim3(256), 0, st, P, n_long);
}

// Arrays on their way to pinned host memory or back: copied by one launch, 16
// bytes per lane, at the link's rate where they are large.  A copy (and, to pageable
// memory, a wait) for each of six arrays cost small calls more than their
// bytes: 64 reads 484 -> 394 us per call, 100,000 plain 5.1 -> 4.45 ms.  Arrays are copied up to the next 16 bytes
// (every device buffer and slice here has that room behind it).
struct GatherParams {
  struct Segment {
    uint4* dst;
    const uint4* src;
    uint64_t end;  // 16-byte units up to this segment's last
  } seg[6];
  int n;
};

__global__ void __launch_bounds__(256) gather_arrays(GatherParams G) {
  const uint64_t units = G.seg[G.n - 1].end, step = gridDim.x * 256ull;
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < units; i += step) {
    uint64_t first = 0;
    for (int q = 0; q < G.n; ++q) {
      if (i < G.seg[q].end) {
        G.seg[q].dst[i - first] = G.seg[q].src[i - first];
        break;
      }
      first = G.seg[q].end;
    }
  }
}

// Device arrays (src) on their way to the caller's memory, laid end to end on
// 256 byte boundaries.
struct FetchParts {
  struct Part {
    void* dst;
    const void* src;
    size_t bytes, at;
  } part[6];
  int n = 0;
  size_t total = 0;
  void add(void* dst, const void* src, size_t bytes) {
    if (!bytes) return;
    part[n++] = {dst, src, bytes, total};
    total += (bytes + 255) & ~(size_t)255;
  }
  // f(part, offset in it, bytes, offset in all) for what lies in [a, z)
  template <typename F>
  void each(size_t a, size_t z, F&& f) const {
    for (int i = 0; i < n; ++i) {
      const Part& p = part[i];
      const size_t b = std::max(a, p.at), e = std::min(z, p.at + p.bytes);
      if (b < e) f(p, b - p.at, e - b, b);
    }
  }
  // what lies in [a, z), a a multiple of 256, to `stage` with one launch
  int launch_gather(size_t a, size_t z, char* stage, hipStream_t st) const { return launch(a, z, stage, false, st); }
  // the other way: from `stage` to the arrays
  int launch_scatter(size_t a, size_t z, char* stage, hipStream_t st) const { return launch(a, z, stage, true, st); }

 private:
  int launch(size_t a, size_t z, char* stage, bool scatter, hipStream_t st) const {
    GatherParams G;
    G.n = 0;
    uint64_t units = 0;
    each(a, z, [&](const Part& p, size_t o, size_t len, size_t at) {
      units += (len + 15) / 16;
      uint4* const device = reinterpret_cast<uint4*>(static_cast<char*>(const_cast<void*>(p.src)) + o);
      uint4* const host = reinterpret_cast<uint4*>(stage + (at - a));
      G.seg[G.n++] = {scatter ? device : host, scatter ? host : device, units};
    });
    if (!units) return GS_OK;
    const unsigned grid = (unsigned)std::min<uint64_t>((units + 255) / 256, 2048);
    hipLaunchKernelGGL(gather_arrays, dim3(grid), dim3(256), 0, st, G);
    return hipGetLastError() == hipSuccess ? GS_OK : GS_EHIP;
  }
};

template <typename AT, int LMAX>
void launch_seed(const SeedParams& P, hipStream_t st) {
  const uint64_t lanes = 2ull * P.n_reads;
  hipLaunchKernelGGL((seed_streams<AT, LMAX>), dim3(grid_for(lanes, kSeedBlock)), dim3(kSeedBlock), 0,
                     st, P);
}

}  // namespace

// ---- device-resident batches ------------------------------------------------

struct gs_batch {
  gs_index* X = nullptr;
  bool holds = false;  // keeps a reference to X (see batch_new)
  hipStream_t stream = nullptr;  // a batch's own stream: batches of one index may run concurrently
  gs_opts opts;
  uint64_t n_reads = 0, span = 0, tasks = 0;
  // gs_seed_noalloc, where the work items do not fit its array: seed_streams
  // instead of the persistent kernel (which needs maxlen and the read scratch)
  bool streams = false;
  uint32_t maxlen = 0;
  DevBuf bases, offs, lens, toff, batch, cand, nF, nR, ns, np, soff, poff, tiles, seeds, rows, scratch;
  DevBuf codes, code_off, queue, counters;  // persistent kernel
  DevBuf items, seg_meta, long_reads, item0, cuts;
  DevBuf seg_link, dyn_items, dyn_meta, dyn_link, wmeta, wlink;  // work splitting
  uint64_t code_chunks = 0, n_items = 0;
  uint32_t n_long = 0, seg_tasks = 64, dyn_cap = 0;
  uint64_t n_seeds = 0, n_pos = 0;
  bool ran = false;
  hipEvent_t ev[6] = {};
  hipEvent_t fev[2] = {};  // around a fetch's copies
  hipEvent_t lev[2] = {};  // around the upload and the plan
  hipEvent_t kev[2] = {};  // around the extension kernel's own launch (t_kernel)
  double t_h2d = 0;
  uint64_t* h_tot = nullptr;  // pinned: totals of the count stage
  // captured pipeline (gs_batch_capture) and its pinned staging
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  bool graph_fresh = false;
  uint64_t graph_seeds = 0, graph_pos = 0;
  char* hs_bases = nullptr;
  uint64_t* hs_offs = nullptr;
  uint32_t* hs_lens = nullptr;
  uint32_t *hr_ns = nullptr, *hr_np = nullptr, *hr_rows = nullptr;
  uint64_t *hr_soff = nullptr, *hr_poff = nullptr;
  gs_seed_rec* hr_seeds = nullptr;
  // pinned result staging of batch_download (grow-only; the server reuses it
  // round after round)
  struct Pinned {
    void* p = nullptr;
    size_t cap = 0;
    int ensure(size_t bytes) {
      if (bytes <= cap) return GS_OK;
      if (p) (void)hipHostFree(p);
      p = nullptr;
      cap = 0;
      const size_t want = bytes + bytes / 4 + 4096;
      if (hipHostMalloc(&p, want, hipHostMallocDefault) != hipSuccess) {
        p = nullptr;
        return GS_ENOMEM;
      }
      cap = want;
      return GS_OK;
    }
    void release() {
      if (p) (void)hipHostFree(p);
      p = nullptr;
      cap = 0;
    }
  };
  Pinned dl_ns, dl_np, dl_soff, dl_poff, dl_seeds, dl_pos;
  Pinned st_a, st_b;            // staged_d2h's two chunks
  hipEvent_t cev[2] = {};       // their copies' completion
};

static void free_graph(gs_batch* B);
static void free_host_results(gs_batch* B);

// Arrays of 4 MB and more on huge pages: the 4 KB page faults of a new array
// of that size cost more than filling it (107 MB of results, copied by one
// thread: 28 ms after a replay whose device work takes 11.6 ms).
void* gs::result_alloc(size_t bytes) {
  constexpr size_t kHuge = 2u << 20;
  if (bytes < 2 * kHuge) return malloc(bytes);
  const size_t whole = (bytes + kHuge - 1) & ~(kHuge - 1);
  void* p = aligned_alloc(kHuge, whole);
  if (p) (void)madvise(p, whole, MADV_HUGEPAGE);
  return p;
}

// Pinned chunks of staged uploads and downloads: two of them, the DMA of one
// under the host's copy of the other, so at least four chunks in a large copy.
constexpr size_t kStageChunk = 64u << 20, kStageChunkMin = 8u << 20;
static size_t stage_chunk(size_t total) {
  return std::min(total, std::max(kStageChunkMin, std::min(kStageChunk, (total / 4 + 4095) & ~(size_t)4095)));
}

// B's pinned chunks for `nch` chunks of `ch` bytes; false if there is no pinned
// memory for them.
static bool have_chunks(gs_batch* B, size_t ch, size_t nch) {
  if (!B->st_a.ensure(ch) && (nch < 2 || !B->st_b.ensure(ch))) return true;
  (void)hipGetLastError();  // not an error of the call
  return false;
}

static void destroy_batch(gs_batch* B) {
  if (!B) return;
  free_graph(B);
  free_host_results(B);
  for (auto* q : {&B->dl_ns, &B->dl_np, &B->dl_soff, &B->dl_poff, &B->dl_seeds, &B->dl_pos, &B->st_a, &B->st_b})
    q->release();
  for (auto& e : B->cev)
    if (e) (void)hipEventDestroy(e);
  if (B->h_tot) (void)hipHostFree(B->h_tot);
  for (auto& e : B->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto& e : B->lev)
    if (e) (void)hipEventDestroy(e);
  for (auto& e : B->fev)
    if (e) (void)hipEventDestroy(e);
  for (auto& e : B->kev)
    if (e) (void)hipEventDestroy(e);
  if (B->stream) (void)hipStreamDestroy(B->stream);
  gs_index* X = B->X;
  const bool holds = B->holds;
  delete B;
  if (holds) gs::index_release(X);
}

// ---- host plan of a batch -----------------------------------------------------
// What gs_batch_create derives on the CPU: the byte pieces to upload, the sizes
// of everything else and the first reads of the reference batches; the rest
// follows on the device (launch_plan).  A plan can hold several groups of
// reads (one per request of a server round); batch ids never span two groups.

int gs::plan_check(const gs_opts* o) {
  if (!o) return GS_EINVAL;
  if (o->k < gs::kPrecalc + 1 || o->k > 1 << 20) return GS_EINVAL;
  if (o->seg_tasks > gs::kSegTasksMax) return GS_EINVAL;
  if (o->wg != 0 && o->wg != 64 && o->wg != 128 && o->wg != 256) return GS_EINVAL;
  if (o->walk_rows != 0 && o->walk_rows != 1 && o->walk_rows != 2 && o->walk_rows != 4) return GS_EINVAL;
  if (o->kernel < 0 || o->kernel > 3) return GS_EINVAL;
  if (o->split_tasks > 64 && o->split_tasks != 0xFFFF) return GS_EINVAL;
  if (o->split_work == 0xFFFF) return GS_EINVAL;
  if (o->direct_min > 64 && o->direct_min != 0xFFFF) return GS_EINVAL;
  if (o->tandem > gs::kTandemMax && o->tandem != 0xFFFF) return GS_EINVAL;
  return GS_OK;
}

void gs::plan_reset(BatchPlan& P, const gs_opts& o) {
  P = BatchPlan();
  P.opts = o;
  P.seg_tasks = o.seg_tasks ? o.seg_tasks : 64u;
}

// Everything that a batch's sizes need, in one pass over the lengths; what
// else follows from them is computed on the device (launch_plan).
int gs::plan_add(BatchPlan& P, const char* bases, const uint64_t* offsets, const uint32_t* lens, uint64_t r0,
                 uint64_t r1) {
  if (r1 <= r0) return GS_OK;
  if (P.n_reads + (r1 - r0) > 0xFFFFFFFFull / 2) return GS_ERANGE;
  const uint32_t k = (uint32_t)P.opts.k;
  const uint32_t batch_bases = P.opts.batch_bases ? P.opts.batch_bases : 1000000u;
  // a group starts a reference batch of its own
  if (P.n_reads) P.cuts.push_back((uint32_t)P.n_reads);
  uint64_t lo = UINT64_MAX, hi = 0, acc = 0;
  ReadSums sum;
  bool closed = false;  // the read before this one closed its reference batch
  for (uint64_t i = r0; i < r1; ++i) {
    const uint32_t L = lens[i];
    if (closed) P.cuts.push_back((uint32_t)(P.n_reads + (i - r0)));
    acc += L;
    closed = acc >= batch_bases;  // a batch closes after the read that reaches the limit (2955-2991)
    if (closed) acc = 0;
    lo = std::min(lo, offsets[i]);
    hi = std::max(hi, offsets[i] + L);
    sum.add(L, k, P.seg_tasks);
  }
  if (hi < lo) lo = hi = 0;
  if (hi > lo) P.pieces.push_back({bases + lo, hi - lo});
  P.groups.push_back({offsets + r0, lens + r0, r1 - r0, lo, P.span});
  P.span += hi - lo;
  P.n_reads += r1 - r0;
  P.tasks += sum.tasks;
  P.code_chunks += sum.chunks;
  P.n_whole += sum.whole;
  P.n_items += sum.whole + sum.items;
  P.n_long += sum.n_long;
  return P.n_items > 0xF0000000ull ? GS_ERANGE : GS_OK;
}

// The reads' offsets and lengths as they are uploaded: the caller's own
// arrays where there is one group of reads and the plan need not outlive the
// call (copy false), else copies, their offsets rebased onto the groups'
// bytes, one after another.
void gs::plan_finish(BatchPlan& P, bool copy) {
  if (P.groups.size() < 2 && !copy) return;
  P.offs.reserve(P.n_reads);
  P.lens.reserve(P.n_reads);
  for (const auto& g : P.groups) {
    for (uint64_t i = 0; i < g.n; ++i) P.offs.push_back(g.offs[i] - g.lo + g.base);
    P.lens.insert(P.lens.end(), g.lens, g.lens + g.n);
  }
}

static gs::BatchSizes plan_sizes(const gs::BatchPlan& P) {
  const bool list = !P.opts.smem && P.cuts.size() > kInlineCuts;
  return {P.span, P.n_reads, P.tasks, P.code_chunks, P.n_items, P.n_long, list ? P.cuts.size() : 0,
          P.opts.split_tasks != 0xFFFF ? gs::piece_cap(P.n_items) : 0u};
}

uint64_t gs::plan_device_bytes(const BatchPlan& P) { return batch_bytes(plan_sizes(P)); }

static int batch_events(gs_batch* B) {
  if (!B->stream && hipStreamCreateWithFlags(&B->stream, hipStreamNonBlocking) != hipSuccess) return GS_EHIP;
  for (auto& e : B->ev)
    if (!e && hipEventCreate(&e) != hipSuccess) return GS_EHIP;
  for (auto& e : B->lev)
    if (!e && hipEventCreate(&e) != hipSuccess) return GS_EHIP;
  for (auto& e : B->fev)
    if (!e && hipEventCreate(&e) != hipSuccess) return GS_EHIP;
  for (auto& e : B->kev)
    if (!e && hipEventCreate(&e) != hipSuccess) return GS_EHIP;
  if (!B->h_tot && hipHostMalloc((void**)&B->h_tot, 16, hipHostMallocDefault) != hipSuccess) return GS_ENOMEM;
  return GS_OK;
}

// f(buffer, bytes) for the device buffers of a batch, those of work splitting
// last; stops where it returns something else than 0.
template <typename F>
static int each_buffer(const gs::BatchSizes& z, F&& f) {
  const uint64_t nr1 = z.n + 1;
  const struct {
    DevBuf gs_batch::*buf;
    uint64_t bytes;
  } all[] = {
      {&gs_batch::codes, 16 * (z.chunks + 1)},
      {&gs_batch::code_off, 8 * nr1},
      {&gs_batch::items, 8 * (z.items + 1)},
      {&gs_batch::long_reads, 4 * (z.n_long + 1)},
      {&gs_batch::item0, 8 * (z.n_long + 1)},
      {&gs_batch::seg_meta, z.n_long ? 16 * z.items : 16},
      {&gs_batch::seg_link, z.n_long ? 4 * z.items : 16},
      {&gs_batch::bases, z.span + 32},
      {&gs_batch::offs, 8 * nr1},
      {&gs_batch::lens, 4 * nr1},
      {&gs_batch::toff, 8 * nr1},
      {&gs_batch::batch, 4 * nr1},
      {&gs_batch::cuts, 4 * z.cuts},
      {&gs_batch::cand, 16 * (2 * z.tasks + 1)},
      {&gs_batch::nF, 4 * nr1},
      {&gs_batch::nR, 4 * nr1},
      {&gs_batch::ns, 4 * nr1},
      {&gs_batch::np, 4 * nr1},
      {&gs_batch::soff, 8 * nr1},
      {&gs_batch::poff, 8 * nr1},
      {&gs_batch::tiles, scan_tile_bytes(z.n)},
      {&gs_batch::queue, 16},
      {&gs_batch::counters, gs::kCounterBytes + gs::kColdBytes},
      {&gs_batch::dyn_items, 16ull * z.dyn_cap},
      {&gs_batch::dyn_meta, 16ull * z.dyn_cap},
      {&gs_batch::dyn_link, 4ull * z.dyn_cap},
      {&gs_batch::wmeta, z.dyn_cap ? 32 * nr1 : 0},
      {&gs_batch::wlink, z.dyn_cap ? 8 * nr1 : 0},
  };
  for (const auto& b : all)
    if (const int rc = f(b.buf, b.bytes)) return rc;
  return GS_OK;
}

uint64_t gs::batch_bytes(const BatchSizes& z) {
  uint64_t sum = 0;
  each_buffer(z, [&](DevBuf gs_batch::*, uint64_t bytes) {
    sum += bytes;
    return 0;
  });
  return sum;
}

// B's device buffers for these sizes; they only grow.
static int ensure_buffers(gs_batch* B, const gs::BatchSizes& z) {
  return each_buffer(z, [&](DevBuf gs_batch::*buf, uint64_t bytes) { return (B->*buf).ensure(bytes); });
}

// Where the device has no room for the pieces of work splitting, the batch
// runs without it, as with split_tasks 0xFFFF (large batches did without by
// default once, so a batch that fitted then still does).
static bool give_up_splitting(gs_batch* B) {
  if (!B->dyn_cap) return false;
  (void)hipGetLastError();  // not an error of the call
  B->dyn_cap = 0;
  for (auto* b : {&B->dyn_items, &B->dyn_meta, &B->dyn_link, &B->wmeta, &B->wlink}) b->release();
  return true;
}

int gs::batch_reserve(gs_batch* B, uint64_t bases, uint64_t reads, uint32_t seg_tasks) {
  if (!B) return GS_EINVAL;
  if (hipSetDevice(B->X->device) != hipSuccess) return GS_EHIP;
  if (!seg_tasks) seg_tasks = 64;
  // every read and long-read segment is an item of each strand; a read has
  // at most as many tasks as bases and code chunks as 32-base spans (+1)
  const uint64_t items = 2 * (reads + bases / seg_tasks + 1);
  // (and its reference batches are no more than the reads)
  const int rc = ensure_buffers(
      B, {bases, reads, bases, 2 * (bases / 32 + reads), items, reads, reads, gs::piece_cap(items)});
  if (!rc) {  // the pinned chunks of staged uploads, which do without where there are none
    const size_t up = bases + 12 * reads + 1024, ch = stage_chunk(up);
    (void)have_chunks(B, ch, ch < up ? 2 : 1);
  }
  return rc;
}

// Copies len bytes to dst by calling part(a, z) for disjoint ranges
// [a, z) of [0, len) on up to 8 threads (the calling thread takes the first
// part, and every part no thread could be started for).
template <typename F>
static void parallel_parts(size_t len, F&& part) {
  constexpr size_t kThreads = 8, kMinPart = 1u << 20;
  const size_t nt = std::max<size_t>(1, std::min(kThreads, len / kMinPart));
  const size_t each = (len + nt - 1) / nt;
  std::vector<std::thread> th;
  size_t done = std::min(len, each);  // bytes covered by this thread or started helpers
  try {
    for (size_t t = 1; t < nt; ++t) {
      const size_t a = std::min(len, t * each), z = std::min(len, a + each);
      th.emplace_back([=, &part] { part(a, z); });
      done = z;
    }
  } catch (...) {  // no thread to spare: this one copies the rest
  }
  part(0, std::min(len, each));
  if (done < len) part(done, len);
  for (auto& t : th) t.join();
}

// A batch's inputs on their way to the device: the reads' bytes (pieces, back
// to back, with 32 zero bytes behind them), offsets and lengths, each array on
// a 256 byte boundary.
struct UploadParts {
  struct Source {
    const char* p;
    size_t bytes, at;
  };
  std::vector<Source> from;  // in the order of `at`
  FetchParts to;             // src: the device array (dst unused)
  void source(const void* p, size_t bytes, size_t at) {
    if (bytes) from.push_back({static_cast<const char*>(p), bytes, at});
  }
  void array(void* device, const void* p, size_t bytes) {
    source(p, bytes, to.total);
    to.add(nullptr, device, bytes);
  }
  // every source by itself, from where it lies
  bool copy(hipStream_t st) const {
    bool ok = true;
    for (const Source& s : from)
      to.each(s.at, s.at + s.bytes, [&](const FetchParts::Part& p, size_t o, size_t len, size_t at) {
        ok = ok && hipMemcpyAsync(static_cast<char*>(const_cast<void*>(p.src)) + o, s.p + (at - s.at), len,
                                  hipMemcpyHostToDevice, st) == hipSuccess;
      });
    return ok;
  }
  // bytes [a, z) of the sources to dst
  void fill(size_t a, size_t z, char* dst) const {
    size_t lo = 0, hi = from.size();  // the first source that ends past a
    while (lo < hi) {
      const size_t mid = (lo + hi) / 2;
      if (from[mid].at + from[mid].bytes <= a)
        lo = mid + 1;
      else
        hi = mid;
    }
    for (; lo < from.size() && from[lo].at < z; ++lo) {
      const size_t b = std::max(a, from[lo].at), e = std::min(z, from[lo].at + from[lo].bytes);
      if (b < e) memcpy(dst + (b - a), from[lo].p + (b - from[lo].at), e - b);
    }
  }
};

// Through two pinned chunks: chunk c+1 is filled on several threads while
// chunk c is copied.  Pageable sources otherwise go through the runtime's own
// staging, an array after another, on one thread at a fraction of the link's
// rate.  Up to kScatterMax one launch reads them all (launch_scatter: a call
// of 10,000 reads 102 -> 70 us); larger ones are copied array by array, which
// reads host memory faster than that kernel (45 MB: 1.1 ms against 1.4).
// Without pinned memory the sources are copied from where they lie.
constexpr size_t kScatterMax = 2u << 20;
static int staged_upload(gs_batch* B, const UploadParts& U) {
  hipStream_t st = B->stream;
  const size_t total = U.to.total;
  if (!total) return GS_OK;
  const size_t ch = stage_chunk(total), nch = (total + ch - 1) / ch;
  if (!have_chunks(B, ch, nch)) return U.copy(st) ? GS_OK : GS_EHIP;
  for (auto& e : B->cev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return GS_EHIP;
  char* stage[2] = {static_cast<char*>(B->st_a.p), static_cast<char*>(B->st_b.p)};
  for (size_t c = 0; c < nch; ++c) {
    // the buffer of chunk c held chunk c-2, which must have been read
    if (c >= 2 && hipEventSynchronize(B->cev[c & 1]) != hipSuccess) return GS_EHIP;
    const size_t off = c * ch, len = std::min(ch, total - off);
    char* sp = stage[c & 1];
    parallel_parts(len, [&](size_t a, size_t z) { U.fill(off + a, off + z, sp + a); });
    if (total <= kScatterMax) {
      if (U.to.launch_scatter(off, off + len, sp, st)) return GS_EHIP;
    } else {
      bool ok = true;
      U.to.each(off, off + len, [&](const FetchParts::Part& p, size_t o, size_t m, size_t at) {
        ok = ok && hipMemcpyAsync(static_cast<char*>(const_cast<void*>(p.src)) + o, sp + (at - off), m,
                                  hipMemcpyHostToDevice, st) == hipSuccess;
      });
      if (!ok) return GS_EHIP;
    }
    if (c + 2 < nch && hipEventRecord(B->cev[c & 1], st) != hipSuccess) return GS_EHIP;
  }
  return GS_OK;
}

static const char kZeros[32] = {0};  // behind the reads' bytes: kernels read whole words of them

// B's part of a plan on the device (PP: lo, n_whole and the reference batches)
static void enqueue_plan(gs_batch* B, PlanParams PP, hipStream_t st) {
  PP.offs = B->offs.as<uint64_t>();
  PP.lens = B->lens.as<uint32_t>();
  PP.n = B->n_reads;
  PP.k = (uint32_t)B->opts.k;
  PP.seg_tasks = B->seg_tasks;
  PP.toff = B->toff.as<uint64_t>();
  PP.code_off = B->streams ? nullptr : B->code_off.as<uint64_t>();
  PP.items = B->streams ? nullptr : B->items.as<uint64_t>();
  PP.long_reads = B->long_reads.as<uint32_t>();
  PP.item0 = B->item0.as<uint64_t>();
  PP.tiles = B->tiles.as<uint64_t>();
  launch_plan(PP, B->n_long, st);
}

static void load_time(gs_batch* B) {
  float ms = 0;
  (void)hipEventElapsedTime(&ms, B->lev[0], B->lev[1]);
  B->t_h2d = ms * 1e-3;
}

// Uploads a finished plan into B, reusing B's device buffers where they are
// large enough.  B's results and any captured graph are dropped.  Without
// `wait` the plan and what it points at must stay as they are until the
// batch's stream has come this far (load_time then says how long it took).
int gs::batch_load(gs_batch* B, const BatchPlan& P, bool wait) {
  gs_index* X = B->X;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  int rc = batch_events(B);
  if (rc) return rc;
  free_graph(B);
  B->opts = P.opts;
  B->n_reads = P.n_reads;
  B->span = P.span;
  B->tasks = P.tasks;
  B->code_chunks = P.code_chunks;
  B->n_items = P.n_items;
  B->n_long = (uint32_t)P.n_long;
  B->seg_tasks = P.seg_tasks;
  B->n_seeds = B->n_pos = 0;
  B->ran = false;
  const uint64_t n = P.n_reads;
  BatchSizes z = plan_sizes(P);
  B->dyn_cap = z.dyn_cap;
  while (ensure_buffers(B, z)) {
    if (!give_up_splitting(B)) return GS_ENOMEM;
    z.dyn_cap = 0;
  }
  hipStream_t st = B->stream;
  if (hipEventRecord(B->lev[0], st) != hipSuccess) return GS_EHIP;
  const bool one = P.offs.empty();
  {
    UploadParts U;
    U.from.reserve(P.pieces.size() + 3);
    size_t at = 0;
    for (const auto& pc : P.pieces) {
      U.source(pc.first, pc.second, at);
      at += pc.second;
    }
    U.source(kZeros, sizeof kZeros, at);
    U.to.add(nullptr, B->bases.p, P.span + sizeof kZeros);
    if (n) {
      U.array(B->offs.p, one ? P.groups[0].offs : P.offs.data(), 8 * n);
      U.array(B->lens.p, one ? P.groups[0].lens : P.lens.data(), 4 * n);
    }
    if ((rc = staged_upload(B, U))) return rc;
  }
  if (n) {
    PlanParams PP{};
    PP.lo = one ? P.groups[0].lo : 0;
    PP.n_whole = P.n_whole;
    if (!P.opts.smem) {  // only MEM's row skip looks at the reference batches
      PP.batch = B->batch.as<uint32_t>();
      PP.n_cuts = (uint32_t)P.cuts.size();
      if (PP.n_cuts <= kInlineCuts) {
        std::copy(P.cuts.begin(), P.cuts.end(), PP.cut);
      } else {
        PP.cuts = B->cuts.as<uint32_t>();
        if (hipMemcpyAsync(B->cuts.p, P.cuts.data(), 4 * P.cuts.size(), hipMemcpyHostToDevice, st) != hipSuccess)
          return GS_EHIP;
      }
    }
    enqueue_plan(B, PP, st);
    if (hipGetLastError() != hipSuccess) return GS_EHIP;
  }
  if (hipEventRecord(B->lev[1], st) != hipSuccess) return GS_EHIP;
  if (wait) {
    if (hipStreamSynchronize(st) != hipSuccess) return GS_EHIP;
    load_time(B);
  }
  return GS_OK;
}

gs_batch* gs::batch_new(gs_index* X, bool hold) {
  gs_batch* B = new gs_batch();
  B->X = X;
  B->holds = hold;
  if (hold) gs::index_acquire(X);
  return B;
}

void gs::batch_free(gs_batch* B) { destroy_batch(B); }

extern "C" GS_API int gs_batch_create(gs_index* X, const char* bases, const uint64_t* offsets,
                                      const uint32_t* lens, uint64_t n_reads, const gs_opts* opts,
                                      gs_batch** out) {
  if (!X || !opts || !out || (n_reads && (!bases || !offsets || !lens))) return GS_EINVAL;
  *out = nullptr;
  int rc = gs::plan_check(opts);
  if (rc) return rc;
  if (n_reads > 0xFFFFFFFFull / 2) return GS_ERANGE;
  gs::BatchPlan P;
  gs::plan_reset(P, *opts);
  if ((rc = gs::plan_add(P, bases, offsets, lens, 0, n_reads))) return rc;
  gs::plan_finish(P);
  gs_batch* B = gs::batch_new(X);
  if ((rc = gs::batch_load(B, P))) {
    destroy_batch(B);
    return rc;
  }
  *out = B;
  return GS_OK;
}

// ---- the device pipeline of a batch -----------------------------------------
// Three stages on the index's stream: extension (pack, persistent kernel,
// segment join; or the plain kernel), counts (per-read counts, scans, totals
// to pinned host memory), records (seed records, SA rows, SA walk).  An eager
// run waits for the totals between counts and records to size the outputs; a
// captured graph replays all three with the sizes of the run before it.

static void fill_params(gs_batch* B, SeedParams& S, PostParams& Q) {
  gs_index* X = B->X;
  S.X = X->dev();
  S.bases = B->bases.as<uint8_t>();
  S.offs = B->offs.as<uint64_t>();
  S.lens = B->lens.as<uint32_t>();
  S.task_off = B->toff.as<uint64_t>();
  S.n_reads = (uint32_t)B->n_reads;
  S.k = (uint32_t)B->opts.k;
  S.smem = B->opts.smem ? 1 : 0;
  S.pad = 0;
  S.cand = B->cand.as<uint4>();
  S.nF = B->nF.as<uint32_t>();
  S.nR = B->nR.as<uint32_t>();
  S.scratch = B->scratch.p;
  Q.cand = S.cand;
  Q.nF = S.nF;
  Q.nR = S.nR;
  Q.task_off = S.task_off;
  Q.lens = S.lens;
  Q.batch = B->batch.as<uint32_t>();
  Q.n_reads = S.n_reads;
  Q.k = S.k;
  Q.smem = S.smem;
  Q.max_occ = B->opts.max_occ;
  Q.nseeds = B->ns.as<uint32_t>();
  Q.npos = B->np.as<uint32_t>();
  Q.seed_off = B->soff.as<uint64_t>();
  Q.pos_off = B->poff.as<uint64_t>();
  Q.seeds = B->seeds.as<gs_seed_rec>();
  Q.rows = B->rows.as<uint32_t>();
  // reads longer than the persistent kernel's window are finalized a wave each
  Q.per_wave = reads_per_wave(B->n_reads);
  Q.long_min = B->n_long ? gs::kPersistLmax : 0xFFFFFFFFu;
  Q.n_long = B->n_long;
  Q.long_reads = B->long_reads.as<uint32_t>();
}

// kev (null under graph capture): two events recorded on st right before and
// after the extension kernel itself, without the code packing, the queue's
// set-up and the join of split streams around it
static int enqueue_extension(gs_batch* B, const SeedParams& S, int kernel, unsigned pgrid, hipStream_t st,
                             hipEvent_t* kev = nullptr) {
  if (!B->n_reads) return GS_OK;
  if (B->streams) {
    if (B->maxlen <= 160)
      launch_seed<uint16_t, 160>(S, st);
    else
      launch_seed<uint16_t, 256>(S, st);
    return hipGetLastError() == hipSuccess ? GS_OK : GS_EHIP;
  }
  gs::PersistParams PP;
  PP.X = S.X;
  PP.bases = S.bases;
  PP.offs = S.offs;
  PP.codes = B->codes.as<uint4>();
  PP.code_off = B->code_off.as<uint64_t>();
  PP.lens = S.lens;
  PP.task_off = S.task_off;
  PP.items = B->items.as<uint64_t>();
  PP.n_items = B->n_items;
  PP.n_long = B->n_long;
  PP.k = S.k;
  PP.smem = S.smem;
  PP.seg_tasks = B->seg_tasks;
  PP.cand = S.cand;
  PP.nF = S.nF;
  PP.nR = S.nR;
  PP.seg_meta = B->seg_meta.as<uint4>();
  PP.seg_link = B->seg_link.as<uint32_t>();
  PP.queue = B->queue.as<uint32_t>();
  PP.counters = B->counters.as<uint64_t>();
  PP.direct_min = !S.X.isa || B->opts.direct_min == 0xFFFF ? 0u : (B->opts.direct_min ? B->opts.direct_min : 4u);
  PP.dyn_items = B->dyn_items.as<uint4>();
  PP.dyn_meta = B->dyn_meta.as<uint4>();
  PP.dyn_link = B->dyn_link.as<uint32_t>();
  PP.wmeta = B->wmeta.as<uint4>();
  PP.wlink = B->wlink.as<uint32_t>();
  PP.dyn_cap = B->dyn_cap;
  PP.split_tasks = B->opts.split_tasks;         // 0: by the launch's size
  PP.split_work = 64u * B->opts.split_work;  // 0: by the launch's size
  // tandem jumps read the index's tandem table
  const bool tandem = B->opts.tandem != 0xFFFF && B->X->tandem;
  PP.tandem = tandem ? (B->opts.tandem ? std::min<uint32_t>(B->opts.tandem, gs::kTandemMax) : gs::kTandemMax) : 0u;
  gs::JoinParams J;
  J.long_reads = B->long_reads.as<uint32_t>();
  J.item0 = B->item0.as<uint64_t>();
  J.lens = S.lens;
  J.task_off = S.task_off;
  J.seg_meta = PP.seg_meta;
  J.cand = S.cand;
  J.nF = S.nF;
  J.nR = S.nR;
  J.n_long = B->n_long;
  J.k = S.k;
  J.smem = S.smem;
  J.seg_tasks = B->seg_tasks;
  J.seg_link = PP.seg_link;
  J.dyn_items = PP.dyn_items;
  J.dyn_meta = PP.dyn_meta;
  J.dyn_link = PP.dyn_link;
  J.wmeta = PP.wmeta;
  J.wlink = PP.wlink;
  J.n_reads = S.n_reads;
  J.dyn_cap = PP.dyn_cap;
  int rc = GS_OK;
  if (kernel)  // the plain kernel reads the bytes
    rc = gs::launch_pack_codes(S.bases, S.offs, S.lens, PP.code_off, S.n_reads, J.long_reads, B->n_long,
                               B->codes.as<uint4>(), st);
  if (!rc) rc = gs::launch_persistent(PP, kernel - 1, B->opts.wg, pgrid, st, kev ? kev[0] : nullptr,
                                      kev ? kev[1] : nullptr);
  if (!rc) rc = gs::launch_join(J, st);
  return rc;
}

static int enqueue_counts(gs_batch* B, const PostParams& Q, hipStream_t st) {
  const uint64_t n = B->n_reads;
  if (n) {
    hipLaunchKernelGGL(finalize_reads<false>, dim3(grid_for(n, 4 * Q.per_wave)), dim3(256), 0, st, Q);
    if (Q.n_long) hipLaunchKernelGGL(finalize_long<false>, dim3((Q.n_long + 3) / 4), dim3(256), 0, st, Q);
    launch_pair_scan({{Q.nseeds, Q.npos}, {B->soff.as<uint64_t>(), B->poff.as<uint64_t>()}, n, 0,
                      B->tiles.as<uint64_t>(), B->h_tot}, st);
  } else {  // no reads: the offset arrays still hold their closing 0
    hipLaunchKernelGGL(zero_bytes, dim3(1), dim3(32), 0, st, B->soff.as<uint8_t>(), 8u);
    hipLaunchKernelGGL(zero_bytes, dim3(1), dim3(32), 0, st, B->poff.as<uint8_t>(), 8u);
  }
  return hipGetLastError() == hipSuccess ? GS_OK : GS_EHIP;
}

static int enqueue_write(gs_batch* B, const PostParams& Q, hipStream_t st) {
  if (B->n_reads) hipLaunchKernelGGL(finalize_reads<true>, dim3(grid_for(B->n_reads, 4 * Q.per_wave)), dim3(256), 0, st, Q);
  if (Q.n_long) hipLaunchKernelGGL(finalize_long<true>, dim3((Q.n_long + 3) / 4), dim3(256), 0, st, Q);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_EHIP;
}

// locate_rows over rows[0, n), R rows per thread, in launches of at most
// launch_chunk() rows (a dispatch's work-item count is a 32-bit quantity).
static void launch_locate(const DevIndex& X, uint32_t* rows, uint64_t n, unsigned R, hipStream_t st) {
  const uint64_t step = gs::launch_chunk();
  for (uint64_t first = 0; first < n; first += step) {
    const uint64_t m = n - first < step ? n - first : step;
    const unsigned grid = grid_for((m + R - 1) / R, 256);
    if (R == 4)
      hipLaunchKernelGGL(locate_rows<4>, dim3(grid), dim3(256), 0, st, X, rows + first, m);
    else if (R == 2)
      hipLaunchKernelGGL(locate_rows<2>, dim3(grid), dim3(256), 0, st, X, rows + first, m);
    else
      hipLaunchKernelGGL(locate_rows<1>, dim3(grid), dim3(256), 0, st, X, rows + first, m);
  }
}

static int enqueue_walk(gs_batch* B, const SeedParams& S, const PostParams& Q, hipStream_t st) {
  if (B->n_pos) launch_locate(S.X, Q.rows, B->n_pos, B->opts.walk_rows ? B->opts.walk_rows : 1u, st);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_EHIP;
}

static int persistent_grid_for(gs_batch* B, int kernel, unsigned* grid) {
  *grid = 0;
  if (B->streams || !B->n_reads) return GS_OK;
  return gs::persistent_grid(kernel - 1, B->opts.wg, grid);
}

// The whole device pipeline on an uploaded batch; results stay in HBM.  kev:
// record the extension kernel's own time; its end is waited for by the caller.
static int run_pipeline(gs_batch* B, int kernel, bool kev) {
  gs_index* X = B->X;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  hipStream_t st = B->stream;
  unsigned pgrid = 0;
  int rc = persistent_grid_for(B, kernel, &pgrid);
  if (rc) return rc;
  SeedParams S;
  PostParams Q;
  fill_params(B, S, Q);
  B->h_tot[0] = B->h_tot[1] = 0;
  GS_HIP(hipEventRecord(B->ev[0], st));
  rc = enqueue_extension(B, S, kernel, pgrid, st, kev ? B->kev : nullptr);
  if (rc) return rc;
  GS_HIP(hipEventRecord(B->ev[1], st));
  rc = enqueue_counts(B, Q, st);
  if (rc) return rc;
  GS_HIP(hipEventRecord(B->ev[2], st));
  GS_HIP(hipStreamSynchronize(st));
  B->n_seeds = B->h_tot[0];
  B->n_pos = B->h_tot[1];
  const void *seeds0 = B->seeds.p, *rows0 = B->rows.p;
  while (B->seeds.ensure(sizeof(gs_seed_rec) * (B->n_seeds + 1)) || B->rows.ensure(4 * (B->n_pos + 1))) {
    if (!give_up_splitting(B)) return GS_ENOMEM;
    free_graph(B);  // it splits
  }
  if (B->graph && (B->seeds.p != seeds0 || B->rows.p != rows0)) free_graph(B);  // it wrote the old buffers
  fill_params(B, S, Q);
  GS_HIP(hipEventRecord(B->ev[3], st));
  if ((rc = enqueue_write(B, Q, st))) return rc;
  GS_HIP(hipEventRecord(B->ev[4], st));
  if ((rc = enqueue_walk(B, S, Q, st))) return rc;
  GS_HIP(hipEventRecord(B->ev[5], st));
  B->ran = true;
  B->graph_fresh = false;
  return GS_OK;
}

// times and sizes of a run that has ended
static void run_stats(gs_batch* B, gs_batch_stats* stats) {
  float ms[5] = {0, 0, 0, 0, 0};
  (void)hipEventElapsedTime(&ms[0], B->ev[0], B->ev[1]);
  (void)hipEventElapsedTime(&ms[1], B->ev[1], B->ev[2]);
  (void)hipEventElapsedTime(&ms[2], B->ev[3], B->ev[4]);
  (void)hipEventElapsedTime(&ms[3], B->ev[4], B->ev[5]);
  (void)hipEventElapsedTime(&ms[4], B->ev[0], B->ev[5]);
  memset(stats, 0, sizeof(*stats));
  stats->t_h2d = B->t_h2d;
  stats->t_seed = ms[0] * 1e-3;
  stats->t_count = ms[1] * 1e-3;
  stats->t_write = ms[2] * 1e-3;
  stats->t_locate = ms[3] * 1e-3;
  stats->t_total = ms[4] * 1e-3;
  stats->n_reads = B->n_reads;
  stats->n_seeds = B->n_seeds;
  stats->n_pos = B->n_pos;
}

extern "C" GS_API int gs_batch_run(gs_batch* B, int kernel_override, gs_batch_stats* stats) {
  if (!B) return GS_EINVAL;
  const int kernel = kernel_override >= 0 ? kernel_override : B->opts.kernel;
  if (hipSetDevice(B->X->device) != hipSuccess) return GS_EHIP;
  if (kernel < 0 || kernel > 3) return GS_EINVAL;
  const int rc = run_pipeline(B, kernel, true);
  if (rc) return rc;
  if (hipStreamSynchronize(B->stream) != hipSuccess) {
    B->ran = false;
    return GS_EHIP;
  }
  if (stats) {
    run_stats(B, stats);
    float kms = 0;
    if (B->n_reads && hipEventElapsedTime(&kms, B->kev[0], B->kev[1]) == hipSuccess) stats->t_kernel = kms * 1e-3;
    if (kernel >= 1) {
      uint64_t c[4] = {0, 0, 0, 0};
      if (hipMemcpy(c, B->counters.p, 32, hipMemcpyDeviceToHost) == hipSuccess) {
        stats->n_table_reads = c[0];
        stats->n_occ_reads = c[1];
        stats->n_direct_reads = c[2];
        stats->n_tandem_reads = c[3];
      }
    }
  }
  return GS_OK;
}

static void free_graph(gs_batch* B) {
  if (B->gexec) (void)hipGraphExecDestroy(B->gexec);
  if (B->graph) (void)hipGraphDestroy(B->graph);
  B->gexec = nullptr;
  B->graph = nullptr;
  B->graph_fresh = false;
}

static void free_host_results(gs_batch* B) {
  for (void* p : {(void*)B->hr_ns, (void*)B->hr_np, (void*)B->hr_soff, (void*)B->hr_poff, (void*)B->hr_seeds,
                  (void*)B->hr_rows, (void*)B->hs_bases, (void*)B->hs_offs, (void*)B->hs_lens})
    if (p) (void)hipHostFree(p);
  B->hr_ns = B->hr_np = nullptr;
  B->hr_soff = B->hr_poff = nullptr;
  B->hr_seeds = nullptr;
  B->hr_rows = nullptr;
  B->hs_bases = nullptr;
  B->hs_offs = nullptr;
  B->hs_lens = nullptr;
}

// Captures upload -> extension -> counts -> records -> download as one graph.
extern "C" GS_API int gs_batch_capture(gs_batch* B, int kernel) {
  if (!B || !B->ran) return GS_EINVAL;
  const int kern = kernel >= 0 ? kernel : B->opts.kernel;
  if (kern < 0 || kern > 3) return GS_EINVAL;
  gs_index* X = B->X;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  hipStream_t st = B->stream;
  free_graph(B);
  free_host_results(B);
  const uint64_t n = B->n_reads, nr1 = n + 1;
  // pinned staging of the inputs and of the results, sized by the last run
  if (hipHostMalloc((void**)&B->hs_bases, B->span + 1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hs_offs, 8 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hs_lens, 4 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hr_ns, 4 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hr_np, 4 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hr_soff, 8 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hr_poff, 8 * nr1, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&B->hr_seeds, sizeof(gs_seed_rec) * (B->n_seeds + 1), hipHostMallocDefault) !=
          hipSuccess ||
      hipHostMalloc((void**)&B->hr_rows, 4 * (B->n_pos + 1), hipHostMallocDefault) != hipSuccess) {
    free_host_results(B);
    return GS_ENOMEM;
  }
  // the graph's upload nodes re-send the batch's resident inputs from these
  if ((B->span && hipMemcpyAsync(B->hs_bases, B->bases.p, B->span, hipMemcpyDeviceToHost, st) != hipSuccess) ||
      (n && (hipMemcpyAsync(B->hs_offs, B->offs.p, 8 * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
             hipMemcpyAsync(B->hs_lens, B->lens.p, 4 * n, hipMemcpyDeviceToHost, st) != hipSuccess)) ||
      hipStreamSynchronize(st) != hipSuccess) {
    free_host_results(B);
    return GS_EHIP;
  }
  unsigned pgrid = 0;
  int rc = persistent_grid_for(B, kern, &pgrid);
  if (rc) return rc;
  SeedParams S;
  PostParams Q;
  fill_params(B, S, Q);
  GS_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeGlobal));
  do {
    if ((B->span && hipMemcpyAsync(B->bases.p, B->hs_bases, B->span, hipMemcpyHostToDevice, st) != hipSuccess) ||
        (n && (hipMemcpyAsync(B->offs.p, B->hs_offs, 8 * n, hipMemcpyHostToDevice, st) != hipSuccess ||
               hipMemcpyAsync(B->lens.p, B->hs_lens, 4 * n, hipMemcpyHostToDevice, st) != hipSuccess))) {
      rc = GS_EHIP;
      break;
    }
    if ((rc = enqueue_extension(B, S, kern, pgrid, st))) break;
    if ((rc = enqueue_counts(B, Q, st))) break;
    if ((rc = enqueue_write(B, Q, st))) break;
    if ((rc = enqueue_walk(B, S, Q, st))) break;
    if ((n && (hipMemcpyAsync(B->hr_ns, B->ns.p, 4 * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
               hipMemcpyAsync(B->hr_np, B->np.p, 4 * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
               hipMemcpyAsync(B->hr_soff, B->soff.p, 8 * nr1, hipMemcpyDeviceToHost, st) != hipSuccess ||
               hipMemcpyAsync(B->hr_poff, B->poff.p, 8 * nr1, hipMemcpyDeviceToHost, st) != hipSuccess)) ||
        (B->n_seeds && hipMemcpyAsync(B->hr_seeds, B->seeds.p, sizeof(gs_seed_rec) * B->n_seeds,
                                      hipMemcpyDeviceToHost, st) != hipSuccess) ||
        (B->n_pos && hipMemcpyAsync(B->hr_rows, B->rows.p, 4 * B->n_pos, hipMemcpyDeviceToHost, st) != hipSuccess))
      rc = GS_EHIP;
  } while (0);
  hipGraph_t g = nullptr;
  const hipError_t ec = hipStreamEndCapture(st, &g);
  if (rc || ec != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return rc ? rc : GS_EHIP;
  }
  B->graph = g;
  if (hipGraphInstantiate(&B->gexec, g, nullptr, nullptr, 0) != hipSuccess) {
    free_graph(B);
    return GS_EHIP;
  }
  B->graph_seeds = B->n_seeds;
  B->graph_pos = B->n_pos;
  return GS_OK;
}

extern "C" GS_API int gs_batch_replay(gs_batch* B, gs_batch_stats* stats) {
  if (!B || !B->gexec) return GS_EINVAL;
  gs_index* X = B->X;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  hipStream_t st = B->stream;
  B->h_tot[0] = B->h_tot[1] = 0;
  GS_HIP(hipEventRecord(B->ev[0], st));
  GS_HIP(hipGraphLaunch(B->gexec, st));
  GS_HIP(hipEventRecord(B->ev[5], st));
  GS_HIP(hipStreamSynchronize(st));
  // the totals the graph copied back must be the sizes it was captured with
  if (B->n_reads && (B->h_tot[0] != B->graph_seeds || B->h_tot[1] != B->graph_pos)) return GS_ERANGE;
  B->n_seeds = B->graph_seeds;
  B->n_pos = B->graph_pos;
  B->graph_fresh = true;
  if (stats) {
    float ms = 0;
    (void)hipEventElapsedTime(&ms, B->ev[0], B->ev[5]);
    memset(stats, 0, sizeof(*stats));
    stats->t_total = ms * 1e-3;
    stats->n_reads = B->n_reads;
    stats->n_seeds = B->n_seeds;
    stats->n_pos = B->n_pos;
  }
  return GS_OK;
}

// Device-to-host copy into pageable memory through two pinned chunks: the DMA
// of chunk c+1 runs while chunk c is copied out, on several threads when it
// is large.  Pageable destinations otherwise go through the runtime's own
// staging at a fraction of the link's rate (and one array after another: a
// call of 1000 reads waited six times).  They do where there is no pinned
// memory; the caller waits for the stream.
static int staged_d2h(gs_batch* B, const FetchParts& P) {
  if (!P.total) return GS_OK;
  hipStream_t st = B->stream;
  const size_t ch = stage_chunk(P.total), nch = (P.total + ch - 1) / ch;
  if (!have_chunks(B, ch, nch)) {
    for (int i = 0; i < P.n; ++i)
      if (hipMemcpyAsync(P.part[i].dst, P.part[i].src, P.part[i].bytes, hipMemcpyDeviceToHost, st) != hipSuccess)
        return GS_EHIP;
    return GS_OK;
  }
  for (auto& e : B->cev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return GS_EHIP;
  char* stage[2] = {static_cast<char*>(B->st_a.p), static_cast<char*>(B->st_b.p)};
  auto issue = [&](size_t c) -> bool {
    const size_t off = c * ch;
    return P.launch_gather(off, std::min(P.total, off + ch), stage[c & 1], st) == GS_OK &&
           hipEventRecord(B->cev[c & 1], st) == hipSuccess;
  };
  if (!issue(0)) return GS_EHIP;
  for (size_t c = 0; c < nch; ++c) {
    // the buffer of chunk c+1 held chunk c-1, already copied out
    if (c + 1 < nch && !issue(c + 1)) return GS_EHIP;
    if (hipEventSynchronize(B->cev[c & 1]) != hipSuccess) return GS_EHIP;
    const size_t off = c * ch;
    const char* sp = stage[c & 1];
    parallel_parts(std::min(ch, P.total - off), [&](size_t a, size_t z) {
      P.each(off + a, off + z, [&](const FetchParts::Part& p, size_t o, size_t len, size_t at) {
        memcpy(static_cast<char*>(p.dst) + o, sp + (at - off), len);
      });
    });
  }
  return GS_OK;
}

extern "C" GS_API int gs_batch_fetch(gs_batch* B, gs_result* out) {
  if (!B || !out || !B->ran) return GS_EINVAL;
  memset(out, 0, sizeof(*out));
  if (hipSetDevice(B->X->device) != hipSuccess) return GS_EHIP;
  hipStream_t st = B->stream;
  const uint64_t n = B->n_reads, nr1 = n + 1;
  out->n_reads = n;
  out->n_seeds = B->n_seeds;
  out->n_pos = B->n_pos;
  out->read_nseeds = (uint32_t*)gs::result_alloc(4 * nr1);
  out->read_npos = (uint32_t*)gs::result_alloc(4 * nr1);
  out->read_seed_off = (uint64_t*)gs::result_alloc(8 * nr1);
  out->read_pos_off = (uint64_t*)gs::result_alloc(8 * nr1);
  out->seeds = (gs_seed_rec*)gs::result_alloc(sizeof(gs_seed_rec) * (B->n_seeds + 1));
  out->pos = (uint32_t*)gs::result_alloc(4 * (B->n_pos + 1));
  if (!out->read_nseeds || !out->read_npos || !out->read_seed_off || !out->read_pos_off || !out->seeds ||
      !out->pos) {
    gs_result_free(out);
    return GS_ENOMEM;
  }
  if (B->graph_fresh) {  // the last replay already downloaded everything
    FetchParts P;
    P.add(out->read_nseeds, B->hr_ns, 4 * n);
    P.add(out->read_npos, B->hr_np, 4 * n);
    if (n) {
      P.add(out->read_seed_off, B->hr_soff, 8 * nr1);
      P.add(out->read_pos_off, B->hr_poff, 8 * nr1);
    } else {
      out->read_seed_off[0] = out->read_pos_off[0] = 0;
    }
    P.add(out->seeds, B->hr_seeds, sizeof(gs_seed_rec) * B->n_seeds);
    P.add(out->pos, B->hr_rows, 4 * B->n_pos);
    parallel_parts(P.total, [&](size_t a, size_t z) {
      P.each(a, z, [&](const FetchParts::Part& p, size_t o, size_t len, size_t) {
        memcpy(static_cast<char*>(p.dst) + o, static_cast<const char*>(p.src) + o, len);
      });
    });
    return GS_OK;
  }
  hipEvent_t e0 = B->fev[0], e1 = B->fev[1];
  int rc = GS_OK;
  if (hipEventRecord(e0, st) != hipSuccess) rc = GS_EHIP;
  FetchParts P;
  P.add(out->read_nseeds, B->ns.p, 4 * n);
  P.add(out->read_npos, B->np.p, 4 * n);
  P.add(out->read_seed_off, B->soff.p, 8 * nr1);
  P.add(out->read_pos_off, B->poff.p, 8 * nr1);
  P.add(out->seeds, B->seeds.p, sizeof(gs_seed_rec) * B->n_seeds);
  P.add(out->pos, B->rows.p, 4 * B->n_pos);
  if (!rc) rc = staged_d2h(B, P);
  if (!rc && (hipEventRecord(e1, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)) rc = GS_EHIP;
  if (rc) {
    gs_result_free(out);
    return rc;
  }
  float ms = 0;
  (void)hipEventElapsedTime(&ms, e0, e1);
  out->t_d2h = ms * 1e-3;
  return GS_OK;
}

int gs::batch_download(gs_batch* B, ResultView* v) {
  if (!B || !v || !B->ran) return GS_EINVAL;
  if (hipSetDevice(B->X->device) != hipSuccess) return GS_EHIP;
  const uint64_t n = B->n_reads, nr1 = n + 1;
  if (B->dl_ns.ensure(4 * nr1) || B->dl_np.ensure(4 * nr1) || B->dl_soff.ensure(8 * nr1) ||
      B->dl_poff.ensure(8 * nr1) || B->dl_seeds.ensure(sizeof(gs_seed_rec) * (B->n_seeds + 1)) ||
      B->dl_pos.ensure(4 * (B->n_pos + 1)))
    return GS_ENOMEM;
  hipStream_t st = B->stream;
  if ((n && (hipMemcpyAsync(B->dl_ns.p, B->ns.p, 4 * n, hipMemcpyDeviceToHost, st) != hipSuccess ||
             hipMemcpyAsync(B->dl_np.p, B->np.p, 4 * n, hipMemcpyDeviceToHost, st) != hipSuccess)) ||
      hipMemcpyAsync(B->dl_soff.p, B->soff.p, 8 * nr1, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(B->dl_poff.p, B->poff.p, 8 * nr1, hipMemcpyDeviceToHost, st) != hipSuccess ||
      (B->n_seeds && hipMemcpyAsync(B->dl_seeds.p, B->seeds.p, sizeof(gs_seed_rec) * B->n_seeds,
                                    hipMemcpyDeviceToHost, st) != hipSuccess) ||
      (B->n_pos && hipMemcpyAsync(B->dl_pos.p, B->rows.p, 4 * B->n_pos, hipMemcpyDeviceToHost, st) != hipSuccess) ||
      hipStreamSynchronize(st) != hipSuccess)
    return GS_EHIP;
  v->n_reads = n;
  v->n_seeds = B->n_seeds;
  v->n_pos = B->n_pos;
  v->nseeds = static_cast<const uint32_t*>(B->dl_ns.p);
  v->npos = static_cast<const uint32_t*>(B->dl_np.p);
  v->soff = static_cast<const uint64_t*>(B->dl_soff.p);
  v->poff = static_cast<const uint64_t*>(B->dl_poff.p);
  v->seeds = static_cast<const gs_seed_rec*>(B->dl_seeds.p);
  v->pos = static_cast<const uint32_t*>(B->dl_pos.p);
  return GS_OK;
}

int gs_batch_set_tuning(gs_batch* B, int kernel, int wg, int walk_rows) {
  if (!B || kernel < 0 || kernel > 3 || (wg != 64 && wg != 128 && wg != 256) ||
      (walk_rows != 1 && walk_rows != 2 && walk_rows != 4))
    return GS_EINVAL;
  B->opts.kernel = kernel;
  B->opts.wg = (uint16_t)wg;
  B->opts.walk_rows = (uint16_t)walk_rows;
  return GS_OK;
}

// Text positions of suffix-array rows as the reference's walk reports them
// (locate_seeds_gpu, seed_gen.cu:668-684), with the same kernel as the
// pipeline (from the full suffix array when the index has it).  The kernel
// reads the rows from pinned chunks that the index keeps, and leaves the
// positions there: the host fills one while the device walks another's, and
// no device buffer is made and no array copied by the runtime (5,000,003 rows
// of a 100 Mbp index 2.53 -> 1.29 ms, of which walks 0.67).  Calls on one index
// follow each other, as their walks did on its stream before (8 threads, 5
// calls of 1,000,000 rows each: 24.0 -> 18.1 ms in all).  Without pinned
// memory the rows are copied to a device buffer and back; so they are where
// `out` starts inside the rows, whose later chunks its first ones would
// overwrite before they are read.
extern "C" GS_API int gs_index_locate(gs_index* X, const uint32_t* rows, uint64_t n, uint32_t* out) {
  if (!X || (n && (!rows || !out))) return GS_EINVAL;
  if (!n) return GS_OK;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  std::lock_guard<std::mutex> lk(X->locate_mu);
  if (!X->locate) X->locate = gs::batch_new(X, false);
  gs_batch* B = X->locate;  // only its pinned chunks and their events
  const size_t total = 4 * n, ch = stage_chunk(total);
  const uint64_t nch = (total + ch - 1) / ch;
  const uintptr_t r0 = (uintptr_t)rows, o0 = (uintptr_t)out;
  if ((o0 > r0 && o0 - r0 < total) || !have_chunks(B, ch, nch)) {
    uint32_t* d = nullptr;
    if (hipMalloc(&d, total) != hipSuccess) return GS_ENOMEM;
    bool ok = hipMemcpyAsync(d, rows, total, hipMemcpyHostToDevice, X->stream) == hipSuccess;
    if (ok) launch_locate(X->dev(), d, n, 1, X->stream);
    ok = ok && hipGetLastError() == hipSuccess &&
         hipMemcpyAsync(out, d, total, hipMemcpyDeviceToHost, X->stream) == hipSuccess;
    ok = hipStreamSynchronize(X->stream) == hipSuccess && ok;
    (void)hipFree(d);
    return ok ? GS_OK : GS_EHIP;
  }
  for (auto& e : B->cev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return GS_EHIP;
  char* const stage[2] = {static_cast<char*>(B->st_a.p), static_cast<char*>(B->st_b.p)};
  const DevIndex D = X->dev();
  auto copy_out = [&](uint64_t c) -> bool {
    if (hipEventSynchronize(B->cev[c & 1]) != hipSuccess) return false;
    const size_t off = c * ch;
    parallel_parts(std::min(ch, total - off), [&](size_t a, size_t z) {
      memcpy(reinterpret_cast<char*>(out) + off + a, stage[c & 1] + a, z - a);
    });
    return true;
  };
  bool ok = true;
  uint64_t done = 0, c = 0;  // chunks copied out, chunks launched
  for (; ok && c < nch; ++c) {
    if (c >= 2) {  // its buffer holds chunk c - 2
      ok = copy_out(c - 2);
      done = c - 1;
      if (!ok) break;
    }
    const size_t off = c * ch, len = std::min(ch, total - off);
    parallel_parts(len, [&](size_t a, size_t z) {
      memcpy(stage[c & 1] + a, reinterpret_cast<const char*>(rows) + off + a, z - a);
    });
    launch_locate(D, reinterpret_cast<uint32_t*>(stage[c & 1]), len / 4, 1, X->stream);
    ok = hipGetLastError() == hipSuccess && hipEventRecord(B->cev[c & 1], X->stream) == hipSuccess;
  }
  for (; ok && done < nch; ++done) ok = copy_out(done);
  if (!ok) (void)hipStreamSynchronize(X->stream);  // nothing may still write the chunks
  return ok ? GS_OK : GS_EHIP;
}

int gs_batch_set_direct_min(gs_batch* B, uint16_t direct_min) {
  if (!B || (direct_min > 64 && direct_min != 0xFFFF)) return GS_EINVAL;
  B->opts.direct_min = direct_min;
  return GS_OK;
}

extern "C" GS_API int gs_batch_destroy(gs_batch* B) {
  if (!B) return GS_EINVAL;
  (void)hipSetDevice(B->X->device);
  destroy_batch(B);
  return GS_OK;
}

// One batch from host memory to host memory: create, run, fetch.
extern "C" GS_API int gs_seed(gs_index* X, const char* bases, const uint64_t* offsets,
                              const uint32_t* lens, uint64_t n_reads, const gs_opts* opts,
                              gs_result* out) {
  if (!out) return GS_EINVAL;
  memset(out, 0, sizeof(*out));
  if (!X || !opts || (n_reads && (!bases || !offsets || !lens))) return GS_EINVAL;
  int rc = gs::plan_check(opts);
  if (rc) return rc;
  if (n_reads > 0xFFFFFFFFull / 2) return GS_ERANGE;
  gs::BatchPlan P;
  gs::plan_reset(P, *opts);
  if ((rc = gs::plan_add(P, bases, offsets, lens, 0, n_reads))) return rc;
  gs::plan_finish(P);
  // the index keeps this batch for the next call: its device buffers are
  // reused (no allocation, which would synchronise the device, once they fit)
  if (!X->work) X->work = gs::batch_new(X, false);
  gs_batch* B = X->work;
  // one stream from upload to fetch, waited for where the host needs the
  // sizes and the results (a wait after each stage, and the counters' copy,
  // made 0.1 ms of a call of 10,000 reads)
  rc = gs::batch_load(B, P, false);
  if (!rc) rc = run_pipeline(B, B->opts.kernel, false);
  if (!rc) rc = gs_batch_fetch(B, out);
  if (rc) {
    if (B->stream) (void)hipStreamSynchronize(B->stream);  // the caller's arrays may still be read
    B->ran = false;
  } else {
    load_time(B);
    gs_batch_stats s;
    run_stats(B, &s);
    out->t_h2d = s.t_h2d;
    out->t_seed = s.t_seed;
    out->t_post = s.t_count + s.t_write;
    out->t_locate = s.t_locate;
  }
  return rc;
}

extern "C" GS_API void gs_result_free(gs_result* r) {
  if (!r) return;
  free(r->read_nseeds);
  free(r->read_npos);
  free(r->read_seed_off);
  free(r->read_pos_off);
  free(r->seeds);
  free(r->pos);
  memset(r, 0, sizeof(*r));
}

// ---- gs_seed_noalloc: the same pipeline without any allocation --------------
// Every device buffer of the call is a slice of `scratch`, a file-scope array
// that each GPU holds from the library's load to the end of the process.  The
// host side keeps no vectors either: where the list of reference batches is
// long, the device finds them (noalloc_batch_ids).  Calls on one GPU share its
// array, so calls that overlap on one GPU race.

namespace {

constexpr uint64_t kNoAllocBytes = 256ull << 20;
constexpr int kNoAllocDevices = 64;

static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

// Small inputs and results of a call go through pinned memory that is set up
// with the scratch array, behind the call's totals.  Larger ones, and all of
// them where that memory could not be had, are copied from and to the caller's
// arrays.
constexpr size_t kNoAllocStage = 1u << 20, kNoAllocTotals = 256;

std::mutex g_scratch_mu;
char* g_scratch_stage[kNoAllocDevices];  // pinned, kNoAllocTotals + kNoAllocStage bytes (null: none yet)
void* g_scratch_ptr[kNoAllocDevices];  // device address of `scratch` on each device (null: not looked up)
int g_scratch_rc[kNoAllocDevices];     // the lookup's result once it has run

// Reference-batch id of every read: a batch closes after the read that
// brings it to batch_bases (seed_gen.cu:2955-2991), a running count with a
// reset.  One wave: the lanes load 64 lengths at a time and every lane
// follows the whole count, keeping the id of its own read.
__global__ void __launch_bounds__(64) noalloc_batch_ids(const uint32_t* __restrict__ lens, uint32_t n,
                                                        uint32_t batch_bases, uint32_t* __restrict__ batch) {
  const uint32_t lane = threadIdx.x;
  uint32_t id = 0;
  uint64_t acc = 0;
  for (uint32_t base = 0; base < n; base += 64) {
    const uint32_t i = base + lane;
    const uint32_t L = i < n ? lens[i] : 0u;
    const uint32_t m = n - base < 64u ? n - base : 64u;
    uint32_t mine = 0;
    for (uint32_t j = 0; j < m; ++j) {
      const uint32_t Lj = (uint32_t)__shfl((int)L, (int)j, 64);
      if (lane == j) mine = id;
      acc += Lj;
      if (acc >= batch_bases) {
        ++id;
        acc = 0;
      }
    }
    if (i < n) batch[i] = mine;
  }
}

inline uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

}  // namespace

// Looks up this device's copy of `scratch` (the current device must be
// `device`); called where an index is set up on a device.
int gs::noalloc_setup(int device) {
  if (device < 0 || device >= kNoAllocDevices) return GS_EINVAL;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    if (g_scratch_rc[device]) return g_scratch_rc[device];
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      g_scratch_rc[device] = GS_EHIP;
      return GS_EHIP;
    }
    g_scratch_ptr[device] = p;
  }
  if (!g_scratch_stage[device]) {
    void* stage = nullptr;
    if (hipHostMalloc(&stage, kNoAllocTotals + kNoAllocStage, hipHostMallocDefault) == hipSuccess)
      g_scratch_stage[device] = static_cast<char*>(stage);
    else
      (void)hipGetLastError();  // calls do without; the next index on the device asks again
  }
  return GS_OK;
}

extern "C" GS_API int gs_seed_noalloc(gs_index* X, const char* bases, const uint64_t* offsets,
                                      const uint32_t* lens, uint64_t n_reads, const gs_opts* opts,
                                      gs_result_buffers* out) {
  if (!X || !opts || !out || (n_reads && (!bases || !offsets || !lens))) return GS_EINVAL;
  if (!out->read_seed_off || !out->read_pos_off || (n_reads && (!out->read_nseeds || !out->read_npos)))
    return GS_EINVAL;
  out->n_seeds = out->n_pos = 0;
  int rc = gs::plan_check(opts);
  if (rc) return rc;
  if (n_reads > 0xFFFFFFFFull / 2) return GS_ERANGE;
  const uint32_t n = (uint32_t)n_reads, k = (uint32_t)opts->k;
  const uint32_t seg_tasks = opts->seg_tasks ? opts->seg_tasks : 64u;
  // sizes from the lengths alone (one pass, nothing allocated)
  const uint32_t batch_bases = opts->batch_bases ? opts->batch_bases : 1000000u;
  uint64_t lo = UINT64_MAX, hi = 0, tasks = 0, chunks = 0, n_items = 0, n_whole = 0, n_long = 0, acc = 0;
  uint32_t maxlen = 0, n_cuts = 0, cut[kInlineCuts];
  bool closed = false;  // the read before this one closed its reference batch
  for (uint32_t i = 0; i < n; ++i) {
    const uint32_t L = lens[i];
    if (closed && n_cuts <= kInlineCuts) {
      if (n_cuts < kInlineCuts) cut[n_cuts] = i;
      ++n_cuts;
    }
    acc += L;
    closed = acc >= batch_bases;
    if (closed) acc = 0;
    if (offsets[i] < lo) lo = offsets[i];
    if (offsets[i] + L > hi) hi = offsets[i] + L;
    tasks += L >= k ? L - k + 1 : 0;
    chunks += 2 * ((L + 31) / 32);
    const uint32_t nseg = gs::n_segments(L, k, seg_tasks);
    if (gs::read_is_long(L, k, nseg))
      ++n_long;
    else
      n_whole += 2ull * nseg;
    n_items += 2ull * nseg;
    if (L > maxlen) maxlen = L;
  }
  if (hi < lo) lo = hi = 0;
  const uint64_t span = hi - lo, nr1 = (uint64_t)n + 1;

  // Slices of the scratch array, in order.  What a call may hold is set by
  // its first layout: reads of at most 160 bases with a batched kernel need
  // their codes and two work items each, every other call the plain kernel
  // seed_streams, which needs none, but for reads of more than 256 bases a
  // size record per base and strand; the outputs come after that.  (o_spare held
  // the tile totals of an earlier scan; it stays, so that the largest call that
  // fits is the same.)
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    const uint64_t o = at;
    at = align256(at + bytes);
    return o;
  };
  const bool short_batched = opts->kernel != 0 && maxlen <= gs::kPersistLmax;
  const bool long_scratch = !short_batched && maxlen > 256;
  const uint64_t o_bases = take(span + 32), o_offs = take(8 * nr1), o_lens = take(4 * nr1),
                 o_toff = take(8 * nr1), o_batch = take(4 * nr1), o_cand = take(16 * (2 * tasks + 1)),
                 o_nF = take(4 * nr1), o_nR = take(4 * nr1), o_ns = take(4 * nr1), o_np = take(4 * nr1),
                 o_soff = take(8 * nr1), o_poff = take(8 * nr1), o_spare = take(8 * (nr1 / kScanTile + 2)),
                 o_tot = take(16), o_queue = take(16), o_counters = take(gs::kCounterBytes + gs::kColdBytes);
  (void)o_spare;
  const uint64_t common = at;
  const uint64_t o_code_off = take(8 * nr1), o_long = long_scratch ? take(4 * (span + 16)) : 0;
  if (short_batched) {
    take(16ull * n + 8);
    take(16 * (chunks + 1));
  }
  if (at > kNoAllocBytes) return GS_ERANGE;
  const uint64_t fixed = at;
  // What runs: the kernel that gs_seed would run, if its buffers fit too
  // (work items, segments of long reads; a call of reads longer than 160
  // bases takes the place of the size records for them), else seed_streams.
  // Everything from `out_at` on is dead once the streams are joined, and the
  // outputs, written after that, take its place (out_at <= fixed: the list of
  // long reads is no larger than the code offsets).
  at = common;
  const uint64_t o_long_reads = take(4 * (n_long + 1)), out_at = at;
  const uint64_t o_code_off2 = take(8 * nr1);
  const bool kernel_codes = opts->kernel != 0;
  const uint64_t o_items = take(8 * (n_items + 1)), o_codes = kernel_codes ? take(16 * (chunks + 1)) : 0,
                 o_tiles2 = take(scan_tile_bytes(n)), o_item0 = take(8 * (n_long + 1)), o_seg_meta = n_long ? take(16 * n_items) : 0;
  const bool streams = at > kNoAllocBytes;
  const uint32_t cap = streams || opts->split_tasks == 0xFFFF ? 0u : gs::piece_cap(n_items);
  const uint64_t o_ditems = take(16ull * cap), o_dmeta = take(16ull * cap), o_dlink = take(4ull * cap),
                 o_wmeta = take(32 * nr1), o_wlink = take(8 * nr1), o_seg_link = n_long ? take(4 * n_items) : 0;
  const bool split_on = cap && at <= kNoAllocBytes;
  const int kernel = streams ? 0 : opts->kernel;

  if (X->device < 0 || X->device >= kNoAllocDevices) return GS_EINVAL;
  if (hipSetDevice(X->device) != hipSuccess) return GS_EHIP;
  uint8_t* base = nullptr;
  char* stage = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    base = static_cast<uint8_t*>(g_scratch_ptr[X->device]);
    stage = g_scratch_stage[X->device];
  }
  if (!base) return GS_EHIP;  // the lookup at set-up failed
  hipStream_t st = X->stream;

  // a batch whose buffers are views into the scratch array; it owns nothing
  gs_batch B;
  B.X = X;
  B.stream = st;
  B.opts = *opts;
  B.opts.kernel = kernel;
  B.n_reads = n;
  B.span = span;
  B.tasks = tasks;
  B.maxlen = maxlen;
  B.code_chunks = chunks;
  B.streams = streams;
  B.n_items = streams ? 0 : n_items;
  B.n_long = streams ? 0 : (uint32_t)n_long;
  B.seg_tasks = seg_tasks;
  B.dyn_cap = split_on ? cap : 0u;
  if (!streams) {
    B.items.view(base + o_items, 8 * (n_items + 1));
    if (kernel_codes) B.codes.view(base + o_codes, 16 * (chunks + 1));
    B.long_reads.view(base + o_long_reads, 4 * (n_long + 1));
    B.item0.view(base + o_item0, 8 * (n_long + 1));
    if (n_long) B.seg_meta.view(base + o_seg_meta, 16 * n_items);
  }
  if (split_on) {
    B.dyn_items.view(base + o_ditems, 16ull * cap);
    B.dyn_meta.view(base + o_dmeta, 16ull * cap);
    B.dyn_link.view(base + o_dlink, 4ull * cap);
    B.wmeta.view(base + o_wmeta, 32 * nr1);
    B.wlink.view(base + o_wlink, 8 * nr1);
    if (n_long) B.seg_link.view(base + o_seg_link, 4 * n_items);
  }
  // the totals: written to pinned memory by the scan, else copied
  uint64_t sums[2] = {0, 0};
  uint64_t* const h_tot = stage ? reinterpret_cast<uint64_t*>(stage) : sums;
  h_tot[0] = h_tot[1] = 0;
  B.h_tot = stage ? h_tot : reinterpret_cast<uint64_t*>(base + o_tot);
  const size_t stage_bytes = stage ? kNoAllocStage : 0;
  if (stage) stage += kNoAllocTotals;
  B.bases.view(base + o_bases, span + 32);
  B.offs.view(base + o_offs, 8 * nr1);
  B.lens.view(base + o_lens, 4 * nr1);
  B.toff.view(base + o_toff, 8 * nr1);
  B.batch.view(base + o_batch, 4 * nr1);
  B.code_off.view(base + (streams ? o_code_off : o_code_off2), 8 * nr1);
  B.cand.view(base + o_cand, 16 * (2 * tasks + 1));
  B.nF.view(base + o_nF, 4 * nr1);
  B.nR.view(base + o_nR, 4 * nr1);
  B.ns.view(base + o_ns, 4 * nr1);
  B.np.view(base + o_np, 4 * nr1);
  B.soff.view(base + o_soff, 8 * nr1);
  B.poff.view(base + o_poff, 8 * nr1);
  // the scans' tile totals: with seed_streams in place of the code offsets it
  // does not read (40 bytes per 2048 reads, 8 per read)
  B.tiles.view(base + (streams ? o_code_off : o_tiles2), scan_tile_bytes(n));
  B.queue.view(base + o_queue, 16);
  B.counters.view(base + o_counters, gs::kCounterBytes + gs::kColdBytes);
  if (streams && long_scratch) B.scratch.view(base + o_long, 4 * (span + 16));

  // inputs, then the plan on the device
  FetchParts in;
  in.add(nullptr, B.bases.p, span + sizeof kZeros);
  in.add(nullptr, B.offs.p, 8ull * n);
  in.add(nullptr, B.lens.p, 4ull * n);
  if (in.total <= stage_bytes) {
    if (span) memcpy(stage, bases + lo, span);
    memcpy(stage + span, kZeros, sizeof kZeros);
    if (n) memcpy(stage + in.part[1].at, offsets, 8ull * n);
    if (n) memcpy(stage + in.part[2].at, lens, 4ull * n);
    if ((rc = in.launch_scatter(0, in.total, stage, st))) return rc;
  } else {
    if ((span && hipMemcpyAsync(B.bases.p, bases + lo, span, hipMemcpyHostToDevice, st) != hipSuccess) ||
        (n && (hipMemcpyAsync(B.offs.p, offsets, 8ull * n, hipMemcpyHostToDevice, st) != hipSuccess ||
               hipMemcpyAsync(B.lens.p, lens, 4ull * n, hipMemcpyHostToDevice, st) != hipSuccess)))
      return GS_EHIP;
    hipLaunchKernelGGL(zero_bytes, dim3(1), dim3(32), 0, st, B.bases.as<uint8_t>() + span, 32u);
  }
  if (n) {
    PlanParams PP{};
    PP.lo = lo;
    PP.n_whole = n_whole;
    if (!opts->smem) {
      if (n_cuts <= kInlineCuts) {
        PP.batch = B.batch.as<uint32_t>();
        PP.n_cuts = n_cuts;
        std::copy(cut, cut + n_cuts, PP.cut);
      } else {  // no room for the list: a running count on the device
        hipLaunchKernelGGL(noalloc_batch_ids, dim3(1), dim3(64), 0, st, B.lens.as<uint32_t>(), n, batch_bases,
                           B.batch.as<uint32_t>());
      }
    }
    enqueue_plan(&B, PP, st);
  }
  if (hipGetLastError() != hipSuccess) return GS_EHIP;

  // extension and counts, as gs_batch_run
  unsigned pgrid = 0;
  if ((rc = persistent_grid_for(&B, kernel, &pgrid))) return rc;
  SeedParams S;
  PostParams Q;
  fill_params(&B, S, Q);
  if ((rc = enqueue_extension(&B, S, kernel, pgrid, st))) return rc;
  if ((rc = enqueue_counts(&B, Q, st))) return rc;
  if (n && !stage) GS_HIP(hipMemcpyAsync(sums, B.h_tot, sizeof sums, hipMemcpyDeviceToHost, st));
  GS_HIP(hipStreamSynchronize(st));
  const uint64_t n_seeds = n ? h_tot[0] : 0, n_pos = n ? h_tot[1] : 0;
  out->n_seeds = n_seeds;
  out->n_pos = n_pos;
  const uint64_t seeds_bytes = align256(sizeof(gs_seed_rec) * (n_seeds + 1));
  if (fixed + seeds_bytes + 4 * (n_pos + 1) > kNoAllocBytes) return GS_ERANGE;
  const uint64_t o_seeds = streams ? fixed : out_at, o_rows = o_seeds + seeds_bytes;
  if (n_seeds > out->seeds_cap || n_pos > out->pos_cap || (n_seeds && !out->seeds) || (n_pos && !out->pos))
    return GS_ERANGE;  // n_seeds and n_pos say what the call needs
  B.n_seeds = n_seeds;
  B.n_pos = n_pos;
  B.seeds.view(base + o_seeds, sizeof(gs_seed_rec) * (n_seeds + 1));
  B.rows.view(base + o_rows, 4 * (n_pos + 1));
  fill_params(&B, S, Q);
  if ((rc = enqueue_write(&B, Q, st))) return rc;
  if ((rc = enqueue_walk(&B, S, Q, st))) return rc;
  FetchParts P;
  P.add(out->read_nseeds, B.ns.p, 4ull * n);
  P.add(out->read_npos, B.np.p, 4ull * n);
  P.add(out->read_seed_off, B.soff.p, 8 * nr1);
  P.add(out->read_pos_off, B.poff.p, 8 * nr1);
  P.add(out->seeds, B.seeds.p, sizeof(gs_seed_rec) * n_seeds);
  P.add(out->pos, B.rows.p, 4 * n_pos);
  const bool staged = P.total <= stage_bytes;
  if (staged) {
    if ((rc = P.launch_gather(0, P.total, stage, st))) return rc;
  } else {
    for (int i = 0; i < P.n; ++i)
      if (hipMemcpyAsync(P.part[i].dst, P.part[i].src, P.part[i].bytes, hipMemcpyDeviceToHost, st) != hipSuccess)
        return GS_EHIP;
  }
  GS_HIP(hipStreamSynchronize(st));
  if (staged)
    for (int i = 0; i < P.n; ++i) memcpy(P.part[i].dst, stage + P.part[i].at, P.part[i].bytes);
  return GS_OK;
}
