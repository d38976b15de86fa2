// Host-side internals shared by the HIP translation units of libgpuseed.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <utility>
#include <vector>

#include "gpuseed.h"
#include "gs_device.h"

#define GS_HIP(call)                        \
  do {                                      \
    hipError_t e_ = (call);                 \
    if (e_ != hipSuccess) return GS_EHIP;   \
  } while (0)

struct gs_index {
  int device = 0;
  hipStream_t stream = nullptr;
  uint32_t primary = 0, seq_len = 0, sa_intv = 0;
  uint32_t L2[5] = {0, 0, 0, 0, 0};
  uint64_t n_blocks = 0;  // 96-base blocks
  uint64_t n_sa = 0;
  uint4* occ = nullptr;
  uint32_t* sa = nullptr;
  uint2* kmer = nullptr;
  uint4* kext = nullptr;  // extended interval table with presence bits (gs_index_set_kmer_len)
  uint32_t ext_len = 0;
  // direct-extension structures (gs_index_set_direct): full suffix array and
  // its inverse (seq_len + 1 words each), the text at 2 bits per base
  uint32_t* sa_full = nullptr;
  uint32_t* isa = nullptr;
  uint32_t* text = nullptr;
  uint64_t text_words = 0;
  // rows whose reference walk passes row primary+1 and their reported
  // positions (locate from the full suffix array); n_quirk > kMaxQuirk: walk
  uint2* quirk = nullptr;
  uint32_t n_quirk = 0;
  uint8_t* pair = nullptr;  // pair table (gs_index_set_pairs), 4^18 bytes
  uint4* tandem = nullptr;  // tandem table, built with the 13-mer table
  double t_pairs = 0;
  uint64_t device_bytes = 0;
  double t_read = 0, t_upload = 0, t_repack = 0, t_table = 0, t_sa = 0, t_write = 0, t_ext = 0, t_direct = 0;
  int sa_rounds = 0;
  gs_batch* work = nullptr;  // gs_seed's batch, kept for the next call (its buffers only grow)
  std::mutex locate_mu;
  gs_batch* locate = nullptr;  // gs_index_locate's pinned chunks (two of at most 80 MB)
  // Lifetime: the caller's handle holds one reference, every batch and
  // server made on the index one more; gs_index_close drops the caller's
  // and the device structures are freed with the last one, so a batch or
  // server that outlives the caller's handle still reads valid memory.
  std::atomic<int> refs{1};
  std::atomic<int> servers{0};  // live servers: their workers launch at any time
  gs::DevIndex dev() const;
};

namespace gs {
void index_acquire(gs_index* X);
void index_release(gs_index* X);  // frees the index with its last reference
// Work-items per launch of the chunked kernels (table levels, presence
// bits, direct-structure chains, suffix-array walk): a dispatch's work-item
// count is a 32-bit quantity, so launches over more items than this are
// split.  2^30 unless a test sets it smaller (gs_set_launch_chunk).
uint64_t launch_chunk();
// allocation of result arrays handed to callers (freed with free())
void* result_alloc(size_t bytes);
// Looks up the device address of gs_seed_noalloc's scratch array on `device`
// (which must be current); called once per device where an index is set up.
int noalloc_setup(int device);
}  // namespace gs

namespace gs {

// Parameters of the persistent extension kernel (gs_persist.hip).
//
// Work items: one per (read, strand) for reads of at most kPersistLmax bases;
// reads longer than that are cut into segments of seg_tasks consecutive task
// ends, one item per (read, segment, strand).  items[i] = read | (segment << 33)
// | (strand << 32); the items of a read are adjacent, segment-major.
// The fields of a persistent launch that the kernel's loop uses only at
// item starts and ends, in work splitting and for its counters.  The launch
// writes them to device memory (the 256 bytes after the counters) and the
// kernel reads them with scalar loads where it uses them, so that its
// arguments fit the scalar registers instead of spilling into vector ones.
struct PersistCold {
  const uint8_t* bases;    // the batch's bytes and the reads' offsets in them (plain kernel)
  const uint64_t* offs;
  const uint64_t* code_off;
  const uint32_t* lens;
  const uint64_t* task_off;
  const uint64_t* items;
  uint4* cand;
  uint32_t* nF;
  uint32_t* nR;
  uint4* seg_meta;
  uint32_t* seg_link;
  uint64_t* counters;
  uint4* dyn_items;
  uint4* dyn_meta;
  uint32_t* dyn_link;
  uint32_t* reserved;
  uint4* wmeta;
  uint32_t* wlink;
  uint32_t seg_tasks, pad;
};
constexpr uint32_t kCounterBytes = 32;   // four 64-bit counters
constexpr uint32_t kColdBytes = 256;     // PersistCold, after the counters
static_assert(sizeof(PersistCold) <= kColdBytes, "PersistCold must fit its slot");

struct PersistParams {
  DevIndex X;
  const uint8_t* bases;      // plain kernel: the batch's bytes and offsets (32 bytes kept after the last read)
  const uint64_t* offs;
  const uint4* codes;        // 4-bit virtual codes, per read: forward chunks then reverse chunks
  const uint64_t* code_off;  // per read, in 16-byte chunks
  const uint32_t* lens;
  const uint64_t* task_off;
  const uint64_t* items;
  uint64_t n_items;
  uint32_t n_long, k, smem, seg_tasks;
  uint4* cand;               // same candidate layout as the plain kernel
  uint32_t* nF;
  uint32_t* nR;
  uint4* seg_meta;           // per item of a segmented read: {emitted, first b, last b, flags}
  uint32_t* seg_link;        // per item of a segmented read: first piece split off it, or ~0
  uint32_t* queue;           // [0] the next item to hand out, [1] pieces reserved
  uint64_t* counters;        // optional: [0] table reads, [1] occ entry reads, [2] direct-extension reads,
                             // [3] tandem-table reads
  uint32_t direct_min;       // size-1 steps before a task reads the text (0: no direct extension)
  // work splitting (dyn_cap 0: off)
  uint4* dyn_items;          // pieces {read, strand, first task, tasks}
  uint4* dyn_meta;           // per piece, as seg_meta
  uint32_t* dyn_link;        // per piece: the next piece in task order, or ~0
  uint4* wmeta;              // per whole-read stream (2 * read + strand) that was split
  uint32_t* wlink;
  uint32_t dyn_cap, split_work, split_tasks;
  uint32_t tandem;                // tandem jumps: largest period (0: off; needs the index's tandem table)
};

// Joins pieces (segments of long reads, split-off pieces) into the per-read
// candidate layout.
struct JoinParams {
  const uint32_t* long_reads;   // reads cut into segments
  const uint64_t* item0;        // per long read: index of its first item
  const uint32_t* lens;
  const uint64_t* task_off;
  const uint4* seg_meta;
  const uint32_t* seg_link;
  const uint4* dyn_items;
  const uint4* dyn_meta;
  const uint32_t* dyn_link;
  const uint4* wmeta;
  const uint32_t* wlink;
  uint4* cand;
  uint32_t* nF;
  uint32_t* nR;
  uint32_t n_long, k, smem, seg_tasks;
  uint32_t n_reads, dyn_cap;
};

constexpr uint32_t kSplitStream = 0xFFFFFFFFu;  // nF/nR of a whole-read stream left for join_whole_wave/thread
// Work splitting (take_pieces): a lane gives half of its task ends away after
// kSplitWork memory operations (at once in a launch of fewer items than
// lanes), while it has at least 2 * kSplitTasks of them left, and once
// kSplitIdle lanes of its wave are idle (kSplitIdleSmall in such a launch).
// Measured, kernel ms: idle lanes 8, 16, 24, 32 in small launches: 10,000
// 150 bp reads on a 100 Mbp index 0.74, 0.80, 0.74, 0.71, 60,000 on the
// 3.1 Gbp index 1.62, 1.61, 1.68, 1.83; task ends 2, 4, 8: 1.42, 1.68, 2.07
// and 1000 reads there 0.58, 0.85, 0.86.  In a launch of 1,000,000 reads all
// of 16-32 idle lanes, 16-64 operations and 1-4 task ends gave 7.2-7.5.
// kSplitTasksLong (launches from the queue, SMEM, some reads in segments):
// 20,000 uneven reads on the 3.1 Gbp index with 2, 4, 8 and 12 task ends 3.41,
// 3.26, 3.18, 3.47 ms, 60,000 6.69, 6.56, 6.35, 6.26, in MEM mode 3.88, 4.04,
// 3.95, 3.96; 500,000 150 bp reads 3.97, 4.03, 4.38, 4.43.  kSplitTasksPlain
// (a plain task has no shortcuts, and so more steps): with 1, 2 and 4 10,000
// uneven reads on a 100 Mbp index 2.60, 2.71, 3.20 ms, 300,000 150 bp reads
// 4.32, 4.41, 4.59.
constexpr uint32_t kSplitWork = 64;
constexpr uint32_t kSplitTasks = 2, kSplitTasksPlain = 1, kSplitTasksLong = 8;
constexpr uint32_t kSplitIdle = 32;
constexpr uint32_t kSplitIdleSmall = 24;
// Pieces a launch can split off (36 bytes each): 8 per item, at least 65,536,
// at most 2^20; beyond that items go on whole.
__host__ inline uint32_t piece_cap(uint64_t n_items) {
  return (uint32_t)(n_items >= (1u << 17) ? 1u << 20 : (n_items < 8192 ? 65536 : 8 * n_items));
}
constexpr uint32_t kRefillGroup = 12;           // idle lanes of a wave that trigger a refill
                                                // (2.5M 150 bp reads, 3.1 Gbp index, an early
                                                // form of the kernel: 1 lane 72.5 ms, 4: 58.0 ms,
                                                // 8: 58.2 ms, 16: 59.6 ms; 10M reads with the
                                                // current one, alternating runs on one box: 8:
                                                // 68.7-69.0 ms, 12: 67.6-68.1 ms median)

constexpr uint32_t kPersistLmax = 160;  // LDS code window of a persistent lane, in bases
// Tandem jumps of the persistent kernel: periods 1..kTandemMax; a stretch
// [R, E) opens at a task end E whose 20 codes to the left have a period and
// spans at least kTandemSpan positions; a task end e of the stretch with
// e - R >= kTandemMin reads the tandem table's row of length
// min(e - R, kTandemLen).  With the 20 codes of the rolling window a period
// is at most 19; the configurations' tandem repeats have periods 1-6.
constexpr uint32_t kTandemMax = 6;
constexpr uint32_t kTandemSpan = 24;
constexpr uint32_t kTandemMin = 20;
constexpr uint32_t kTandemLen = 256;
// The tandem table: for every unit of 1..kTandemMax bases (key base(p) +
// sum of code_j * 4^j, the unit's last base as j = 0, base(p) = (4^p - 4) / 3)
// and every length n in [kTandemMin, kTandemLen], the 16-byte entry
// {l, u, m, 0} of the string of length n that ends with the unit repeated
// (the unit's last base at its end): m = the longest length <= n whose
// string occurs, [l, u] the interval of that length.
constexpr uint32_t kTandemKeys = (4096u * 4u - 4u) / 3u;  // 5460
constexpr uint32_t kTandemRows = kTandemLen - kTandemMin + 1;
__host__ __device__ constexpr uint32_t tandem_key_base(uint32_t p) { return ((1u << (2 * p)) - 4u) / 3u; }
constexpr uint32_t kSegTasksMax = 112;  // task ends per segment: the window keeps every 13-base start

// segments of a read of length L (1 for reads held whole in the LDS window)
__host__ __device__ inline uint32_t n_segments(uint32_t L, uint32_t k, uint32_t seg_tasks) {
  if (L <= kPersistLmax || L < k) return 1;
  const uint32_t ntask = L - k + 1;
  return (ntask + seg_tasks - 1) / seg_tasks;
}

__host__ __device__ __forceinline__ bool read_is_long(uint32_t L, uint32_t k, uint32_t nseg) {
  return nseg > 1 || (L > kPersistLmax && L >= k);
}

// What the reads of a batch need, added up read by read.
struct ReadSums {
  uint64_t tasks = 0, chunks = 0, whole = 0, items = 0, n_long = 0;  // items: those of long reads' segments
  void add(uint32_t L, uint32_t k, uint32_t seg_tasks) {
    tasks += L >= k ? L - k + 1 : 0;
    chunks += 2 * (uint64_t)((L + 31ull) / 32);
    const uint32_t nseg = n_segments(L, k, seg_tasks);
    if (read_is_long(L, k, nseg)) {
      ++n_long;
      items += 2ull * nseg;
    } else {
      whole += 2ull * nseg;
    }
  }
};

// The sizes that a batch's device buffers follow from: bytes of its reads,
// reads, task slots per strand, 16-byte code chunks, work items, reads in
// segments, reference batches that need a list, room for split-off pieces.
struct BatchSizes {
  uint64_t span, n, tasks, chunks, items, n_long, cuts;
  uint32_t dyn_cap;
};
uint64_t batch_bytes(const BatchSizes& z);  // all of them, outputs excluded

int launch_pack_codes(const uint8_t* bases, const uint64_t* offs, const uint32_t* lens, const uint64_t* code_off,
                      uint32_t n_reads, const uint32_t* long_reads, uint32_t n_long, uint4* codes, hipStream_t st);
// variant -1: the plain kernel (wg ignored), 0: 8-bit size records, 1: 16-bit
// and 2: 4-bit size records; wg 64, 128 or 256 (0 = 128); grid from persistent_grid (called outside any graph capture)
int persistent_grid(int variant, int wg, unsigned* grid);
// e0, e1 (optional): recorded on st right before and after seed_persistent
int launch_persistent(const PersistParams& P, int variant, int wg, unsigned grid, hipStream_t st,
                      hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
int launch_join(const JoinParams& J, hipStream_t st);

}  // namespace gs

namespace gs {

// The CPU side of a batch (see gs_batch_create): built on any thread, then
// uploaded by batch_load.  Sizes and the sources of the uploads; offsets of
// tasks and codes, reference-batch ids and work items (n_items of them, n_whole
// of reads held whole, n_long reads cut into segments) are written on the
// device when the batch is loaded.  The reads' bytes, and a single group's
// arrays unless plan_finish copied them, must stay as they are until then.
struct BatchPlan {
  gs_opts opts{};
  uint32_t seg_tasks = 64;
  uint64_t n_reads = 0, span = 0, tasks = 0, code_chunks = 0, n_items = 0, n_whole = 0, n_long = 0;
  std::vector<std::pair<const char*, uint64_t>> pieces;  // bytes uploaded back to back
  struct Group {  // reads of one source: offsets less lo, plus base, are theirs in the batch
    const uint64_t* offs;
    const uint32_t* lens;
    uint64_t n, lo, base;
  };
  std::vector<Group> groups;
  std::vector<uint32_t> cuts;  // first reads of the second reference batch and those after it
  std::vector<uint64_t> offs;  // of several groups (plan_finish)
  std::vector<uint32_t> lens;
};

int plan_check(const gs_opts* o);
void plan_reset(BatchPlan& P, const gs_opts& o);
// appends reads [r0, r1) of one source as a group of their own
int plan_add(BatchPlan& P, const char* bases, const uint64_t* offsets, const uint32_t* lens, uint64_t r0,
             uint64_t r1);
void plan_finish(BatchPlan& P, bool copy = false);
uint64_t plan_device_bytes(const BatchPlan& P);  // device buffers the plan needs, outputs excluded
// hold: the batch keeps a reference to X (every batch but gs_seed's own,
// which the index owns and frees)
gs_batch* batch_new(gs_index* X, bool hold = true);
int batch_load(gs_batch* B, const BatchPlan& P, bool wait = true);
// Grows B's device buffers for any plan of at most `bases` bases and `reads`
// reads, so that loading such plans allocates (and synchronises) nothing (but
// tries again for pinned chunks that it could not have).
int batch_reserve(gs_batch* B, uint64_t bases, uint64_t reads, uint32_t seg_tasks);
void batch_free(gs_batch* B);

// Results of the batch's last run, downloaded into pinned staging that the
// batch keeps (valid until the next download or the batch's end).
struct ResultView {
  uint64_t n_reads, n_seeds, n_pos;
  const uint32_t *nseeds, *npos;
  const uint64_t *soff, *poff;
  const gs_seed_rec* seeds;
  const uint32_t* pos;
};
int batch_download(gs_batch* B, ResultView* v);

}  // namespace gs

// Tuning fields of an existing batch (the autotuner's knobs that need no new
// work items): kernel variant, workgroup size, suffix-array walk rows.
int gs_batch_set_tuning(gs_batch* B, int kernel, int wg, int walk_rows);
int gs_batch_set_direct_min(gs_batch* B, uint16_t direct_min);  // as gs_opts.direct_min

// ceil(2^64 / d) for d >= 2 (exact quotient for every 32-bit numerator), 0 for d == 1
uint64_t gs_reciprocal64(uint32_t d);

// Builds the 4^13 interval table on the index's stream (pre_calc_seed_intervals_gpu,
// seed_gen.cu:2648-2675), level by level.
int gs_build_kmer_table(gs_index* X);
