// Shared host/device definitions of the MI355X matching engine.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace dsm {

constexpr int kMaxQ = 16;       // query vertices per query (the reference's MAX_VQ, defs.h:18)
constexpr int kWave = 64;       // CDNA wavefront
constexpr int kMaxRel = 32;     // labels that can appear in an NLF requirement
constexpr int kMaxVertexChanges = 1024;  // per vertex per apply round (host splits beyond)
constexpr uint8_t kNoLabel = 255;  // device label of vertices whose label no query uses
#ifndef DSM_DONATE_BURST
#define DSM_DONATE_BURST 4  // ranges a busy wave may hand out per check
#endif
#ifndef DSM_LABEL_SORTED
#define DSM_LABEL_SORTED 64
#endif
constexpr uint32_t kLabelSorted = DSM_LABEL_SORTED;  // vertices of higher degree keep a label-sorted list copy
static_assert(kLabelSorted <= 64, "k_filter_light counts the entries of shorter lists in bytes");

// Matching plan of one (query, ordered query edge (u0,u1)) pair: positions 0
// and 1 hold the seeded edge, later positions follow a greedy order in which
// every vertex has an earlier neighbour.
struct alignas(16) Plan {
  uint8_t n;             // query vertices
  uint8_t pad0;
  uint16_t query;        // query index
  uint8_t qv[kMaxQ];     // query vertex at each position
  uint16_t sig[kMaxQ];   // candidate bitmap of each position
  uint16_t back[kMaxQ];  // earlier positions adjacent in the query
  uint16_t inj[kMaxQ];   // earlier positions with the same label (injectivity)
  uint8_t lix[kMaxQ];    // dense label index of each position (label-sorted lists)
  uint32_t pad1[3];
};
static_assert(sizeof(Plan) == 144, "plan layout");

// LDF/NLF requirement of one candidate bitmap: label, minimum degree and, for
// each of up to 32 relevant labels (dense index), the minimum number of
// neighbours with that label, one byte each (<= 15).
struct alignas(8) SigReq {
  uint32_t label;
  uint32_t deg;
  uint64_t nlc[4];
};

// A unit of DFS work: levels [0, level) are fixed in f; level `level` scans
// source-list indices [lo, hi). Every wave of the grid has a mailbox of its own
// (a 128-byte line): a busy wave that has claimed it while its owner waits
// (IdleWord) writes a task there and adds one to `mail`; `stop` takes the
// launch's epoch once no wave of the grid has work left.
struct alignas(128) Mailbox {
  uint32_t plan;
  uint32_t level;
  uint32_t lo, hi;
  uint32_t f[kMaxQ];
  uint32_t tag;          // count slot << 1 | sign (1 positive, 0 negative)
  uint32_t pad0;
  uint32_t mail;         // tasks delivered so far (never reset); read with stop as one 8-byte word
  uint32_t stop;
  uint32_t pad[8];
};
static_assert(sizeof(Mailbox) == 128, "mailbox layout");
constexpr int kTaskWords = 5 + kMaxQ;  // payload words (21)
constexpr uint32_t kMaxSlots = 64;     // count slots: requests served in one step

// Device-resident control block of one seed + DFS round. Every counter that
// waves update or poll concurrently has a 128-byte line of its own, so polling
// by idle waves does not serialise the atomics of busy ones.
template <typename T>
struct alignas(128) CtlLine {
  T v;
  uint32_t pad[(128 - sizeof(T)) / 4];
};
constexpr uint32_t kSeedHeads = 16;
struct DfsCtl {
  CtlLine<uint32_t> nseeds;        // seeds written by the seed kernel
  CtlLine<uint32_t> seed_head[kSeedHeads];  // seed shares claimed: head h counts shares h, h + kSeedHeads, ...
  CtlLine<uint32_t> seed_overflow; // seeds dropped for lack of capacity (must stay 0)
  CtlLine<uint32_t> donated;       // tasks handed to waiting waves, counted where they have a limit
  CtlLine<uint32_t> abort;         // set when an idle wave outlived the watchdog
};
// The waiting state of 16 waves of the grid (wave w of those that begin at once, or of the
// reserve, is in word w mod the words of its kind),
// a line each: bits 0..15 waiting for work, bits 16..31 started, bits 32..63 the
// number of claims so far. Busy waves look at one word after another for a
// waiting wave, so that no line is polled by the whole grid.
using IdleWord = CtlLine<unsigned long long>;
constexpr uint32_t kIdleGroup = 16;

// What a block of a DFS launch did, written to pinned host memory by the block
// when it ends; valid when epoch is the launch's (a block of the reserve that the round
// did without leaves it as it was). Times are wall-clock ticks.
struct alignas(128) BlockRec {
  unsigned long long epoch;
  unsigned long long active;       // waves that had a task
  unsigned long long busy;         // their time on tasks, summed
  unsigned long long first_min, first_sum;  // start of a wave's first task
  unsigned long long last_max, last_sum;    // end of its last one
  unsigned long long donated;      // tasks handed to waiting waves
  unsigned long long scanned;      // source-list entries tested
  unsigned long long loads;        // 4-byte reads of membership searches
  unsigned long long mbytes;       // 4 B x degree of every backward list of every expanded partial match
  unsigned long long nseeds, seed_overflow, abort;  // the control block as the block saw it last
  unsigned long long pad[2];
};
static_assert(sizeof(BlockRec) == 128, "block record layout");

// Status of the apply kernels of one batch.
struct alignas(64) ApplyCtl {
  unsigned long long scratch_used;
  unsigned long long pool_used;     // bump pointer of the neighbour pool
  uint32_t overflow;                // commits that found no room (host grows the pool)
  uint32_t relocated;
  uint32_t ndirty;                  // vertices on the dirty list
  uint32_t relabeled;
  uint32_t nrelabel_segs;           // pieces of the relabelled vertices' lists on BatchDev::segs
  uint32_t nsegs;                   // pieces of the touched lists (kApplySeg entries) on BatchDev::segs
  uint32_t merge_overflow;          // merges that found no room in the scratch (must stay 0)
  uint32_t filter_bits;             // candidate bits the re-filter writes (work measure)
  unsigned long long filter_entries;  // list entries of the vertices re-filtered (work measure)
  uint32_t max_deg;                 // no list has been longer (never lowered): kernels of longer lists are skipped
  uint32_t sync_queued[4];          // long lists queued by the catch-up (block, grid) and the sorted catch-up
  uint32_t chunks_dropped;          // refinement: chunks of long lists past the queue's end (must stay 0)
  uint32_t pad[11];
};
static_assert(sizeof(ApplyCtl) == 128, "apply status layout");

struct DevGraph {
  uint32_t n;
  uint32_t *pool;     // neighbour lists, sorted ascending, with slack
  uint32_t *start;    // first pool entry of each list
  uint32_t *deg;      // list length
  uint32_t *cap;      // slot capacity
  uint8_t *lab;       // vertex label (kNoLabel when no query uses it)
  // Vertices of degree > kLabelSorted also keep their list sorted by (dense
  // label, id) at lpool[start .. start + deg), with the bucket offsets of
  // label index i at loff[v * (nbuckets + 1) + i] (bucket nbuckets - 1 holds
  // labels no query uses).
  uint32_t *lpool;
  uint32_t *loff;
  uint32_t nbuckets;
};

struct FilterTables {
  const SigReq *sigs;       // [nsig]
  const uint32_t *sig_lo;   // [256] first sig of each label (sigs sorted by label)
  const uint32_t *sig_hi;   // [256] one past the last
  const uint8_t *lmap;      // [256] label -> dense relevant index or 0xFF
  uint32_t nsig;
  uint64_t *bm;             // [nsig][words]
  uint32_t words;           // ceil(n/64)
};

// Batch description uploaded per apply round.
struct BatchDev {
  uint32_t ntouched;
  const uint32_t *tv;       // touched vertices
  const uint32_t *ioff;     // [ntouched+1] into ins
  const uint32_t *doff;     // [ntouched+1] into del
  const uint32_t *ins;
  const uint32_t *del;
  // what the kernels of the round pass on, per touched vertex: the new degree,
  // how many of its inserts are new, where its merged list goes in the scratch
  // and where it ends up in the pool, and how far it is
  uint32_t *ndeg, *nnew, *dst, *state;
  unsigned long long *soff;
  uint32_t *ri;             // [ins] positions in the old list of t's new inserts, ascending, from ioff[t]
  uint32_t *rd;             // [del] positions of its deletes that are there, ascending, from doff[t]
  uint2 *segs;              // (t, piece): the touched lists in pieces of kApplySeg entries; once they are
                            // committed (vertex, piece | old label << 24): the relabelled vertices' lists
  uint32_t nrelabel;
  const uint32_t *rl_v;
  const uint32_t *rl_l;     // device label (already clamped)
};

constexpr uint32_t kNoDonateCap = 0xFFFFFFFFu;
struct DfsArgs {
  DevGraph g;
  const uint64_t *bm;
  uint32_t words;
  const Plan *plans;
  const uint32_t *seed_plan;
  const uint32_t *seed_s;
  const uint32_t *seed_d;
  Mailbox *mail;                 // [waves of the grid]
  IdleWord *idle;                // [ceil(waves / kIdleGroup)] of those that begin at once, then of the reserve
  uint32_t donate_cap;           // most tasks the round may hand to waiting waves
  uint32_t crew;                 // waves of the blocks that begin at once; the others are a reserve
  uint32_t cgroups, ngroups;     // their waiting words, and all
  unsigned long long join_after; // wall-clock ticks after which the reserve joins
  uint32_t epoch;
  uint32_t donate_min;
  uint32_t lane_work;            // longest leaf list one lane scans alone
  uint32_t leaf_budget;          // inline leaf-count work of a window before a candidate descends
  uint32_t donate_every;         // chunks between checks for waiting waves
  uint32_t donate_min_n2;        // smallest range split off one level above the leaf
  uint32_t leaf_segments;        // leaf lists scanned as one segmented array
  uint32_t poll_max;             // longest sleep between polls of a waiting wave (s_sleep 8 units)
  uint32_t leaf_sets;            // fused leaf level on/off
  uint32_t bit_probe_last;       // candidate bit probed after the membership tests
  uint32_t fshift;               // ids >> fshift < 512: the leaf set's bucket of an id
  uint32_t nq;                   // queries (count layout)
  const uint32_t *seed_tag;      // per seed: count slot << 1 | sign
  unsigned long long watchdog;   // wall-clock ticks an idle wave may wait
  DfsCtl *ctl;
  unsigned long long *counts;    // [slot][nq][2]: index (slot*nq + q)*2 + sign
  uint32_t *tuples;              // [tuple_cap][kMaxQ+2] or null
  unsigned long long tuple_cap;
  unsigned long long *tuple_count;  // tuples found this batch
  BlockRec *rec;                    // [blocks of the grid], pinned host memory
  unsigned long long *query_busy;   // per query: wall-clock ticks of its tasks (or null)
};

struct SeedArgs {
  DevGraph g;
  const uint64_t *bm;
  uint32_t words;
  const Plan *plans;
  const uint8_t *lmap;        // device label -> dense index of the query labels (0xFF: none)
  const uint2 *plan_of;       // [kMaxRel][kMaxRel]: first plan and number of plans of a pair of them
  uint32_t nplans;
  // two record lists, each with the tag written to its seeds
  const uint32_t *rs[2];
  const uint32_t *rd[2];
  uint32_t nrec[2];
  uint32_t tag[2];
  uint32_t *seed_plan;
  uint32_t *seed_s;
  uint32_t *seed_d;
  uint32_t *seed_tag;
  uint32_t seed_cap;
  DfsCtl *ctl;
};

struct DirtyArgs {
  uint8_t *marks;      // [n rounded up to 16] dirty marks
  uint32_t *list;      // dirty vertices
  uint32_t list_cap;
  ApplyCtl *actl;
};

// Message of the last failed call that has no engine (dsm_last_error(NULL)).
void set_global_error(const char *fmt, ...);

// Words that a kernel copies between pinned host memory and the device on its way
// (none if words is 0). A copy of its own costs a launch, an API call and a blit
// kernel, some 8 us in all; one block reads a few hundred words over the host link in
// 3 us and 3,000 in 10 (a call with either takes as long with the line at 1,024).
constexpr uint32_t kSmallCopy = 4096;
struct SmallCopy {
  const uint32_t *from;
  uint32_t *to;
  uint32_t words;
};
// A copy of at most kSmallCopy words.
hipError_t launch_small_copy(const SmallCopy &c, hipStream_t s);
// Several arrays copied by one launch (from and to aligned to 16 bytes).
struct ArrayCopies {
  static constexpr uint32_t kMost = 10;
  const void *from[kMost];
  void *to[kMost];
  size_t bytes[kMost];  // multiples of 4
  uint32_t n;
};
hipError_t launch_array_copies(const ArrayCopies &c, hipStream_t s);

// The adjacency of an edge list (dsm_build.hip). Keys are source << bits | target,
// two an edge (count = 2 m); hist has csr_scan_words(count) words, sums
// csr_sum_words of what is scanned (hist, or n slots).
struct CsrCtl {
  unsigned long long bad;     // the first edge with an endpoint out of range (set to ~0 before)
  unsigned long long unique;  // keys left once equal ones are dropped
  unsigned long long total;   // pool entries the slots take
  uint32_t max_deg;
  uint32_t pad;
};
size_t csr_scan_words(size_t count);
size_t csr_sum_words(size_t items);
hipError_t launch_csr_keys(const uint32_t *src, const uint32_t *dst, size_t m, uint32_t n, uint32_t bits,
                           unsigned long long *keys, CsrCtl *ctl, hipStream_t s);
// One stable pass of the sort over the 8 bits from shift up.
hipError_t launch_radix_pass(const unsigned long long *from, unsigned long long *to, size_t count, uint32_t shift,
                             unsigned long long *hist, unsigned long long *sums, hipStream_t s);
hipError_t launch_csr_unique(const unsigned long long *from, unsigned long long *to, size_t count,
                             unsigned long long *hist, unsigned long long *sums, CsrCtl *ctl, hipStream_t s);
// Degrees, capacities and slot starts of ctl->unique keys; deg must be clear.
hipError_t launch_csr_slots(const unsigned long long *keys, size_t count, uint32_t n, uint32_t bits, uint32_t *begin,
                            uint32_t *deg, uint32_t *cap, uint32_t *start, unsigned long long *slot,
                            unsigned long long *sums, CsrCtl *ctl, hipStream_t s);
hipError_t launch_csr_fill(const unsigned long long *keys, size_t count, uint32_t bits, const uint32_t *begin,
                           const uint32_t *start, uint32_t *pool, const CsrCtl *ctl, hipStream_t s);

// The lists of a graph packed: off[0, n] from the degrees (sums: csr_sum_words(n + 1)
// words), then the total = off[n] entries.
hipError_t launch_graph_offsets(uint32_t n, const uint32_t *deg, unsigned long long *off, unsigned long long *sums,
                                hipStream_t s);
hipError_t launch_graph_lists(uint32_t n, const unsigned long long *off, const uint32_t *start, const uint32_t *pool,
                              size_t total, uint32_t *out, hipStream_t s);

// ---- cluster-encoding refinement (dsm_cluster_plan.cpp, dsm_cluster.hip) ---

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kMaxClusters = 150;       // MAX_CLUSTERS, defs.h:22
constexpr uint32_t kMaxClusterLayers = 100;  // MAX_LAYERS, defs.h:23
constexpr uint32_t kMaxSmallClusters = 32;   // per combine (filter.cu:1056-1061)

// Host plan of one query's refinement: clusters with their bit positions, the
// combines, the passes in execution order and each query vertex's final
// position (its refined candidate set).
struct ClusterPlan {
  struct Cluster {
    std::vector<uint32_t> members;  // core first, then its neighbours
    bool valid = true;
    bool merged = false;            // made by a merge of clusters left and right
    uint32_t left = kNone, right = kNone;
    uint32_t left_pos = kNone, right_pos = kNone;  // the core's positions in left / right
    uint32_t pos = 0;               // first bit position
  };
  struct Combine {
    uint32_t big = kNone;           // the cluster that receives the combination
    bool keep = false;              // big existed (AND into it) or was created (OR)
    std::vector<uint32_t> small;
  };
  enum { kEncode = 0, kMerge = 1, kCombine = 2 };
  struct Pass {
    uint32_t kind, arg;             // encode / merge: cluster; combine: index into combines
  };
  std::vector<Cluster> clusters;
  std::vector<Combine> combines;
  std::vector<Pass> passes;
  std::vector<uint32_t> final_pos;  // per query vertex
  uint32_t final_cluster = 0;
  uint32_t positions = 0;
};

// Returns 0, or -1 when the plan exceeds one of the reference's limits.
int build_cluster_plan(uint32_t n, uint32_t m, const uint32_t *eu, const uint32_t *ev, ClusterPlan &out);

// One pass of one query on the device. Bitmap rows index `bm` (signature rows
// first, then every query's position rows); `alive` rows are the candidate
// lists the passes prune (d_u_candidate_vs_ of the reference).
enum : uint32_t { kOpEncode = 0, kOpMerge = 1, kOpCombineNew = 2, kOpCombineKeep = 3 };
struct alignas(16) ClusterOp {
  uint32_t kind;
  uint32_t alive;       // alive row of the cluster's core
  uint32_t core;        // bm row of the core position; targets at core+1 .. core+ntarget
  uint32_t ntarget;
  uint32_t check_off;   // a core candidate survives when all rows crow[check_off ..+ncheck) hold it
  uint32_t ncheck;
  uint32_t pad[2];
  uint16_t toff[kMaxQ]; // target t: the AND of rows crow[toff[t] .. +tcnt[t]) at the neighbour
  uint16_t tcnt[kMaxQ];
  uint8_t tlab[kMaxQ];  // device label of target t's query vertex (every condition implies it)
  uint8_t tlix[kMaxQ];  // its dense label index (the bucket of the label-sorted lists)
  uint8_t lix[kMaxQ];   // the distinct tlix values, nlix of them
  uint32_t nlix;
  uint32_t pad2[3];
};

struct ClusterHeavy {
  // entries [lo, lo + kClusterChunk) of candidate v's label bucket li (in the
  // label-sorted copy) for pass op
  uint32_t op, v, lo, li;
};
constexpr uint32_t kClusterChunk = 4096;

struct ClusterArgs {
  DevGraph g;
  uint64_t *bm;
  uint32_t words;
  uint64_t *alive;
  const ClusterOp *ops;
  uint32_t nops;
  const uint32_t *crow;
  ClusterHeavy *heavy;
  uint32_t heavy_cap;
  uint32_t *ctl;        // [1]: heavy entries queued
  ApplyCtl *actl;       // status of the update before it
};

// Zeroes bm rows [first_row, first_row + nrows), copies the listed (alive row,
// bm row) pairs into the alive rows and zeroes nctl counters. Like the kernels of the
// passes it does nothing while the update of actl is held up.
hipError_t launch_cluster_init(uint64_t *bm, uint32_t words, uint32_t first_row, uint32_t nrows, uint64_t *alive,
                               const uint32_t *alive_src, uint32_t nalive_src, uint32_t *ctl, uint32_t nctl,
                               const ApplyCtl *actl, hipStream_t s);
hipError_t launch_cluster_pass(const ClusterArgs &a, uint32_t max_blocks, hipStream_t s);
hipError_t launch_cluster_heavy(const ClusterArgs &a, uint32_t blocks, hipStream_t s);

// ---- launchers (dsm_kernels.hip) -------------------------------------------
// Launches of an update. Every kernel after the commit does nothing once a
// commit found no room (ApplyCtl::overflow) or a merge none (merge_overflow), so
// that the whole update is enqueued at once and the host looks at the status
// when it is done. `longest` is a length no list exceeds: kernels that only work
// on longer lists are not launched.
constexpr uint32_t kApplySeg = 1024;     // entries of a touched list a wave merges or commits at a time
// states of a touched vertex
constexpr uint32_t kInPlace = 0;   // its list fits its slot: merged into the scratch, then committed
constexpr uint32_t kDirect = 1;    // merged into a new slot
constexpr uint32_t kNoRoom = 2;    // merged into the scratch, needs a slot the pool has no room for
constexpr uint32_t kRetried = 3;   // has one now: to be committed
constexpr uint32_t kDone = 4;      // committed by an earlier try
constexpr uint32_t kSyncWave = 4096;     // longer lists are brought up to date by the whole grid
constexpr uint32_t kBuildSeg = 1024;     // label-sorted copies of longer lists are built in pieces

// Takes over the status `from` (null: keeps its own) and clears what an update
// counts, also bctl[4] (SortedBuild::ctl).
hipError_t launch_update_begin(ApplyCtl *actl, const ApplyCtl *from, uint32_t *bctl, const SmallCopy &up,
                               hipStream_t s);
// Clears what the merges of one round count (updates with more than one).
hipError_t launch_round_begin(ApplyCtl *actl, const SmallCopy &up, hipStream_t s);
// The merges and commits of a round; max_segs bounds the pieces.
hipError_t launch_apply(const DevGraph &g, const BatchDev &b, uint32_t *scratch, unsigned long long scratch_cap,
                        unsigned long long pool_cap, ApplyCtl *actl, const DirtyArgs &d, size_t max_segs,
                        hipStream_t s);
// The commits that found no room, again.
hipError_t launch_commit_again(const DevGraph &g, const BatchDev &b, const uint32_t *scratch,
                               unsigned long long pool_cap, ApplyCtl *actl, const DirtyArgs &d, size_t max_segs,
                               hipStream_t s);
// The dirty list (d.list, its length added to d.actl->ndirty) from the dirty
// bits of the update's n vertices.
hipError_t launch_dirty_compact(const DevGraph &g, const DirtyArgs &d, hipStream_t s);
// What the last update changed, from graph copy x to the stale copy y: the
// touched vertices' slots and lists, the relabelled vertices' labels and the
// nbm words of the signature rows. q (qcap entries) is scratch for the long
// lists.
struct CatchUp {
  DevGraph x, y;
  const uint32_t *touched, *relabeled;
  uint32_t ntouched, nrelabeled;
  const uint64_t *bm_x;
  uint64_t *bm_y;
  size_t nbm;
  uint32_t *q;
  uint32_t qcap;
  ApplyCtl *actl;  // y's
};
hipError_t launch_catch_up(const CatchUp &c, uint32_t longest, hipStream_t s);
// The label-sorted copies and bucket offsets of the listed (dirty) vertices
// from x to y, except those whose bit is set in skip.
hipError_t launch_sync_sorted(const DevGraph &x, const DevGraph &y, const uint32_t *dirty, const uint32_t *ndirty,
                              const uint8_t *skip, uint32_t *q, uint32_t qcap, ApplyCtl *actl, uint32_t longest,
                              hipStream_t s);
hipError_t launch_relabel(const DevGraph &g, const BatchDev &b, const FilterTables &ft,
                          const DirtyArgs &d, size_t max_segs, hipStream_t s);
hipError_t launch_filter_full(const DevGraph &g, const FilterTables &ft, hipStream_t s);
// Label-sorted copies: lists of up to kBuildSeg entries are built by a wave each,
// longer ones in pieces (at most kBuildPieces a list), whose bucket counts go to
// hist.
constexpr uint32_t kBuildPieces = 512;
struct SortedBuild {
  uint32_t *ctl;       // [4]: short lists queued, long ones queued, pieces dealt
  uint32_t *mid;       // [n]: vertices with short lists
  uint2 *big;          // [pool / kBuildSeg]: (vertex with a long list, its first piece)
  uint2 *pieces;       // [2 pool / kBuildSeg]: (vertex, piece)
  uint32_t *hist;      // [pieces][kMaxRel + 2]
  // one byte per pool entry (indexed like the pool): the bucket of each entry,
  // written by the counting pass so that the scatter pass reads it back
  // instead of gathering the neighbour's label again (null: gather twice)
  uint8_t *bucket_bytes;
  const ApplyCtl *actl;  // the update's status (null: a full build)
};

// Rebuilds the label-sorted copies of the listed vertices (list + count on the
// device), or of every vertex when list is null, and, if asked, sets those
// vertices' candidate bits. hs.ctl must be clear.
hipError_t launch_lbuild(const DevGraph &g, const FilterTables &ft, const uint32_t *list, const uint32_t *count,
                         const SortedBuild &hs, uint32_t longest, bool filter, hipStream_t s);
hipError_t launch_build_reset(const SortedBuild &hs, hipStream_t s);
// A whole update in one launch: begin, apply, relabel, builds and re-filter, with its
// status written to pinned host memory. longest <= kBuildSeg, kSmallChanges changes,
// the arrays small enough for `up`.
constexpr uint32_t kSmallChanges = 128;
hipError_t launch_update_small(const DevGraph &g, const BatchDev &b, const FilterTables &ft, const DirtyArgs &d,
                               const SortedBuild &hs, uint32_t *scratch, unsigned long long scratch_cap,
                               unsigned long long pool_cap, uint32_t longest, const SmallCopy &up, ApplyCtl *status,
                               hipStream_t s);
// The candidate bits of the dirty vertices without a label-sorted copy.
hipError_t launch_filter_dirty(const DevGraph &g, const FilterTables &ft, const DirtyArgs &d, hipStream_t s);
hipError_t launch_seed(const SeedArgs &a, hipStream_t s);
hipError_t launch_dfs(const DfsArgs &a, uint32_t blocks, uint32_t waves_per_block, uint32_t max_query_vertices,
                      hipStream_t s);
// Resets the DFS control block (ctl) with the nidle waiting words, the tuple
// counter and ncounts match counts; null pointers are skipped. Also the copy `up`
// (the round's records).
hipError_t launch_ctl_reset(DfsCtl *ctl, unsigned long long *tuple_count, unsigned long long *counts,
                            uint32_t ncounts, IdleWord *idle, uint32_t nidle, const SmallCopy &up, hipStream_t s);
hipError_t launch_pool_move(const uint32_t *old_pool, uint32_t *new_pool, const uint32_t *old_start,
                            const uint32_t *new_start, const uint32_t *deg, uint32_t n,
                            hipStream_t s);
int dfs_max_blocks_per_cu(uint32_t waves_per_block, uint32_t max_query_vertices);

uint32_t dfs_lds_bytes_per_wave(uint32_t max_query_vertices);

}  // namespace dsm
