// Host side of the MI355X continuous subgraph matching engine: the C ABI of
// include/dsm.h over the kernels of dsm_kernels.hip.
//
// Per batch (dsm_apply_batch + dsm_match_batch):
//   1. delete records seed DFS roots in the pre-batch graph (negatives)
//   2. host: symmetrise, stable (src,dst) sort, final op per key, final label
//      per vertex (the update rule of cpuGraph.cpp:521-607)
//   3. device: merge/commit the per-vertex deltas in place, relabel, refresh
//      the candidate bitmaps of the dirty vertices
//   4. insert records seed DFS roots in the post-batch graph (positives)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "../../include/dsm.h"
#include "dsm_internal.h"

using namespace dsm;

namespace {

thread_local std::string g_create_error;

}  // namespace

namespace dsm {
void set_global_error(const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_create_error = buf;
}
}  // namespace dsm

namespace {

struct QueryHost {
  uint32_t n = 0;
  uint32_t lab[kMaxQ] = {};
  uint32_t adj[kMaxQ] = {};  // bitmask
  uint32_t order_variant = 0;  // rule of its matching orders (next_in_order)
};

constexpr uint32_t kOrderVariants = 4;

#ifndef DSM_DELTA_SYNC
#define DSM_DELTA_SYNC 1
#endif
// 1: an overlapped update brings the second copy of the graph up to date by
// copying only what the previous update changed (catch_up)
constexpr bool kDeltaSync = DSM_DELTA_SYNC;

// The next query vertex of a matching order, among the unplaced vertices with
// an earlier neighbour, by rule `variant` (ties: lowest id). An order never
// changes a count, only the work: the tuner picks the rule per query.
//   0: most earlier neighbours, then the rarest label in the data graph, then
//      the highest query degree;
//   1: most earlier neighbours, then the highest query degree, then the
//      rarest label;
//   2: the rarest label, then most earlier neighbours, then the highest degree;
//   3: most earlier neighbours, then the most frequent label, then the highest
//      query degree.
uint32_t next_in_order(const QueryHost &Q, uint32_t placed, const std::vector<uint64_t> &label_freq,
                       uint32_t variant) {
  int best = -1;
  int64_t bk[3] = {0, 0, 0};
  for (uint32_t w = 0; w < Q.n; w++) {
    if (placed >> w & 1) continue;
    const int64_t b = __builtin_popcount(Q.adj[w] & placed);
    if (b == 0) continue;
    const int64_t dg = __builtin_popcount(Q.adj[w]);
    const int64_t f = Q.lab[w] < label_freq.size() ? (int64_t)label_freq[Q.lab[w]] : 0;
    int64_t k[3];
    switch (variant) {
      case 1: k[0] = b; k[1] = dg; k[2] = -f; break;
      case 2: k[0] = -f; k[1] = b; k[2] = dg; break;
      case 3: k[0] = b; k[1] = f; k[2] = dg; break;
      default: k[0] = b; k[1] = -f; k[2] = dg; break;
    }
    if (best < 0 || k[0] > bk[0] || (k[0] == bk[0] && (k[1] > bk[1] || (k[1] == bk[1] && k[2] > bk[2])))) {
      best = (int)w;
      bk[0] = k[0];
      bk[1] = k[1];
      bk[2] = k[2];
    }
  }
  return (uint32_t)best;
}

template <typename T>
struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  ~DevBuf() { reset(); }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t alloc(size_t count) {
    reset();
    if (count == 0) count = 1;
    hipError_t e = hipMalloc(&p, count * sizeof(T));
    if (e == hipSuccess) n = count;
    return e;
  }
  hipError_t ensure(size_t count) { return count <= n ? hipSuccess : alloc(count + count / 2); }
};

template <typename T>
struct PinnedBuf {
  T *p = nullptr;
  size_t n = 0;
  ~PinnedBuf() { reset(); }
  void reset() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t ensure(size_t count) {
    if (count <= n && p) return hipSuccess;
    reset();
    size_t c = count + count / 2 + 16;
    hipError_t e = hipHostMalloc(&p, c * sizeof(T), hipHostMallocDefault);
    if (e == hipSuccess) n = c;
    return e;
  }
};

// Buffers of a batch's sort (host_delta), kept with the engine.
struct DeltaSort {
  std::vector<uint64_t> key[2];
  std::vector<uint32_t> pos[2];
};

uint8_t clamp_label(uint32_t l, const bool used[256]) { return (l < 255 && used[l]) ? (uint8_t)l : kNoLabel; }

}  // namespace

struct dsm_engine {
  dsm_options opt{};
  std::string err;
  hipStream_t stream = nullptr;
  int num_cu = 0;
  uint32_t n = 0;
  std::vector<QueryHost> queries;
  bool label_used[256] = {};

  // candidate signatures and plans
  std::vector<SigReq> sigs;
  std::vector<uint32_t> sig_lo, sig_hi;  // 256
  std::vector<uint8_t> lmap;             // 256
  std::vector<std::vector<uint16_t>> qsig;  // per query, per query vertex
  std::vector<Plan> plans;
  std::vector<uint32_t> plan_key;
  uint32_t max_plans_per_key = 0;
  std::vector<uint64_t> label_freq;  // data vertices per label (orders the matching only)

  // device graph
  DevBuf<uint32_t> pool, start, deg, cap;
  DevBuf<uint8_t> lab;
  DevBuf<uint32_t> lpool, loff;  // label-sorted copies of long lists
  // builds of the label-sorted copies (SortedBuild)
  DevBuf<uint32_t> build_ctl, build_mid, build_hist;
  DevBuf<uint2> build_big, build_pieces;
  uint32_t nbuckets = 1;
  unsigned long long pool_cap = 0;
  // filter
  DevBuf<uint64_t> bm;
  uint32_t words = 0;
  DevBuf<SigReq> d_sigs;
  DevBuf<uint32_t> d_sig_lo, d_sig_hi;
  DevBuf<uint8_t> d_lmap;
  DevBuf<Plan> d_plans;
  DevBuf<uint2> d_plan_of;
  // batch
  DevBuf<uint32_t> scratch;
  unsigned long long scratch_cap = 0;
  DevBuf<uint8_t> dirty_marks;
  DevBuf<uint32_t> dirty_list;
  DevBuf<uint32_t> bbuf;              // an update's arrays (device)
  PinnedBuf<uint32_t> hbuf;           // the same (pinned staging)
  PinnedBuf<uint32_t> hrec;           // a round's records (pinned staging)
  // the copies out of hbuf / hrec: done before either is filled again
  hipEvent_t ev_hbuf = nullptr, ev_hrec = nullptr;
  DevBuf<uint32_t> tinfo;             // per touched vertex: new degree, new inserts, slot, state
  DevBuf<unsigned long long> soff;
  DevBuf<uint2> segs;                 // pieces of the touched lists
  DevBuf<ApplyCtl> actl;
  PinnedBuf<ApplyCtl> h_actl;
  // DFS
  DevBuf<DfsCtl> ctl;
  DevBuf<Mailbox> mail;          // one per wave of the largest grid
  DevBuf<IdleWord> idle;         // their waiting states
  PinnedBuf<BlockRec> h_rec;     // what each block of the last DFS launch did
  uint32_t epoch = 0;            // of the last DFS launch
  DevBuf<uint32_t> seed_plan, seed_s, seed_d, seed_tag;
  uint32_t seed_cap = 0;
  // the tuple counter, then the match counts; both are cleared by the reset of
  // the round that follows counts_stale
  DevBuf<unsigned long long> results;
  PinnedBuf<unsigned long long> h_results;
  unsigned long long *tuple_count() { return results.p; }
  unsigned long long *counts() { return results.p + 1; }
  unsigned long long *h_counts() { return h_results.p + 1; }
  bool counts_stale = false;
  uint32_t *tuples = nullptr;
  bool tuples_host = false;
  unsigned long long tuple_cap = 0;
  uint32_t dfs_blocks = 0, dfs_wpb = 4, max_qn = 2;
  uint32_t donate_min = 256, lane_work = 16, donate_every = 4, donate_min_n2 = 64, leaf_budget = 8192;
  bool leaf_sets = true;
  bool bit_probe_last = false;
  bool seeding_timed = false;
  PinnedBuf<uint32_t> pipe_h_rec;  // records of a pipelined round (dsm_process_batches)
  DevBuf<uint32_t> pipe_d_rec;
  bool leaf_segments = true;
  uint32_t poll_max = 16;
  // Second copy of the graph: a pipelined round matches on the engine's copy
  // while the next batch is applied to this one on stream2; then they swap.
  struct GraphCopy {
    DevBuf<uint32_t> pool, start, deg, cap, lpool, loff;
    DevBuf<uint8_t> lab;
    DevBuf<uint64_t> bm;
    DevBuf<ApplyCtl> actl;
    unsigned long long pool_cap = 0;
  } shadow;
  hipStream_t stream2 = nullptr;
  hipEvent_t ev_pre = nullptr;  // all work on stream before a pipelined round
  bool overlap_apply = true;
  bool lpool_stale = false;  // the pool grew during the current update
  // The second copy of the graph differs from the current one only by the
  // last update, whose touched and relabelled vertices are kept here (its
  // dirty vertices stay on dirty_list): the next overlapped update copies just
  // those instead of the whole graph. Any other change clears it.
  bool shadow_delta_ok = false;
  bool grew = false;  // the pool grew during the update being applied
  std::vector<uint32_t> last_touched, last_relabel;
  DevBuf<uint32_t> sync_q;
  int cu_lds = 160 * 1024;   // LDS bytes per CU
  DevBuf<unsigned long long> query_busy;  // per query: DFS task ticks since the last read
  uint32_t wave_slots = 0;       // waves of the largest grid
  uint32_t last_blocks = 0, last_wpb = 0;  // grid of the last DFS launch
  uint32_t last_crew = 0;                  // its blocks that began at once
  uint32_t last_nrec = 0;                  // its records
  double busy_per_record = -1;             // most ms of task time a record in recent rounds (-1: no round yet)
  bool grid_given = false;                 // blocks_per_cu set by the caller or by dsm_autotune
  bool results_here = false;  // h_results holds the counts of the batch applied last
  uint32_t watchdog_ms = 60000;
  int wall_khz = 100000;
  DeltaSort delta_sort;  // used by one thread at a time: the caller, or the worker it waits for
  // records of the last batch (file order)
  std::vector<uint32_t> pos_s, pos_d, neg_s, neg_d;
  DevBuf<uint32_t> rec_neg, rec_pos;  // records on the device: src[k] | dst[k]
  bool batch_pending = false;
  hipEvent_t ev[12] = {};
  dsm_stats stats{};
  // cluster-encoding refinement (opt.cluster_filter): every query's position
  // rows follow the signature rows in bm; the DFS and the seeding read the
  // final positions
  bool cluster = false;
  uint32_t nsig_rows = 0, npos_rows = 0;
  std::vector<std::vector<uint32_t>> qref;  // per query, per vertex: the bitmap row the DFS uses
  std::vector<uint32_t> cstep_off;          // ops of pass step s: [cstep_off[s], cstep_off[s + 1])
  uint32_t cmax_step_ops = 0;
  DevBuf<ClusterOp> d_cops;
  DevBuf<uint32_t> d_crow, d_alive_src, cctl;
  uint32_t nalive_src = 0, nalive_rows = 0;
  DevBuf<uint64_t> calive;
  DevBuf<ClusterHeavy> cheavy;
  hipEvent_t ev_ref[2] = {};
  bool refine_timed = false;

  ~dsm_engine() {
    for (auto &x : ev_ref)
      if (x) (void)hipEventDestroy(x);
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
    if (tuples) {
      if (tuples_host) (void)hipHostFree(tuples);
      else (void)hipFree(tuples);
    }
    for (hipEvent_t x : {ev_pre, ev_hbuf, ev_hrec})
      if (x) (void)hipEventDestroy(x);
    if (stream2) (void)hipStreamDestroy(stream2);
    if (stream) (void)hipStreamDestroy(stream);
  }

  int fail_msg(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    err = buf;
    return code;
  }

  DevGraph dev_graph() {
    DevGraph g;
    g.n = n;
    g.pool = pool.p;
    g.start = start.p;
    g.deg = deg.p;
    g.cap = cap.p;
    g.lab = lab.p;
    g.lpool = lpool.p;
    g.loff = loff.p;
    g.nbuckets = nbuckets;
    return g;
  }
  FilterTables tables() {
    FilterTables t;
    t.sigs = d_sigs.p;
    t.sig_lo = d_sig_lo.p;
    t.sig_hi = d_sig_hi.p;
    t.lmap = d_lmap.p;
    t.nsig = (uint32_t)sigs.size();
    t.bm = bm.p;
    t.words = words;
    return t;
  }
  SortedBuild sorted_build() {
    SortedBuild h;
    h.ctl = build_ctl.p;
    h.mid = build_mid.p;
    h.big = build_big.p;
    h.pieces = build_pieces.p;
    h.hist = build_hist.p;
    // the merge scratch (at least one entry per pool entry) is idle while the
    // label-sorted copies are rebuilt
    h.bucket_bytes = scratch_cap >= pool_cap ? reinterpret_cast<uint8_t *>(scratch.p) : nullptr;
    h.actl = actl.p;
    return h;
  }
  DirtyArgs dirty() {
    DirtyArgs d;
    d.marks = dirty_marks.p;
    d.list = dirty_list.p;
    d.list_cap = n;
    d.actl = actl.p;
    return d;
  }
};

#define HIPCHK(expr)                                                                          \
  do {                                                                                        \
    hipError_t _e = (expr);                                                                   \
    if (_e != hipSuccess)                                                                     \
      return e->fail_msg(DSM_EDEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                         __FILE__, __LINE__);                                                 \
  } while (0)

namespace {

// ------------------------------------------------------------ query set-up

// The refinement's passes for every query (dsm_cluster_plan.cpp), as device
// ops grouped by pass step: step s holds pass s of every query that has one.
// Rows: position p of query q is bitmap row nsig + qbase[q] + p; the alive row
// of query vertex u of q is abase[q] + u.
int build_cluster_ops(dsm_engine *e, const dsm_query_desc *qs, uint32_t nq) {
  std::vector<ClusterPlan> plans(nq);
  std::vector<uint32_t> qbase(nq), abase(nq);
  uint32_t npos = 0, nalive = 0, nsteps = 0;
  for (uint32_t q = 0; q < nq; q++) {
    if (build_cluster_plan(qs[q].num_vertices, qs[q].num_edges, qs[q].edge_src, qs[q].edge_dst, plans[q]))
      return e->fail_msg(DSM_ELIMIT, "query %u: its cluster plan exceeds the reference's limits (%u clusters, "
                         "%u small clusters per combine)", q, kMaxClusters, kMaxSmallClusters);
    qbase[q] = npos;
    abase[q] = nalive;
    npos += plans[q].positions;
    nalive += e->queries[q].n;
    nsteps = std::max<uint32_t>(nsteps, (uint32_t)plans[q].passes.size());
  }
  if ((uint64_t)e->nsig_rows + npos > 65535)
    return e->fail_msg(DSM_ELIMIT, "cluster positions of the queries exceed 65,535 bitmap rows");
  const uint32_t nsig = e->nsig_rows;
  auto row = [&](uint32_t q, uint32_t p) { return nsig + qbase[q] + p; };
  std::vector<std::vector<ClusterOp>> steps(nsteps);
  std::vector<uint32_t> crow;
  std::vector<bool> core_alive(nalive, false);
  for (uint32_t q = 0; q < nq; q++) {
    const ClusterPlan &P = plans[q];
    const QueryHost &Q = e->queries[q];
    for (size_t s = 0; s < P.passes.size(); s++) {
      const auto &pass = P.passes[s];
      ClusterOp op{};
      const ClusterPlan::Cluster &c =
          P.clusters[pass.kind == ClusterPlan::kCombine ? P.combines[pass.arg].big : pass.arg];
      const uint32_t core = c.members[0];
      op.alive = abase[q] + core;
      core_alive[op.alive] = true;
      op.core = row(q, c.pos);
      op.ntarget = (uint32_t)c.members.size() - 1;
      op.check_off = (uint32_t)crow.size();
      for (uint32_t t = 0; t < op.ntarget; t++) {
        op.tlab[t] = (uint8_t)Q.lab[c.members[t + 1]];
        op.tlix[t] = e->lmap[Q.lab[c.members[t + 1]]];
        bool seen = false;
        for (uint32_t k = 0; k < op.nlix; k++) seen = seen || op.lix[k] == op.tlix[t];
        if (!seen) op.lix[op.nlix++] = op.tlix[t];
      }
      if (pass.kind == ClusterPlan::kEncode) {
        // encodeKernel: a neighbour of a core candidate is a target's candidate
        op.kind = kOpEncode;
        for (uint32_t t = 0; t < op.ntarget; t++) {
          op.toff[t] = (uint16_t)crow.size();
          op.tcnt[t] = 1;
          crow.push_back(e->qsig[q][c.members[t + 1]]);
        }
      } else if (pass.kind == ClusterPlan::kMerge) {
        // mergeKernel: the core in both merged clusters; the targets are the
        // merged clusters' cores
        op.kind = kOpMerge;
        crow.push_back(row(q, c.left_pos));
        crow.push_back(row(q, c.right_pos));
        op.ncheck = 2;
        const uint32_t src[2] = {P.clusters[c.left].pos, P.clusters[c.right].pos};
        for (uint32_t t = 0; t < op.ntarget; t++) {
          op.toff[t] = (uint16_t)crow.size();
          op.tcnt[t] = 1;
          crow.push_back(row(q, src[t]));
        }
      } else {
        // combineMultipleClustersKernel: the core in every small cluster; a
        // target in every small cluster that holds it
        const ClusterPlan::Combine &cb = P.combines[pass.arg];
        op.kind = cb.keep ? kOpCombineKeep : kOpCombineNew;
        for (uint32_t sm : cb.small) crow.push_back(row(q, P.clusters[sm].pos));
        op.ncheck = (uint32_t)cb.small.size();
        for (uint32_t t = 0; t < op.ntarget; t++) {
          op.toff[t] = (uint16_t)crow.size();
          const uint32_t tu = c.members[t + 1];
          for (uint32_t sm : cb.small) {
            const auto &mm = P.clusters[sm].members;
            for (size_t x = 1; x < mm.size(); x++)
              if (mm[x] == tu) {
                crow.push_back(row(q, P.clusters[sm].pos + (uint32_t)x));
                break;
              }
          }
          op.tcnt[t] = (uint16_t)(crow.size() - op.toff[t]);
        }
      }
      if (crow.size() > 65535) return e->fail_msg(DSM_ELIMIT, "cluster plans too large");
      steps[s].push_back(op);
    }
    for (uint32_t u = 0; u < Q.n; u++) e->qref[q][u] = row(q, P.final_pos[u]);
  }
  std::vector<ClusterOp> ops;
  e->cstep_off.assign(1, 0);
  e->cmax_step_ops = 0;
  for (auto &st : steps) {
    ops.insert(ops.end(), st.begin(), st.end());
    e->cstep_off.push_back((uint32_t)ops.size());
    e->cmax_step_ops = std::max<uint32_t>(e->cmax_step_ops, (uint32_t)st.size());
  }
  // alive rows: every core's candidate list starts as its LDF/NLF row
  std::vector<uint32_t> asrc;
  for (uint32_t q = 0; q < nq; q++)
    for (uint32_t u = 0; u < e->queries[q].n; u++)
      if (core_alive[abase[q] + u]) {
        asrc.push_back(abase[q] + u);
        asrc.push_back(e->qsig[q][u]);
      }
  e->npos_rows = npos;
  e->nalive_rows = nalive;
  e->nalive_src = (uint32_t)asrc.size() / 2;
  HIPCHK(e->d_cops.alloc(ops.size()));
  HIPCHK(hipMemcpy(e->d_cops.p, ops.data(), ops.size() * sizeof(ClusterOp), hipMemcpyHostToDevice));
  HIPCHK(e->d_crow.alloc(crow.size()));
  if (!crow.empty()) HIPCHK(hipMemcpy(e->d_crow.p, crow.data(), crow.size() * 4, hipMemcpyHostToDevice));
  HIPCHK(e->d_alive_src.alloc(asrc.size()));
  if (!asrc.empty()) HIPCHK(hipMemcpy(e->d_alive_src.p, asrc.data(), asrc.size() * 4, hipMemcpyHostToDevice));
  HIPCHK(e->cctl.alloc(std::max<uint32_t>(nsteps, 1)));
  for (auto &x : e->ev_ref) HIPCHK(hipEventCreate(&x));
  return DSM_OK;
}

// The plans: every query edge in both orientations, each with its matching
// order (the query's order rule), grouped by the seed edge's label pair.
void build_plans(dsm_engine *e) {
  // plans: every query edge in both orientations
  struct PK {
    uint32_t key;
    Plan p;
  };
  std::vector<PK> pk;
  const uint32_t nq = (uint32_t)e->queries.size();
  for (uint32_t q = 0; q < nq; q++) {
    const QueryHost &Q = e->queries[q];
    for (uint32_t u = 0; u < Q.n; u++)
      for (uint32_t v = 0; v < Q.n; v++) {
        if (!(Q.adj[u] >> v & 1)) continue;
        Plan P{};
        P.n = (uint8_t)Q.n;
        P.query = (uint16_t)q;
        uint32_t order[kMaxQ];
        order[0] = u;
        order[1] = v;
        uint32_t placed = (1u << u) | (1u << v);
        for (uint32_t k = 2; k < Q.n; k++) {
          order[k] = next_in_order(Q, placed, e->label_freq, Q.order_variant);
          placed |= 1u << order[k];
        }
        for (uint32_t k = 0; k < Q.n; k++) {
          P.qv[k] = (uint8_t)order[k];
          P.sig[k] = (uint16_t)e->qref[q][order[k]];
          uint16_t back = 0, inj = 0;
          for (uint32_t j = 0; j < k; j++) {
            if (Q.adj[order[k]] >> order[j] & 1) back |= (uint16_t)(1u << j);
            if (Q.lab[order[j]] == Q.lab[order[k]]) inj |= (uint16_t)(1u << j);
          }
          P.back[k] = back;
          P.inj[k] = inj;
          P.lix[k] = e->lmap[Q.lab[order[k]]];
        }
        pk.push_back({(Q.lab[u] << 8) | Q.lab[v], P});
      }
  }
  std::stable_sort(pk.begin(), pk.end(), [](const PK &a, const PK &b) { return a.key < b.key; });
  e->plans.clear();
  e->plan_key.clear();
  e->max_plans_per_key = 0;
  for (size_t i = 0; i < pk.size();) {
    size_t j = i;
    while (j < pk.size() && pk[j].key == pk[i].key) j++;
    e->max_plans_per_key = std::max<uint32_t>(e->max_plans_per_key, (uint32_t)(j - i));
    i = j;
  }
  for (auto &x : pk) {
    e->plans.push_back(x.p);
    e->plan_key.push_back(x.key);
  }}

// label_freq[l]: data vertices of label l (l < 255), used only to order the
// matching: it never changes a count.
int build_queries(dsm_engine *e, const dsm_query_desc *qs, uint32_t nq, const std::vector<uint64_t> &label_freq) {
  if (nq == 0 || nq > DSM_MAX_QUERIES) return e->fail_msg(DSM_EINVAL, "need 1..%d queries", DSM_MAX_QUERIES);
  e->queries.resize(nq);
  for (uint32_t q = 0; q < nq; q++) {
    const dsm_query_desc &d = qs[q];
    QueryHost &Q = e->queries[q];
    if (d.num_vertices < 2 || d.num_vertices > (uint32_t)kMaxQ)
      return e->fail_msg(DSM_ELIMIT, "query %u: %u vertices (2..%d supported)", q, d.num_vertices, kMaxQ);
    Q.n = d.num_vertices;
    for (uint32_t u = 0; u < Q.n; u++) {
      if (d.labels[u] > DSM_MAX_LABEL)
        return e->fail_msg(DSM_ELIMIT, "query %u: label %u > %d", q, d.labels[u], DSM_MAX_LABEL);
      Q.lab[u] = d.labels[u];
      e->label_used[d.labels[u]] = true;
    }
    for (uint32_t i = 0; i < d.num_edges; i++) {
      uint32_t a = d.edge_src[i], b = d.edge_dst[i];
      if (a >= Q.n || b >= Q.n || a == b) return e->fail_msg(DSM_EINVAL, "query %u: bad edge %u-%u", q, a, b);
      Q.adj[a] |= 1u << b;
      Q.adj[b] |= 1u << a;
    }
    // connected (every later DFS position needs an earlier neighbour)
    uint32_t seen = 1, frontier = 1;
    while (frontier) {
      uint32_t nf = 0;
      for (uint32_t u = 0; u < Q.n; u++)
        if (frontier >> u & 1) nf |= Q.adj[u];
      frontier = nf & ~seen;
      seen |= nf;
    }
    if (seen != ((1u << Q.n) - 1)) return e->fail_msg(DSM_EINVAL, "query %u is not connected", q);
  }
  // relevant labels: those of query vertices with a neighbour (all of them)
  e->lmap.assign(256, 0xFF);
  uint32_t nrel = 0;
  for (uint32_t l = 0; l < 255; l++)
    if (e->label_used[l]) {
      if (nrel == (uint32_t)kMaxRel)
        return e->fail_msg(DSM_ELIMIT, "queries use more than %d distinct labels", kMaxRel);
      e->lmap[l] = (uint8_t)nrel++;
    }
  // signatures: (label, degree, neighbour-label counts) of every query vertex
  std::map<std::vector<uint64_t>, uint32_t> sigidx;
  std::vector<SigReq> tmp;
  e->qsig.assign(nq, std::vector<uint16_t>());
  for (uint32_t q = 0; q < nq; q++) {
    const QueryHost &Q = e->queries[q];
    e->qsig[q].resize(Q.n);
    for (uint32_t u = 0; u < Q.n; u++) {
      SigReq r{};
      r.label = Q.lab[u];
      r.deg = (uint32_t)__builtin_popcount(Q.adj[u]);
      uint8_t cnt[kMaxRel] = {};
      for (uint32_t w = 0; w < Q.n; w++)
        if (Q.adj[u] >> w & 1) cnt[e->lmap[Q.lab[w]]]++;
      for (int l = 0; l < kMaxRel; l++) r.nlc[l >> 3] |= (uint64_t)cnt[l] << ((l & 7) * 8);
      std::vector<uint64_t> key = {r.label, r.deg, r.nlc[0], r.nlc[1], r.nlc[2], r.nlc[3]};
      auto it = sigidx.find(key);
      if (it == sigidx.end()) {
        it = sigidx.emplace(key, (uint32_t)tmp.size()).first;
        tmp.push_back(r);
      }
      e->qsig[q][u] = (uint16_t)it->second;
    }
  }
  if (tmp.size() > 65535) return e->fail_msg(DSM_ELIMIT, "too many distinct query vertex signatures");
  // sort signatures by label; remap
  std::vector<uint32_t> ord(tmp.size());
  for (uint32_t i = 0; i < ord.size(); i++) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) { return tmp[a].label < tmp[b].label; });
  std::vector<uint32_t> newidx(tmp.size());
  e->sigs.resize(tmp.size());
  for (uint32_t i = 0; i < ord.size(); i++) {
    e->sigs[i] = tmp[ord[i]];
    newidx[ord[i]] = i;
  }
  for (auto &v : e->qsig)
    for (auto &s : v) s = (uint16_t)newidx[s];
  e->sig_lo.assign(256, 0);
  e->sig_hi.assign(256, 0);
  for (uint32_t i = 0; i < e->sigs.size(); i++) {
    uint32_t l = e->sigs[i].label;
    if (e->sig_hi[l] == 0) e->sig_lo[l] = i;
    e->sig_hi[l] = i + 1;
  }
  // cluster-encoding refinement: position rows after the signature rows
  e->nsig_rows = (uint32_t)e->sigs.size();
  e->qref.assign(nq, std::vector<uint32_t>());
  for (uint32_t q = 0; q < nq; q++)
    for (uint32_t u = 0; u < e->queries[q].n; u++) e->qref[q].push_back(e->qsig[q][u]);
  if (e->cluster) {
    if (int rc = build_cluster_ops(e, qs, nq)) return rc;
  }
  e->label_freq = label_freq;
  build_plans(e);

  return DSM_OK;
}

// ------------------------------------------------------------- graph set-up

// Queues of the label-sorted builds: every vertex once among the short lists; at
// most pool / kBuildSeg lists are longer, in at most twice as many pieces.
int size_sorted_build(dsm_engine *e) {
  const size_t lists = (size_t)(e->pool_cap / kBuildSeg) + 1;
  if (lists > e->build_big.n) {
    HIPCHK(e->build_big.alloc(lists));
    HIPCHK(e->build_pieces.alloc(2 * lists));
    HIPCHK(e->build_hist.alloc(2 * lists * (kMaxRel + 2)));
  }
  if (!e->build_ctl.p) {
    HIPCHK(e->build_ctl.alloc(4));
    HIPCHK(e->build_mid.alloc(e->n));
  }
  return DSM_OK;
}

int upload_graph(dsm_engine *e, const dsm_graph_desc *g) {
  const uint32_t n = g->num_vertices;
  const uint64_t m = g->num_edges;
  const size_t count = 2 * m;
  const uint32_t bits = n > 1 ? 32u - (uint32_t)__builtin_clz(n - 1) : 1u;
  // the sort's buffers go before the pool's copies come, which are larger
  DevBuf<unsigned long long> keys[2], hist, sums, slot;
  DevBuf<uint32_t> begin;
  DevBuf<CsrCtl> ctl;
  CsrCtl c0{~0ull, 0, 0, 0, 0};
  HIPCHK(ctl.alloc(1));
  HIPCHK(hipMemcpy(ctl.p, &c0, sizeof c0, hipMemcpyHostToDevice));
  HIPCHK(sums.alloc(csr_sum_words(std::max<size_t>(csr_scan_words(count), n))));
  uint32_t cur = 0;
  if (m) {
    for (auto &k : keys) HIPCHK(k.alloc(count));
    HIPCHK(hist.alloc(csr_scan_words(count)));
    // the edges lie in the buffer that the first pass fills
    uint32_t *edges = reinterpret_cast<uint32_t *>(keys[1].p);
    HIPCHK(hipMemcpyAsync(edges, g->edge_src, m * 4, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipMemcpyAsync(edges + m, g->edge_dst, m * 4, hipMemcpyHostToDevice, e->stream));
    HIPCHK(launch_csr_keys(edges, edges + m, m, n, bits, keys[0].p, ctl.p, e->stream));
    for (uint32_t shift = 0; shift < 2 * bits; shift += 8, cur ^= 1)
      HIPCHK(launch_radix_pass(keys[cur].p, keys[cur ^ 1].p, count, shift, hist.p, sums.p, e->stream));
    HIPCHK(launch_csr_unique(keys[cur].p, keys[cur ^ 1].p, count, hist.p, sums.p, ctl.p, e->stream));
    cur ^= 1;
  }
  HIPCHK(e->start.alloc(n));
  HIPCHK(e->deg.alloc(n));
  HIPCHK(e->cap.alloc(n));
  HIPCHK(begin.alloc(n));
  HIPCHK(slot.alloc(n));
  HIPCHK(hipMemsetAsync(e->deg.p, 0, (size_t)n * 4, e->stream));
  HIPCHK(launch_csr_slots(keys[cur].p, count, n, bits, begin.p, e->deg.p, e->cap.p, e->start.p, slot.p, sums.p, ctl.p,
                          e->stream));
  std::vector<uint8_t> hl(n);
  for (uint32_t v = 0; v < n; v++) hl[v] = clamp_label(g->labels[v], e->label_used);
  HIPCHK(hipStreamSynchronize(e->stream));
  HIPCHK(hipMemcpy(&c0, ctl.p, sizeof c0, hipMemcpyDeviceToHost));
  if (c0.bad != ~0ull) return e->fail_msg(DSM_EINVAL, "edge %llu: endpoint out of range", c0.bad);
  const unsigned long long total = c0.total, pcap = total + total / 2 + (1ull << 20);
  if (c0.unique >= (1ull << 32) || pcap >= (1ull << 32))
    return e->fail_msg(DSM_ELIMIT, "graph too large for 32-bit pool offsets");
  keys[cur ^ 1].reset();
  hist.reset();
  HIPCHK(e->pool.alloc(pcap));
  HIPCHK(launch_csr_fill(keys[cur].p, count, bits, begin.p, e->start.p, e->pool.p, ctl.p, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  keys[cur].reset();
  HIPCHK(e->lab.alloc(((size_t)n + 15) / 16 * 16));  // read 16 at a time
  HIPCHK(e->lpool.alloc(pcap));
  e->nbuckets = 1;
  for (int l = 0; l < 255; l++)
    if (e->lmap[l] != 0xFF) e->nbuckets = std::max<uint32_t>(e->nbuckets, e->lmap[l] + 2u);
  HIPCHK(e->loff.alloc((size_t)n * (e->nbuckets + 1)));
  e->pool_cap = pcap;
  if (int rc = size_sorted_build(e)) return rc;
  HIPCHK(hipMemcpy(e->lab.p, hl.data(), n, hipMemcpyHostToDevice));
  // scratch holds one merged copy of every touched list
  e->scratch_cap = pcap + (1ull << 20);
  HIPCHK(e->scratch.alloc(e->scratch_cap));
  HIPCHK(e->actl.alloc(1));
  HIPCHK(e->h_actl.ensure(1));
  ApplyCtl a0{};
  a0.pool_used = total;
  a0.max_deg = c0.max_deg;
  HIPCHK(hipMemcpy(e->actl.p, &a0, sizeof a0, hipMemcpyHostToDevice));
  *e->h_actl.p = a0;
  HIPCHK(e->dirty_marks.alloc(((size_t)n + 15) / 16 * 16));
  HIPCHK(hipMemset(e->dirty_marks.p, 0, e->dirty_marks.n));
  HIPCHK(e->dirty_list.alloc(n));
  return DSM_OK;
}

int upload_tables(dsm_engine *e) {
  e->words = (e->n + 63) / 64;
  const size_t rows = (size_t)e->nsig_rows + e->npos_rows;
  HIPCHK(e->bm.alloc(rows * e->words));
  HIPCHK(hipMemset(e->bm.p, 0, rows * e->words * 8));
  if (e->cluster) HIPCHK(e->calive.alloc((size_t)e->nalive_rows * e->words));
  HIPCHK(e->d_sigs.alloc(e->sigs.size()));
  HIPCHK(hipMemcpy(e->d_sigs.p, e->sigs.data(), e->sigs.size() * sizeof(SigReq), hipMemcpyHostToDevice));
  HIPCHK(e->d_sig_lo.alloc(256));
  HIPCHK(e->d_sig_hi.alloc(256));
  HIPCHK(e->d_lmap.alloc(256));
  HIPCHK(hipMemcpy(e->d_sig_lo.p, e->sig_lo.data(), 256 * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(e->d_sig_hi.p, e->sig_hi.data(), 256 * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(e->d_lmap.p, e->lmap.data(), 256, hipMemcpyHostToDevice));
  HIPCHK(e->d_plans.alloc(e->plans.size()));
  HIPCHK(hipMemcpy(e->d_plans.p, e->plans.data(), e->plans.size() * sizeof(Plan), hipMemcpyHostToDevice));
  std::vector<uint2> plan_of(kMaxRel * kMaxRel, uint2{0, 0});
  for (size_t i = 0; i < e->plan_key.size(); i++) {
    const uint32_t l0 = e->lmap[e->plan_key[i] >> 8], l1 = e->lmap[e->plan_key[i] & 0xFF];
    uint2 &x = plan_of[l0 * kMaxRel + l1];
    if (x.y++ == 0) x.x = (uint32_t)i;
  }
  HIPCHK(e->d_plan_of.alloc(plan_of.size()));
  HIPCHK(hipMemcpy(e->d_plan_of.p, plan_of.data(), plan_of.size() * sizeof(uint2), hipMemcpyHostToDevice));
  const uint32_t nq = (uint32_t)e->queries.size();
  HIPCHK(e->results.alloc((size_t)nq * 2 * kMaxSlots + 1));
  HIPCHK(e->query_busy.alloc(nq));
  HIPCHK(hipMemset(e->query_busy.p, 0, (size_t)nq * 8));
  HIPCHK(e->h_results.ensure((size_t)nq * 2 * kMaxSlots + 1));
  HIPCHK(e->ctl.alloc(1));
  if (e->opt.tuple_capacity) {
    e->tuple_cap = e->opt.tuple_capacity;
    size_t bytes = (size_t)e->tuple_cap * (kMaxQ + 2) * 4;
    if (e->opt.tuples_in_host_memory) {
      HIPCHK(hipHostMalloc((void **)&e->tuples, bytes, hipHostMallocMapped));
      e->tuples_host = true;
    } else {
      HIPCHK(hipMalloc((void **)&e->tuples, bytes));
    }
  }
  return DSM_OK;
}

// ------------------------------------------------------------- DFS rounds

int ensure_seed_cap(dsm_engine *e, uint32_t nrec) {
  const uint64_t need = (uint64_t)nrec * std::max<uint32_t>(e->max_plans_per_key, 1);
  if (need > 0xFFFFFFF0ull) return e->fail_msg(DSM_ELIMIT, "seed table too large");
  if (need > e->seed_cap) {
    uint32_t c = (uint32_t)std::min<uint64_t>(need + need / 2 + 1024, 0xFFFFFFF0ull);
    HIPCHK(e->seed_plan.alloc(c));
    HIPCHK(e->seed_s.alloc(c));
    HIPCHK(e->seed_d.alloc(c));
    HIPCHK(e->seed_tag.alloc(c));
    e->seed_cap = c;
  }
  return DSM_OK;
}

// A DFS round: reset the control block (and the results with counts_stale, or
// a count slot), seed up to two record lists (each with its count tag, slot << 1
// | sign), one persistent DFS launch over all their seeds. The seed table must
// hold the seeds of both lists.
struct RoundPart {
  const uint32_t *rs, *rd;
  uint32_t n, tag;
};
struct ClearSpan {
  unsigned long long *tuple_count, *counts;
  uint32_t ncounts;
};

SeedArgs seed_args(dsm_engine *e, const RoundPart *parts, int nparts) {
  SeedArgs sa;
  sa.g = e->dev_graph();
  sa.bm = e->bm.p;
  sa.words = e->words;
  sa.plans = e->d_plans.p;
  sa.lmap = e->d_lmap.p;
  sa.plan_of = e->d_plan_of.p;
  sa.nplans = (uint32_t)e->plans.size();
  for (int i = 0; i < 2; i++) {
    sa.rs[i] = i < nparts ? parts[i].rs : nullptr;
    sa.rd[i] = i < nparts ? parts[i].rd : nullptr;
    sa.nrec[i] = i < nparts ? parts[i].n : 0;
    sa.tag[i] = i < nparts ? parts[i].tag : 0;
  }
  sa.seed_plan = e->seed_plan.p;
  sa.seed_s = e->seed_s.p;
  sa.seed_d = e->seed_d.p;
  sa.seed_tag = e->seed_tag.p;
  sa.seed_cap = e->seed_cap;
  sa.ctl = e->ctl.p;
  return sa;
}

DfsArgs dfs_args(dsm_engine *e) {
  DfsArgs da;
  da.g = e->dev_graph();
  da.bm = e->bm.p;
  da.words = e->words;
  da.plans = e->d_plans.p;
  da.seed_plan = e->seed_plan.p;
  da.seed_s = e->seed_s.p;
  da.seed_d = e->seed_d.p;
  da.seed_tag = e->seed_tag.p;
  da.mail = e->mail.p;
  da.idle = e->idle.p;
  da.donate_cap = e->opt.queue_capacity ? e->opt.queue_capacity - 1 : kNoDonateCap;
  da.epoch = ++e->epoch;
  da.donate_min = e->donate_min;
  da.lane_work = e->lane_work;
  da.leaf_budget = e->leaf_budget;
  da.bit_probe_last = e->bit_probe_last ? 1u : 0u;
  da.fshift = 0;
  while ((e->n > 0 ? (e->n - 1) >> da.fshift : 0u) >= 512u) da.fshift++;
  da.donate_every = e->donate_every;
  da.donate_min_n2 = e->donate_min_n2;
  da.leaf_segments = e->leaf_segments ? 1u : 0u;
  da.poll_max = e->poll_max;
  da.leaf_sets = e->leaf_sets ? 1u : 0u;
  da.nq = (uint32_t)e->queries.size();
  da.watchdog = (unsigned long long)e->wall_khz * e->watchdog_ms;
  da.ctl = e->ctl.p;
  da.counts = e->counts();
  da.tuples = e->tuples;
  da.tuple_cap = e->tuple_cap;
  da.tuple_count = e->tuple_count();
  da.rec = e->h_rec.p;
  da.query_busy = e->query_busy.p;
  return da;
}

// The blocks that begin a round with so much task time (ms, as the engine's recent
// rounds took it a record). Waves share a CU's issue slots and L1: at 12 a CU they take
// twice as long for a task as at 4, and a round that ends with a few long tasks ends
// sooner with 4. Measured at 4, 8 and 12 waves a CU: 20 ms of tasks (22 seeds, 100,000
// vertices) 87, 100 and 106 us; 170 ms 186, 185 and 205; 270 ms 223, 221 and 220;
// 880 ms (1,000,000 vertices) 541, 499 and 513; 2,600 ms 1,320, 932 and 948; 9,900 ms
// 6.8, 4.3 and 3.7 ms.
//
// As many more as give every CU four waves are a reserve that joins the round when it has
// lasted kJoinUs, so that heavy records after light ones do not stay with the few waves
// that those need: 400 records of squares over lists of 1,000 entries after 300 rounds of
// lists of two take 17.7 ms, without the reserve 32.1, and 9.9 with all blocks from the
// start. (All other blocks as a reserve: 12.8 ms, but the light rounds take 91 us, not 87
// or, without a reserve, 83. Joining after 100 or 400 us makes no difference.)
constexpr uint32_t kJoinUs = 200;
uint32_t dfs_layer(const dsm_engine *e) { return std::max(1u, 4 / e->dfs_wpb) * (uint32_t)e->num_cu; }
uint32_t blocks_for_work(const dsm_engine *e, double ms) {
  return ms <= 250 ? dfs_layer(e) : ms <= 2500 ? 2 * dfs_layer(e) : 0xFFFF0000u;
}

// The grid: a round over a handful of records gets one block per CU, so that few
// waves pay the start-up and termination atomics, and fewer where neither a list is long
// enough to give a CU's waves anything to share nor a query deep enough: a 4-vertex query
// on lists of 30 entries is matched by a few waves, and 256 blocks' records cost more than
// that. What a seed can expand is at most the longest list's length to the power of the
// positions after it. One record, lists of 16 entries, paths of 6, 7 and 8 vertices, in
// two calls: 317, 992 and 7,061 us with a block per 4,096 entries of that, 334, 997 and
// 7,109 per 16,384, 476, 4,109 and 58,452 by the lists' length alone; of 5 vertices 202
// with either.
uint32_t dfs_grid(dsm_engine *e, uint32_t nrec) {
  const uint64_t want =
      ((uint64_t)nrec * std::max<uint32_t>(e->max_plans_per_key, 1) * 8 + e->dfs_wpb - 1) / e->dfs_wpb;
  const uint32_t longest = e->h_actl.p->max_deg;
  uint64_t tree = 1;
  for (uint32_t l = 2; l < e->max_qn && tree < (1ull << 32); l++) tree *= longest;
  const uint64_t share = std::max<uint64_t>({1, longest / 16, tree / 4096});
  const uint64_t least = share >= (uint64_t)e->num_cu ? (uint64_t)e->num_cu
                                                      : std::min<uint64_t>((uint64_t)e->num_cu, want * share);
  uint32_t b = (uint32_t)std::min<uint64_t>(e->dfs_blocks, std::max<uint64_t>(want, least));
  e->last_nrec = nrec;
  e->last_wpb = e->tuples ? 4u : e->dfs_wpb;
  b = std::min(b, e->wave_slots / e->last_wpb);  // a mailbox for every wave
  uint32_t crew = b;
  if (!e->grid_given && e->busy_per_record >= 0) crew = std::min(b, blocks_for_work(e, e->busy_per_record * nrec));
  e->last_crew = crew;
  e->last_blocks = std::min(b, crew + dfs_layer(e));
  return e->last_blocks;
}

// The waiting words of a grid.
uint32_t idle_words(uint32_t waves) { return (waves + kIdleGroup - 1) / kIdleGroup; }

// One round. ev0 / ev1 / ev2 (may be null) mark its start, the end of seeding (its
// start, unless seeding is timed on its own) and its end; `up` brings the records,
// where they have not been sent. Three launches: as one HIP graph with its nodes
// updated for every round, a round of 11 us of kernels took 25 to 28 us on the
// device (a call with 8 records on a dense graph: 165 us, with launches 117).
int dfs_round(dsm_engine *e, const RoundPart *parts, int nparts, hipEvent_t ev0, hipEvent_t ev1,
              hipEvent_t ev2, const SmallCopy &up, ClearSpan clear = {}) {
  uint32_t nrec = 0;
  for (int i = 0; i < nparts; i++) nrec += parts[i].n;
  if (e->counts_stale) {
    clear = ClearSpan{e->tuple_count(), e->counts(), (uint32_t)e->queries.size() * 2};
    e->counts_stale = false;
  }
  if (ev0) HIPCHK(hipEventRecord(ev0, e->stream));
  e->results_here = false;
  if (ev1 && !e->seeding_timed) HIPCHK(hipEventRecord(ev1, e->stream));
  DfsArgs da = dfs_args(e);
  const uint32_t blocks = dfs_grid(e, nrec);
  da.crew = e->last_crew * e->last_wpb;
  da.cgroups = idle_words(da.crew);
  da.ngroups = da.cgroups + idle_words((blocks - e->last_crew) * e->last_wpb);
  da.join_after = (unsigned long long)e->wall_khz * kJoinUs / 1000;
  HIPCHK(launch_ctl_reset(e->ctl.p, clear.tuple_count, clear.counts, clear.ncounts, e->idle.p,
                          da.ngroups, up, e->stream));
  HIPCHK(launch_seed(seed_args(e, parts, nparts), e->stream));
  if (ev1 && e->seeding_timed) HIPCHK(hipEventRecord(ev1, e->stream));
  HIPCHK(launch_dfs(da, blocks, e->dfs_wpb, e->max_qn, e->stream));
  if (ev2) HIPCHK(hipEventRecord(ev2, e->stream));
  return DSM_OK;
}

// count values to pinned host memory.
template <typename T>
hipError_t to_host(T *to, const T *from, size_t count, hipStream_t s) {
  const size_t words = count * sizeof(T) / 4;
  if (words <= kSmallCopy && ((uintptr_t)from & 7) == 0 && ((uintptr_t)to & 7) == 0)
    return launch_small_copy({reinterpret_cast<const uint32_t *>(from), reinterpret_cast<uint32_t *>(to),
                              (uint32_t)words}, s);
  return hipMemcpyAsync(to, from, count * sizeof(T), hipMemcpyDeviceToHost, s);
}

// The tuple counter and the counts of slot 0 to the host; waits for the stream.
int fetch_results(dsm_engine *e) {
  const uint32_t n = (uint32_t)e->queries.size() * 2;
  if (e->counts_stale) HIPCHK(launch_ctl_reset(nullptr, e->tuple_count(), e->counts(), n, nullptr, 0, {}, e->stream));
  e->counts_stale = false;
  HIPCHK(to_host(e->h_results.p, e->results.p, n + 1, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return DSM_OK;
}

int run_round(dsm_engine *e, const uint32_t *rs, const uint32_t *rd, uint32_t nrec, uint32_t tag,
              hipEvent_t ev0, hipEvent_t ev1, hipEvent_t ev2, const SmallCopy &up = {}) {
  const RoundPart p{rs, rd, nrec, tag};
  if (int rc = dfs_round(e, &p, 1, ev0, ev1, ev2, up)) return rc;
  if (up.words) HIPCHK(hipEventRecord(e->ev_hrec, e->stream));
  return DSM_OK;
}

// The last round's errors: the records of its blocks, which have ended; and its work
// for the grids of later rounds.
int round_error(dsm_engine *e) {
  unsigned long long busy = 0;
  for (uint32_t b = 0; b < e->last_blocks; b++) {
    const BlockRec &r = e->h_rec.p[b];
    if (r.epoch != e->epoch) {
      if (b >= e->last_crew) continue;  // the round did without it
      return e->fail_msg(DSM_EDEVICE, "DFS: block %u of %u left no record", b, e->last_blocks);
    }
    if (r.seed_overflow)
      return e->fail_msg(DSM_ELIMIT, "seed table overflow (%llu seeds dropped)", r.seed_overflow);
    if (r.abort) return e->fail_msg(DSM_EDEVICE, "DFS watchdog: a wave waited more than %u ms for work", e->watchdog_ms);
    busy += r.busy;
  }
  if (e->last_nrec) {
    const double x = (double)busy / (double)e->wall_khz / e->last_nrec;
    // the most, fading: light rounds in between leave the heavy ones their grid
    e->busy_per_record = std::max(x, 0.97 * e->busy_per_record);
  }
  return DSM_OK;
}

// The last round's errors, and its work and balance into the statistics.
int check_round(dsm_engine *e, uint64_t *seeds) {
  if (int rc = round_error(e)) return rc;
  uint32_t nb = 0;  // blocks that took part
  *seeds = e->last_blocks ? e->h_rec.p[0].nseeds : 0;
  unsigned long long busy = 0, busiest = 0, active = 0, t0 = ~0ull, t1 = 0;
  double first = 0, last = 0;  // summed over the active waves
  for (uint32_t b = 0; b < e->last_blocks; b++) {
    const BlockRec &r = e->h_rec.p[b];
    if (r.epoch != e->epoch) continue;
    nb++;
    e->stats.tasks_donated += r.donated;
    e->stats.dfs_entries += r.scanned;
    e->stats.dfs_search_loads += r.loads;
    e->stats.dfs_merge_bytes += r.mbytes;
    busy += r.busy;
    busiest = std::max(busiest, r.busy);
    if (!r.active) continue;
    active += r.active;
    t0 = std::min(t0, r.first_min);
    t1 = std::max(t1, r.last_max);
    first += (double)r.first_sum;
    last += (double)r.last_sum;
  }
  const uint32_t nw = nb * e->last_wpb;
  e->stats.dfs_busy_ms += (double)busy / (double)e->wall_khz;
  e->stats.dfs_waves += nw;
  if (busy) e->stats.dfs_block_imbalance += (double)busiest / ((double)busy / nb);
  // head and tail idle: a wave without tasks counts as idle in the tail
  if (t1 > t0) {
    const double span = (double)(t1 - t0), na = (double)active;
    e->stats.dfs_head_idle += (first - na * (double)t0) / (span * nw);
    e->stats.dfs_tail_idle += (na * (double)t1 - last + span * (nw - na)) / (span * nw);
  }
  e->stats.dfs_launches += 1;
  return DSM_OK;
}

// ------------------------------------------------------------ apply rounds

// Inserts and deletes per touched vertex (ascending), at most kMaxVertexChanges of
// each in one round of merges and commits: an update with more on one vertex takes
// several rounds.
struct Slice {
  std::vector<uint32_t> tv, ioff, doff, ins, del;
};
// A batch's update: all its changes and relabels.
struct HostDelta : Slice {
  std::vector<uint32_t> rl_v, rl_l;
};

// Sorts keys[0, n), and pos with them, by the low `bits` bits of both halves of
// the keys, stably: a counting pass per digit of at most 11 bits, low half first.
// Returns which of the two buffers holds the result.
uint32_t sort_pairs(DeltaSort &w, size_t n, uint32_t bits) {
  const uint32_t digits = (bits + 10) / 11, width = (bits + digits - 1) / digits;
  const uint64_t mask = (1ull << width) - 1;
  uint32_t cur = 0;
  for (uint32_t pass = 0; pass < 2 * digits; pass++) {
    const uint32_t shift = pass < digits ? pass * width : 32 + (pass - digits) * width;
    uint32_t at[2048] = {};
    const uint64_t *k = w.key[cur].data();
    for (size_t i = 0; i < n; i++) at[k[i] >> shift & mask]++;
    uint32_t run = 0;
    for (uint64_t x = 0; x <= mask; x++) {
      const uint32_t c = at[x];
      at[x] = run;
      run += c;
    }
    const uint32_t *p = w.pos[cur].data();
    uint64_t *k2 = w.key[cur ^ 1].data();
    uint32_t *p2 = w.pos[cur ^ 1].data();
    for (size_t i = 0; i < n; i++) {
      const uint32_t o = at[k[i] >> shift & mask]++;
      k2[o] = k[i];
      p2[o] = p[i];
    }
    cur ^= 1;
  }
  return cur;
}

// The update rule of cpuGraph.cpp:521-607 reduced to its net effect: records
// symmetrised, stably sorted by (src,dst) (original records before reversed
// copies on ties), each directed key ends in the state of its LAST record, and
// each vertex's label becomes the label of the last insert record with that
// vertex as src.
//
// Long batches are sorted by counting passes over the ids' bits (65,536 directed
// records, 19-bit ids: four passes, 0.6 ms; std::sort of records took 4.0 ms and
// bounded batches of that size), short ones by std::sort (its cost meets that of
// the passes' counters at about 500 records).
void host_delta(dsm_engine *e, const dsm_change *ch, uint32_t k, HostDelta &d) {
  constexpr size_t kCountingSort = 512;
  const size_t m = 2 * (size_t)k;
  DeltaSort &w = e->delta_sort;
  for (int i = 0; i < 2; i++)
    if (w.key[i].size() < m) {
      w.key[i].resize(m);
      w.pos[i].resize(m);
    }
  for (uint32_t i = 0; i < k; i++) {
    w.key[0][i] = (uint64_t)ch[i].src << 32 | ch[i].dst;
    w.key[0][k + i] = (uint64_t)ch[i].dst << 32 | ch[i].src;
    w.pos[0][i] = i;
    w.pos[0][k + i] = k + i;
  }
  uint32_t at = 0;
  if (m >= kCountingSort) {
    at = sort_pairs(w, m, e->n > 1 ? 32 - (uint32_t)__builtin_clz(e->n - 1) : 1u);
  } else {
    std::sort(w.pos[0].begin(), w.pos[0].begin() + m, [&](uint32_t a, uint32_t b) {
      return w.key[0][a] != w.key[0][b] ? w.key[0][a] < w.key[0][b] : a < b;
    });
    for (size_t i = 0; i < m; i++) w.key[1][i] = w.key[0][w.pos[0][i]];
    std::copy(w.pos[0].begin(), w.pos[0].begin() + m, w.pos[1].begin());
    at = 1;
  }
  const uint64_t *key = w.key[at].data();
  const uint32_t *pos = w.pos[at].data();
  auto rec = [&](size_t i) -> const dsm_change & { return ch[pos[i] < k ? pos[i] : pos[i] - k]; };
  d = HostDelta();
  for (auto *v : {&d.tv, &d.ioff, &d.doff, &d.ins, &d.del, &d.rl_v, &d.rl_l}) v->reserve(m + 1);
  d.ioff.push_back(0);
  d.doff.push_back(0);
  for (size_t i = 0; i < m;) {
    const uint32_t s = (uint32_t)(key[i] >> 32);
    const dsm_change *last_add = nullptr;
    while (i < m && (uint32_t)(key[i] >> 32) == s) {
      const uint64_t same = key[i];
      const dsm_change *last = nullptr;
      for (; i < m && key[i] == same; i++) {
        last = &rec(i);
        if (last->add) last_add = last;
      }
      (last->add ? d.ins : d.del).push_back((uint32_t)same);
    }
    d.tv.push_back(s);
    d.ioff.push_back((uint32_t)d.ins.size());
    d.doff.push_back((uint32_t)d.del.size());
    if (e->opt.relabel && last_add) {
      d.rl_v.push_back(s);
      d.rl_l.push_back(clamp_label(last_add->label, e->label_used));
    }
  }
}

int grow_pool(dsm_engine *e, unsigned long long extra);

// The arrays of an update's round on the device: what the host sends (b's const
// members, the relabels, and for a catch-up the last update's touched and
// relabelled vertices), then what only kernels write.
struct RoundArrays {
  BatchDev b;
  const uint32_t *last_touched, *last_relabel;
  SmallCopy up;
};

// A bound on the pieces of T touched lists and their inserts.
size_t max_segs(const dsm_engine *e, size_t T, size_t inserts) {
  return T + (size_t)((e->pool_cap + inserts) / kApplySeg);
}

// Sends a round's arrays in one copy, or leaves it to the kernel that begins the round
// (out.up); the caller records ev_hbuf after that.
int upload_round(dsm_engine *e, const Slice &sl, const HostDelta *relabels, bool last, RoundArrays &out) {
  static const std::vector<uint32_t> none;
  const uint32_t T = (uint32_t)sl.tv.size();
  const std::vector<uint32_t> &rl_v = relabels ? relabels->rl_v : none, &rl_l = relabels ? relabels->rl_l : none;
  const std::vector<uint32_t> &lt = last ? e->last_touched : none, &lr = last ? e->last_relabel : none;
  const std::vector<uint32_t> *parts[] = {&sl.tv, &sl.ioff, &sl.doff, &sl.ins, &sl.del, &rl_v, &rl_l, &lt, &lr};
  size_t off[10] = {};
  for (int i = 0; i < 9; i++) off[i + 1] = off[i] + parts[i]->size();
  const size_t total = off[9], R = rl_v.size();
  // the changes' positions
  const size_t o_ri = total, o_rd = o_ri + sl.ins.size(), dtotal = o_rd + sl.del.size();
  // an earlier round may still read the arrays, its copy the staging buffer
  if (dtotal > e->bbuf.n) HIPCHK(hipStreamSynchronize(e->stream));
  HIPCHK(hipEventSynchronize(e->ev_hbuf));
  HIPCHK(e->hbuf.ensure(total));
  HIPCHK(e->bbuf.ensure(dtotal));
  for (int i = 0; i < 9; i++) std::copy(parts[i]->begin(), parts[i]->end(), e->hbuf.p + off[i]);
  out.up = {};
  if (total <= kSmallCopy) out.up = {e->hbuf.p, e->bbuf.p, (uint32_t)total};
  else HIPCHK(hipMemcpyAsync(e->bbuf.p, e->hbuf.p, total * 4, hipMemcpyHostToDevice, e->stream));
  // first the touched lists' pieces, then the relabelled vertices'
  const size_t segs = max_segs(e, std::max<size_t>(T, R), sl.ins.size());
  if (T > e->soff.n || segs > e->segs.n) HIPCHK(hipStreamSynchronize(e->stream));
  HIPCHK(e->soff.ensure(T));
  HIPCHK(e->tinfo.ensure(4 * e->soff.n));
  HIPCHK(e->segs.ensure(segs));
  BatchDev b{};
  b.ntouched = T;
  b.tv = e->bbuf.p + off[0];
  b.ioff = e->bbuf.p + off[1];
  b.doff = e->bbuf.p + off[2];
  b.ins = e->bbuf.p + off[3];
  b.del = e->bbuf.p + off[4];
  b.nrelabel = (uint32_t)R;
  b.rl_v = e->bbuf.p + off[5];
  b.rl_l = e->bbuf.p + off[6];
  b.ndeg = e->tinfo.p;
  b.nnew = e->tinfo.p + e->soff.n;
  b.dst = e->tinfo.p + 2 * e->soff.n;
  b.state = e->tinfo.p + 3 * e->soff.n;
  b.soff = e->soff.p;
  b.ri = e->bbuf.p + o_ri;
  b.rd = e->bbuf.p + o_rd;
  b.segs = e->segs.p;
  out.b = b;
  out.last_touched = e->bbuf.p + off[7];
  out.last_relabel = e->bbuf.p + off[8];
  return DSM_OK;
}

// Room in the scratch for every touched list once plus the inserts: at most the
// pool's entries plus the round's inserts.
int ensure_scratch(dsm_engine *e, size_t inserts) {
  const unsigned long long need = e->pool_cap + inserts + (1ull << 20);
  if (need <= e->scratch_cap) return DSM_OK;
  HIPCHK(hipStreamSynchronize(e->stream));  // an earlier round may still use it
  HIPCHK(e->scratch.alloc(need + need / 4));
  e->scratch_cap = need + need / 4;
  return DSM_OK;
}

int status_error(dsm_engine *e) {
  if (e->h_actl.p->merge_overflow)
    return e->fail_msg(DSM_ELIMIT, "update: %u merged lists found no room in the merge scratch",
                       e->h_actl.p->merge_overflow);
  if (e->h_actl.p->chunks_dropped)
    return e->fail_msg(DSM_ELIMIT, "refinement: %u chunks of long lists found no room in their queue",
                       e->h_actl.p->chunks_dropped);
  return DSM_OK;
}

// Waits for the update's status.
int take_status(dsm_engine *e) {
  HIPCHK(to_host(e->h_actl.p, e->actl.p, 1, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return status_error(e);
}

// Grows the pool for the commits that found no room and tries them again (the
// status has been taken; their merged lists are in the scratch).
int retry_commits(dsm_engine *e, const BatchDev &b) {
  for (int attempt = 0; e->h_actl.p->overflow && attempt < 4; attempt++) {
    if (int rc = grow_pool(e, e->pool_cap / 2 + (1ull << 22))) return rc;
    HIPCHK(launch_commit_again(e->dev_graph(), b, e->scratch.p, e->pool_cap, e->actl.p, e->dirty(),
                               e->h_actl.p->nsegs, e->stream));
    if (int rc = take_status(e)) return rc;
  }
  if (e->h_actl.p->overflow) return e->fail_msg(DSM_ENOMEM, "neighbour pool could not be grown");
  return DSM_OK;
}

// Re-lays the pool with fresh slack (capacity deg*1.25+8 per vertex) into a
// new allocation of the live size plus `extra` entries.
int grow_pool(dsm_engine *e, unsigned long long extra) {
  const uint32_t n = e->n;
  std::vector<uint32_t> dg(n), st_new(n), cp_new(n);
  HIPCHK(hipMemcpy(dg.data(), e->deg.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  unsigned long long total = 0;
  for (uint32_t v = 0; v < n; v++) {
    cp_new[v] = dg[v] + dg[v] / 4 + 8;
    st_new[v] = (uint32_t)total;
    total += cp_new[v];
  }
  const unsigned long long ncap = total + extra;
  if (ncap >= (1ull << 32)) return e->fail_msg(DSM_ELIMIT, "neighbour pool exceeds 32-bit offsets");
  DevBuf<uint32_t> np, nst;
  HIPCHK(np.alloc(ncap));
  HIPCHK(nst.alloc(n));
  // on the engine's stream, ahead of the kernels that read the new starts
  HIPCHK(hipMemcpyAsync(nst.p, st_new.data(), (size_t)n * 4, hipMemcpyHostToDevice, e->stream));
  HIPCHK(launch_pool_move(e->pool.p, np.p, e->start.p, nst.p, e->deg.p, n, e->stream));
  HIPCHK(hipMemcpyAsync(e->cap.p, cp_new.data(), (size_t)n * 4, hipMemcpyHostToDevice, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  std::swap(e->pool.p, np.p);
  std::swap(e->pool.n, np.n);
  std::swap(e->start.p, nst.p);
  std::swap(e->start.n, nst.n);
  e->pool_cap = ncap;
  if (int rc = size_sorted_build(e)) return rc;
  // every label-sorted copy moves with the pool: the update that grew it
  // rebuilds them all once its commits are done (the rebuild uses the merge
  // scratch, which still holds the lists of the commits that failed)
  HIPCHK(e->lpool.alloc(ncap));
  e->lpool_stale = true;
  e->grew = true;
  // scratch must hold one copy of every list; the failed commits' lists move
  // with it
  if (e->scratch_cap < ncap + (1ull << 20)) {
    DevBuf<uint32_t> ns;
    HIPCHK(ns.alloc(ncap + (1ull << 20)));
    HIPCHK(hipMemcpyAsync(ns.p, e->scratch.p, e->scratch_cap * 4, hipMemcpyDeviceToDevice, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    std::swap(e->scratch.p, ns.p);
    std::swap(e->scratch.n, ns.n);
    e->scratch_cap = ncap + (1ull << 20);
  }
  ApplyCtl a = *e->h_actl.p;
  a.pool_used = total;
  a.overflow = 0;
  // ordered before the retried commits on the engine's stream; `a` must stay
  // alive until the copy is done
  HIPCHK(hipMemcpyAsync(e->actl.p, &a, sizeof a, hipMemcpyHostToDevice, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  *e->h_actl.p = a;
  return DSM_OK;
}

// Records on the device, src[k] | dst[k]; few of them are left to the next round's
// first kernel (up), where it is given.
int upload_records(dsm_engine *e, const std::vector<uint32_t> &s, const std::vector<uint32_t> &d,
                   DevBuf<uint32_t> &dev, SmallCopy *up = nullptr) {
  const size_t k = s.size();
  if (2 * k > dev.n) HIPCHK(hipStreamSynchronize(e->stream));
  HIPCHK(dev.ensure(2 * k));
  HIPCHK(hipEventSynchronize(e->ev_hrec));
  HIPCHK(e->hrec.ensure(2 * k));
  std::copy(s.begin(), s.end(), e->hrec.p);
  std::copy(d.begin(), d.end(), e->hrec.p + k);
  if (up && 2 * k <= kSmallCopy) {
    *up = {e->hrec.p, dev.p, (uint32_t)(2 * k)};
    return DSM_OK;
  }
  HIPCHK(hipMemcpyAsync(dev.p, e->hrec.p, 2 * k * 4, hipMemcpyHostToDevice, e->stream));
  HIPCHK(hipEventRecord(e->ev_hrec, e->stream));
  return DSM_OK;
}


// The cluster-encoding refinement of every query on the current graph,
// enqueued on the engine's stream after the LDF/NLF rows are current: the
// position rows are cleared, each core's alive row loaded, then pass step s of
// every query runs as one k_cluster_pass launch plus one k_cluster_heavy
// launch for the chunks of candidates with long lists (filter.cu:936-1177 runs
// one kernel and one device synchronisation per cluster of one query). No list is
// longer than `longest`, and all together hold at most `entries`.
int cluster_refine(dsm_engine *e, uint32_t longest, unsigned long long entries) {
  if (!e->cluster) return DSM_OK;
  const uint32_t nsteps = (uint32_t)e->cstep_off.size() - 1;
  // heavy chunks of one pass: at most 2 x (list entries) / kClusterChunk
  const size_t need = (size_t)e->cmax_step_ops * (2 * entries / kClusterChunk + 64);
  if (need > e->cheavy.n) HIPCHK(e->cheavy.alloc(need));
  HIPCHK(hipEventRecord(e->ev_ref[0], e->stream));
  HIPCHK(launch_cluster_init(e->bm.p, e->words, e->nsig_rows, e->npos_rows, e->calive.p, e->d_alive_src.p,
                             e->nalive_src, e->cctl.p, nsteps, e->actl.p, e->stream));
  ClusterArgs a{};
  a.g = e->dev_graph();
  a.bm = e->bm.p;
  a.words = e->words;
  a.alive = e->calive.p;
  a.crow = e->d_crow.p;
  a.actl = e->actl.p;
  a.heavy = e->cheavy.p;
  a.heavy_cap = (uint32_t)std::min<size_t>(e->cheavy.n, 0xFFFFFFF0u);
  for (uint32_t st = 0; st < nsteps; st++) {
    a.ops = e->d_cops.p + e->cstep_off[st];
    a.nops = e->cstep_off[st + 1] - e->cstep_off[st];
    a.ctl = e->cctl.p + st;
    HIPCHK(launch_cluster_pass(a, (uint32_t)e->num_cu * 8, e->stream));
    if (longest > kClusterChunk) HIPCHK(launch_cluster_heavy(a, (uint32_t)e->num_cu * 4, e->stream));
  }
  HIPCHK(hipEventRecord(e->ev_ref[1], e->stream));
  e->refine_timed = true;
  return DSM_OK;
}

// Adds the device time of the last refinement to the batch statistics (the
// refinement's stream must have been synchronised).
void take_refine_time(dsm_engine *e) {
  if (!e->refine_timed) return;
  e->refine_timed = false;
  float ms = 0;
  if (hipEventElapsedTime(&ms, e->ev_ref[0], e->ev_ref[1]) == hipSuccess) e->stats.ms_refine += ms;
}

DevGraph graph_of(const dsm_engine *e, const dsm_engine::GraphCopy &c) {
  DevGraph g;
  g.n = e->n;
  g.pool = c.pool.p;
  g.start = c.start.p;
  g.deg = c.deg.p;
  g.cap = c.cap.p;
  g.lab = c.lab.p;
  g.lpool = c.lpool.p;
  g.loff = c.loff.p;
  g.nbuckets = e->nbuckets;
  return g;
}

// An update that one block does in less time than the launches of many take
// (k_update_small): few lists, none with pieces, and few vertices that can become dirty
// (the relabelled ones' neighbours), in a graph whose marks one block looks through
// in a few steps. One record on lists of 30: 81 us a call instead of 105. With 500
// vertices that may be dirty (8 records, 400 vertices) it takes 30 us, but behind the
// negatives' round instead of beside it: 1,180 us for four such calls instead of 1,120.
bool small_update(const dsm_engine *e, const HostDelta &d) {
  const size_t T = d.tv.size(), R = d.rl_v.size(), changes = d.ins.size() + d.del.size();
  const size_t longest = (size_t)e->h_actl.p->max_deg + d.ins.size();
  return T && T <= 32 && R <= 64 && changes <= kSmallChanges && longest <= kBuildSeg && T + R * longest <= 256 &&
         e->n <= 65536 && !e->lpool_stale;
}

// One batch's update and candidate refresh from its host delta, on the engine's
// stream: merge and commit the lists, relabel, rebuild the dirty vertices'
// label-sorted copies, then refilter the dirty vertices (long lists take their
// neighbour-label counts from those copies). Everything is enqueued at once;
// kernels after the commit do nothing when a commit found no room, and are
// launched again once the pool has grown. The update is done when this returns,
// and *h_actl is its status; `done` (may be null) is recorded at its end.
//
// With `from`, the engine's graph lags behind that copy by exactly the last
// update (shadow_delta_ok) and catches up first, by what that update touched and
// relabelled and the signature rows. The label-sorted copies of its dirty
// vertices (the shared dirty list holds them until the next compaction) follow
// once the new update has marked its own, whose copies are rebuilt anyway.
int apply_delta_and_refresh(dsm_engine *e, const HostDelta &d, const dsm_engine::GraphCopy *from = nullptr,
                            hipEvent_t done = nullptr) {
  const bool small = !from && small_update(e, d);
  const uint32_t T = (uint32_t)d.tv.size();
  e->shadow_delta_ok = false;
  e->grew = false;
  uint32_t rounds = 1, most_ins = 0;
  for (uint32_t t = 0; t < T; t++) {
    const uint32_t ni = d.ioff[t + 1] - d.ioff[t], m = std::max(ni, d.doff[t + 1] - d.doff[t]);
    rounds = std::max(rounds, (m + kMaxVertexChanges - 1) / kMaxVertexChanges);
    most_ins = std::max(most_ins, ni);
  }
  // no list is longer before the update, or after it
  const uint32_t before = e->h_actl.p->max_deg;
  const uint32_t longest = (uint32_t)std::min<uint64_t>((uint64_t)before + most_ins, 0xFFFFFFFFull);
  // nor do the lists hold more than the pool's used part before, and the inserts
  const unsigned long long entries = e->h_actl.p->pool_used + d.ins.size();
  Slice part;
  RoundArrays ra{};
  for (uint32_t rd = 0; rd < rounds; rd++) {
    if (rounds > 1) {
      part = Slice{{}, {0}, {0}, {}, {}};
      for (uint32_t t = 0; t < T; t++) {
        const uint32_t i0 = d.ioff[t] + rd * kMaxVertexChanges, i1 = std::min(d.ioff[t + 1], i0 + kMaxVertexChanges);
        const uint32_t d0 = d.doff[t] + rd * kMaxVertexChanges, d1 = std::min(d.doff[t + 1], d0 + kMaxVertexChanges);
        if (i0 >= i1 && d0 >= d1 && rd > 0) continue;
        part.tv.push_back(d.tv[t]);
        if (i0 < i1) part.ins.insert(part.ins.end(), d.ins.begin() + i0, d.ins.begin() + i1);
        if (d0 < d1) part.del.insert(part.del.end(), d.del.begin() + d0, d.del.begin() + d1);
        part.ioff.push_back((uint32_t)part.ins.size());
        part.doff.push_back((uint32_t)part.del.size());
      }
    }
    const Slice &sl = rounds > 1 ? part : static_cast<const Slice &>(d);
    const bool final_round = rd + 1 == rounds;
    if (int rc = upload_round(e, sl, final_round ? &d : nullptr, from && rd == 0, ra)) return rc;
    if (small) {
      if (int rc = ensure_scratch(e, sl.ins.size())) return rc;
      HIPCHK(launch_update_small(e->dev_graph(), ra.b, e->tables(), e->dirty(), e->sorted_build(), e->scratch.p,
                                 e->scratch_cap, e->pool_cap, longest, ra.up, e->h_actl.p, e->stream));
      HIPCHK(hipEventRecord(e->ev_hbuf, e->stream));
      break;
    }
    if (rd == 0) {
      HIPCHK(launch_update_begin(e->actl.p, from ? from->actl.p : nullptr, e->build_ctl.p, ra.up, e->stream));
      HIPCHK(hipEventRecord(e->ev_hbuf, e->stream));
      if (from) {
        CatchUp c;
        c.x = graph_of(e, *from);
        c.y = e->dev_graph();
        c.touched = ra.last_touched;
        c.ntouched = (uint32_t)e->last_touched.size();
        c.relabeled = ra.last_relabel;
        c.nrelabeled = (uint32_t)e->last_relabel.size();
        c.bm_x = from->bm.p;
        c.bm_y = e->bm.p;
        c.nbm = (size_t)e->nsig_rows * e->words;
        c.q = e->sync_q.p;
        c.qcap = (uint32_t)e->sync_q.n;
        c.actl = e->actl.p;
        HIPCHK(launch_catch_up(c, before, e->stream));
      }
    } else {
      HIPCHK(launch_round_begin(e->actl.p, ra.up, e->stream));
      HIPCHK(hipEventRecord(e->ev_hbuf, e->stream));
    }
    if (int rc = ensure_scratch(e, sl.ins.size())) return rc;
    // pieces: one a list, and what no list can go past
    const size_t segs = std::min<size_t>(max_segs(e, sl.tv.size(), sl.ins.size()),
                                         sl.tv.size() * (1 + (size_t)(longest / kApplySeg)));
    HIPCHK(launch_apply(e->dev_graph(), ra.b, e->scratch.p, e->scratch_cap, e->pool_cap, e->actl.p, e->dirty(), segs,
                        e->stream));
    if (!final_round) {
      if (int rc = take_status(e)) return rc;
      if (int rc = retry_commits(e, ra.b)) return rc;
    }
  }
  e->stats.touched_vertices = T;
  for (bool done_small = small;; done_small = false) {
    if (done_small) {
      if (int rc = cluster_refine(e, longest, entries)) return rc;
      if (done) HIPCHK(hipEventRecord(done, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
      if (int rc = status_error(e)) return rc;
      if (!e->h_actl.p->overflow) break;
      if (int rc = retry_commits(e, ra.b)) return rc;
      continue;
    }
    const size_t R = ra.b.nrelabel;
    HIPCHK(launch_relabel(e->dev_graph(), ra.b, e->tables(), e->dirty(),
                          std::min(max_segs(e, R, 0), R * (1 + (size_t)(longest / kApplySeg))), e->stream));
    // after a pool growth the slots moved and every copy is rebuilt instead
    if (from && !e->grew && !e->lpool_stale)
      HIPCHK(launch_sync_sorted(graph_of(e, *from), e->dev_graph(), e->dirty_list.p, &from->actl.p->ndirty,
                                e->dirty_marks.p, e->sync_q.p, (uint32_t)e->sync_q.n, e->actl.p, before, e->stream));
    HIPCHK(launch_dirty_compact(e->dev_graph(), e->dirty(), e->stream));
    // the dirty list (touched vertices, relabelled ones and their neighbours) is
    // exactly the set whose label-sorted copies changed, unless the pool grew
    const uint32_t *list = e->lpool_stale ? nullptr : e->dirty_list.p;
    HIPCHK(launch_lbuild(e->dev_graph(), e->tables(), list, list ? &e->actl.p->ndirty : nullptr, e->sorted_build(),
                         longest, true, e->stream));
    HIPCHK(launch_filter_dirty(e->dev_graph(), e->tables(), e->dirty(), e->stream));
    if (int rc = cluster_refine(e, longest, entries)) return rc;
    if (done) HIPCHK(hipEventRecord(done, e->stream));
    if (int rc = take_status(e)) return rc;
    if (!e->h_actl.p->overflow) break;
    // the kernels above waited for this
    if (int rc = retry_commits(e, ra.b)) return rc;
  }
  e->lpool_stale = false;
  e->stats.relocated_vertices = e->h_actl.p->relocated;
  return DSM_OK;
}

// Blocks per CU of a DFS shape: the occupancy limit and, with overlap_apply,
// at most what leaves 32 KB of the CU's LDS to the update kernels that run
// beside a pipelined round (k_apply_rank takes 16 KB per block). A shape
// that fills the LDS makes them wait for the round.
uint32_t dfs_bpc(const dsm_engine *e, uint32_t wpb) {
  uint32_t b = (uint32_t)std::max(1, dfs_max_blocks_per_cu(wpb, e->max_qn));
  if (e->overlap_apply) {
    const uint32_t per_block = wpb * dfs_lds_bytes_per_wave(e->max_qn);
    const int room = e->cu_lds - 32 * 1024;
    const uint32_t cap = room > (int)per_block ? (uint32_t)room / per_block : 1u;
    b = std::min(b, cap);
  }
  return b;
}

int create_impl(dsm_engine *e, const dsm_graph_desc *graph, const dsm_query_desc *queries,
                uint32_t num_queries) {
  int rc = 0;
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
  for (hipEvent_t *x : {&e->ev_pre, &e->ev_hbuf, &e->ev_hrec})
    HIPCHK(hipEventCreateWithFlags(x, hipEventDisableTiming));
  HIPCHK(hipDeviceGetAttribute(&e->num_cu, hipDeviceAttributeMultiprocessorCount, e->opt.device));
  HIPCHK(hipDeviceGetAttribute(&e->wall_khz, hipDeviceAttributeWallClockRate, e->opt.device));
  {
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, e->opt.device) ==
            hipSuccess &&
        lds > 0)
      e->cu_lds = lds;
  }
  e->overlap_apply = e->opt.overlap_apply != 0;
  HIPCHK(hipStreamCreateWithFlags(&e->stream2, hipStreamNonBlocking));
  if (e->wall_khz <= 0) e->wall_khz = 100000;
  if (e->opt.watchdog_ms) e->watchdog_ms = e->opt.watchdog_ms;
  for (auto &x : e->ev) HIPCHK(hipEventCreate(&x));
  e->cluster = e->opt.cluster_filter != 0;
  std::vector<uint64_t> label_freq(256, 0);
  for (uint32_t v = 0; graph->labels && v < graph->num_vertices; v++)
    if (graph->labels[v] < 255) label_freq[graph->labels[v]]++;
  if ((rc = build_queries(e, queries, num_queries, label_freq))) return rc;
  if ((rc = upload_graph(e, graph))) return rc;
  if ((rc = upload_tables(e))) return rc;
  uint32_t wpb = e->opt.waves_per_block;
  if (wpb != 1 && wpb != 2 && wpb != 4 && wpb != 8) wpb = 4;
  e->dfs_wpb = wpb;
  e->max_qn = 2;
  for (auto &q : e->queries) e->max_qn = std::max(e->max_qn, q.n);
  // keep a block's LDS (waves x per-wave stack) within 64 KB
  while (wpb > 1 && wpb * dfs_lds_bytes_per_wave(e->max_qn) > 65536) wpb /= 2;
  e->dfs_wpb = wpb;
  int per_cu = (int)dfs_bpc(e, wpb);
  if (e->opt.blocks_per_cu && (int)e->opt.blocks_per_cu < per_cu) per_cu = (int)e->opt.blocks_per_cu;
  e->dfs_blocks = (uint32_t)(per_cu * e->num_cu);
  e->grid_given = e->opt.blocks_per_cu != 0;
  // room for the largest grid any launch shape can have (the autotuner may
  // pick another shape later)
  {
    uint32_t most = 0;
    for (uint32_t w : {1u, 2u, 4u, 8u}) most = std::max<uint32_t>(most, (uint32_t)dfs_max_blocks_per_cu(w, e->max_qn) * w);
    e->wave_slots = most * (uint32_t)e->num_cu;
    HIPCHK(e->mail.alloc(e->wave_slots));
    HIPCHK(hipMemset(e->mail.p, 0, (size_t)e->wave_slots * sizeof(Mailbox)));  // stop = 0: no epoch
    HIPCHK(e->idle.alloc(idle_words(e->wave_slots) + 1));  // the reserve's begin with a word of their own
    HIPCHK(e->h_rec.ensure(e->wave_slots));
  }
  e->donate_min = e->opt.donate_min ? e->opt.donate_min : 256;
  e->lane_work = e->opt.lane_work ? e->opt.lane_work : 16;
  e->leaf_budget = e->opt.leaf_budget ? e->opt.leaf_budget : 8192;
  e->donate_every = e->opt.donate_every ? e->opt.donate_every : 4;
  e->donate_min_n2 = e->opt.donate_min_n2 ? e->opt.donate_min_n2 : 64;
  e->leaf_sets = e->opt.leaf_sets != 0;
  e->bit_probe_last = e->opt.bit_probe_last != 0;
  e->seeding_timed = e->opt.graph_rounds == 0;
  e->leaf_segments = e->opt.leaf_segments != 0;
  e->poll_max = e->opt.poll_max ? std::min<uint32_t>(e->opt.poll_max, 16u) : 16u;
  HIPCHK(launch_filter_full(e->dev_graph(), e->tables(), e->stream));
  HIPCHK(launch_build_reset(e->sorted_build(), e->stream));
  HIPCHK(launch_lbuild(e->dev_graph(), e->tables(), nullptr, nullptr, e->sorted_build(), e->h_actl.p->max_deg, false,
                       e->stream));
  if ((rc = cluster_refine(e, e->h_actl.p->max_deg, e->h_actl.p->pool_used))) return rc;
  if ((rc = take_status(e))) return rc;
  e->refine_timed = false;
  return DSM_OK;
}

template <typename T>
void swap_buf(DevBuf<T> &a, DevBuf<T> &b) {
  std::swap(a.p, b.p);
  std::swap(a.n, b.n);
}

// Exchanges the engine's graph with the second copy.
void swap_graph(dsm_engine *e) {
  auto &c = e->shadow;
  swap_buf(e->pool, c.pool);
  swap_buf(e->start, c.start);
  swap_buf(e->deg, c.deg);
  swap_buf(e->cap, c.cap);
  swap_buf(e->lpool, c.lpool);
  swap_buf(e->loff, c.loff);
  swap_buf(e->lab, c.lab);
  swap_buf(e->bm, c.bm);
  swap_buf(e->actl, c.actl);
  std::swap(e->pool_cap, c.pool_cap);
}

// Allocates the second copy of the graph at the current sizes; its contents
// are written by the first overlapped update.
int reserve_shadow(dsm_engine *e) {
  auto &c = e->shadow;
  auto like = [](auto &dst, const auto &src) -> hipError_t {
    return dst.n < src.n ? dst.alloc(src.n) : hipSuccess;
  };
  HIPCHK(like(c.pool, e->pool));
  HIPCHK(like(c.lpool, e->lpool));
  HIPCHK(like(c.start, e->start));
  HIPCHK(like(c.deg, e->deg));
  HIPCHK(like(c.cap, e->cap));
  HIPCHK(like(c.loff, e->loff));
  HIPCHK(like(c.lab, e->lab));
  HIPCHK(like(c.bm, e->bm));
  HIPCHK(like(c.actl, e->actl));
  return DSM_OK;
}

// Makes the engine's graph a copy of `c` on the engine's stream. The pool
// and the label-sorted copies are copied up to the pool's used end (the
// host's ApplyCtl mirror holds it after every update).
int copy_graph(dsm_engine *e, const dsm_engine::GraphCopy &c) {
  unsigned long long used = e->h_actl.p->pool_used;
  if (used == 0 || used > c.pool_cap) used = c.pool_cap;
  ArrayCopies a{};
  auto add = [&](auto &dst, const auto &src, size_t count) -> hipError_t {
    a.from[a.n] = src.p;
    a.bytes[a.n] = count * sizeof(*src.p);
    const hipError_t err = dst.n < src.n ? dst.alloc(src.n) : hipSuccess;
    a.to[a.n++] = dst.p;
    return err;
  };
  HIPCHK(add(e->pool, c.pool, used));
  HIPCHK(add(e->lpool, c.lpool, used));
  HIPCHK(add(e->start, c.start, c.start.n));
  HIPCHK(add(e->deg, c.deg, c.deg.n));
  HIPCHK(add(e->cap, c.cap, c.cap.n));
  HIPCHK(add(e->loff, c.loff, c.loff.n));
  HIPCHK(add(e->lab, c.lab, c.lab.n));
  // the signature rows; the cluster position rows are recomputed by the update
  HIPCHK(add(e->bm, c.bm, (size_t)e->nsig_rows * e->words));
  HIPCHK(add(e->actl, c.actl, 1));
  HIPCHK(launch_array_copies(a, e->stream));
  e->pool_cap = c.pool_cap;
  return DSM_OK;
}

// The second copy lags by exactly the last update, in slots of the same places.
bool catch_up_by_delta(const dsm_engine *e, const dsm_engine::GraphCopy &c) {
  return kDeltaSync && e->shadow_delta_ok && e->pool_cap == c.pool_cap && e->n < (1u << 31);
}

// Applies one batch to the second copy of the graph while a round that was
// enqueued on `stream` matches on the first: the copies swap, the new current
// one becomes a copy of the old one (after ev_pre, i.e. after every update
// enqueued before the round) and takes the batch, all on stream2. Returns
// once the update is done; the copies stay swapped, or with keep = false
// swap back (the update is dropped: the tuner's load).
int overlap_apply(dsm_engine *e, const HostDelta &d, bool stats, bool keep = true) {
  const ApplyCtl mirror = *e->h_actl.p;
  std::swap(e->stream, e->stream2);
  swap_graph(e);
  int rc = DSM_OK;
  auto run = [&]() -> int {
    HIPCHK(hipStreamWaitEvent(e->stream, e->ev_pre, 0));
    if (stats) HIPCHK(hipEventRecord(e->ev[0], e->stream));
    const bool by_delta = catch_up_by_delta(e, e->shadow);
    // long lists queued: at most one per touched and one per dirty vertex
    if (by_delta) HIPCHK(e->sync_q.ensure(2 * (size_t)e->n));
    else if (int r = copy_graph(e, e->shadow)) return r;
    if (int r = apply_delta_and_refresh(e, d, by_delta ? &e->shadow : nullptr, stats ? e->ev[2] : nullptr)) return r;
    if (stats) {
      e->stats.filter_entries += e->h_actl.p->filter_entries;
      e->stats.dirty_groups += e->h_actl.p->ndirty;
      e->stats.filter_bits += e->h_actl.p->filter_bits;
    }
    if (stats) {
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, e->ev[0], e->ev[2]));
      e->stats.ms_apply += ms;
      take_refine_time(e);
    }
    e->refine_timed = false;
    return DSM_OK;
  };
  rc = run();
  std::swap(e->stream, e->stream2);
  if (!keep) {
    swap_graph(e);
    *e->h_actl.p = mirror;
  } else if (rc == DSM_OK && !e->grew) {
    // the other copy now lags by exactly this update
    e->shadow_delta_ok = true;
    e->last_touched = d.tv;
    e->last_relabel = d.rl_v;
  }
  return rc;
}

// Applies one batch to the current graph, and its statistics.
int apply_in_place(dsm_engine *e, const HostDelta &d) {
  HIPCHK(hipEventRecord(e->ev[0], e->stream));
  if (int rc = apply_delta_and_refresh(e, d, nullptr, e->ev[2])) return rc;
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, e->ev[0], e->ev[2]));
  e->stats.ms_apply = ms;
  take_refine_time(e);
  e->stats.filter_entries = e->h_actl.p->filter_entries;
  e->stats.dirty_groups = e->h_actl.p->ndirty;
  e->stats.filter_bits = e->h_actl.p->filter_bits;
  return DSM_OK;
}

}  // namespace

// =============================================================== C ABI

extern "C" {

void dsm_options_default(dsm_options *opt) {
  std::memset(opt, 0, sizeof *opt);
  opt->device = 0;
  opt->relabel = 1;
  opt->count_negatives = 1;
  opt->waves_per_block = 4;
  opt->leaf_sets = 1;
  opt->graph_rounds = 1;
  opt->leaf_segments = 1;
  opt->overlap_apply = 1;
}

const char *dsm_last_error(const dsm_engine *e) {
  if (!e) return g_create_error.c_str();
  return e->err.c_str();
}

int dsm_create(const dsm_graph_desc *graph, const dsm_query_desc *queries, uint32_t num_queries,
               const dsm_options *opt, dsm_engine **out) {
  if (!out || !graph || !queries) {
    g_create_error = "null argument";
    return DSM_EINVAL;
  }
  *out = nullptr;
  std::unique_ptr<dsm_engine> e(new dsm_engine());
  if (opt) e->opt = *opt;
  else dsm_options_default(&e->opt);
  auto fail = [&](int rc) {
    g_create_error = e->err;
    return rc;
  };
  if (graph->num_vertices == 0) {
    e->err = "empty data graph";
    return fail(DSM_EINVAL);
  }
  e->n = graph->num_vertices;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    e->err = "no HIP device available";
    return fail(DSM_EDEVICE);
  }
  if (e->opt.device < 0 || e->opt.device >= ndev) {
    e->err = "device ordinal out of range";
    return fail(DSM_EINVAL);
  }
  int rc = create_impl(e.get(), graph, queries, num_queries);
  if (rc) return fail(rc);
  *out = e.release();
  return DSM_OK;
}

void dsm_destroy(dsm_engine *e) {
  if (!e) return;
  (void)hipSetDevice(e->opt.device);
  (void)hipStreamSynchronize(e->stream);
  delete e;
}

int dsm_apply_batch(dsm_engine *e, const dsm_change *changes, uint32_t k) {
  if (!e || (!changes && k)) return DSM_EINVAL;
  for (uint32_t i = 0; i < k; i++)
    if (changes[i].src >= e->n || changes[i].dst >= e->n)
      return e->fail_msg(DSM_EINVAL, "change %u: endpoint out of range (%u,%u) for %u vertices", i,
                         changes[i].src, changes[i].dst, e->n);
  HIPCHK(hipSetDevice(e->opt.device));
  e->stats = dsm_stats{};
  e->pos_s.clear();
  e->pos_d.clear();
  e->neg_s.clear();
  e->neg_d.clear();
  for (uint32_t i = 0; i < k; i++) {
    if (changes[i].add) {
      e->pos_s.push_back(changes[i].src);
      e->pos_d.push_back(changes[i].dst);
    } else {
      e->neg_s.push_back(changes[i].src);
      e->neg_d.push_back(changes[i].dst);
    }
  }
  e->counts_stale = true;
  e->results_here = false;
  int rc;
  bool applied = false;
  // 1. negatives in the pre-batch graph; with overlap_apply the batch is
  // applied to the second copy of the graph meanwhile
  if (e->opt.count_negatives && !e->neg_s.empty()) {
    const uint32_t nn = (uint32_t)e->neg_s.size();
    if ((rc = ensure_seed_cap(e, nn))) return rc;
    DevBuf<uint32_t> &rb = e->rec_neg;
    SmallCopy up{};
    if ((rc = upload_records(e, e->neg_s, e->neg_d, rb, &up))) return rc;
    if (e->overlap_apply) HIPCHK(hipEventRecord(e->ev_pre, e->stream));
    if ((rc = run_round(e, rb.p, rb.p + nn, nn, 0, nullptr, e->ev[7], e->ev[8], up))) return rc;
    // with no positives to come these are the batch's counts
    if (e->pos_s.empty()) HIPCHK(to_host(e->h_results.p, e->results.p, 2 * e->queries.size() + 1, e->stream));
    if (e->overlap_apply) {
      HostDelta d;
      host_delta(e, changes, k, d);
      // a small update is over before the second copy would be made, and follows
      // the round on its stream
      if (!small_update(e, d)) rc = overlap_apply(e, d, true);
      else rc = apply_in_place(e, d);
      if (rc) return rc;
      applied = true;
    }
    HIPCHK(hipStreamSynchronize(e->stream));
    e->results_here = e->pos_s.empty();
    if ((rc = check_round(e, &e->stats.seeds_neg))) return rc;
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[7], e->ev[8]));
    e->stats.ms_dfs_neg = ms;
  }
  // 2-3. apply + relabel + filter (update, relabel, refilter and
  // label-sorted copies; already done beside the negatives with overlap)
  if (!applied) {
    HostDelta d;
    host_delta(e, changes, k, d);
    if ((rc = apply_in_place(e, d))) return rc;
  }
  e->stats.ms_filter = 0;
  e->stats.relabeled_vertices = e->h_actl.p->relabeled;
  e->stats.pool_entries_used = e->h_actl.p->pool_used;
  e->stats.pool_entries_capacity = e->pool_cap;
  e->batch_pending = true;
  return DSM_OK;
}

int dsm_match_batch(dsm_engine *e, uint64_t *pos, uint64_t *neg) {
  if (!e) return DSM_EINVAL;
  HIPCHK(hipSetDevice(e->opt.device));
  int rc;
  bool fetched = false;
  const uint32_t nq = (uint32_t)e->queries.size();
  if (e->batch_pending && !e->pos_s.empty()) {
    const uint32_t np = (uint32_t)e->pos_s.size();
    if ((rc = ensure_seed_cap(e, np))) return rc;
    DevBuf<uint32_t> &rb = e->rec_pos;
    SmallCopy up{};
    if ((rc = upload_records(e, e->pos_s, e->pos_d, rb, &up))) return rc;
    hipEvent_t seeding = e->seeding_timed ? e->ev[3] : nullptr;  // else part of the DFS time
    if ((rc = run_round(e, rb.p, rb.p + np, np, 1, seeding, e->ev[4], e->ev[5], up))) return rc;
    if ((rc = fetch_results(e))) return rc;
    fetched = true;
    if ((rc = check_round(e, &e->stats.seeds_pos))) return rc;
    float ms = 0;
    if (seeding) HIPCHK(hipEventElapsedTime(&ms, seeding, e->ev[4]));
    e->stats.ms_seed = ms;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[4], e->ev[5]));
    e->stats.ms_dfs_pos = ms;
  }
  e->batch_pending = false;
  if (!fetched && !e->results_here && (rc = fetch_results(e))) return rc;
  e->stats.tuples = *e->h_results.p;
  for (uint32_t q = 0; q < nq; q++) {
    if (pos) pos[q] = e->h_counts()[2 * q + 1];
    if (neg) neg[q] = e->h_counts()[2 * q + 0];
  }
  return DSM_OK;
}

int dsm_process_batch(dsm_engine *e, const dsm_change *changes, uint32_t k, uint64_t *pos, uint64_t *neg) {
  int rc = dsm_apply_batch(e, changes, k);
  if (rc) return rc;
  return dsm_match_batch(e, pos, neg);
}

int dsm_get_tuples(dsm_engine *e, uint32_t *out, uint64_t cap, uint64_t *num_out) {
  if (!e || !num_out) return DSM_EINVAL;
  const uint64_t found = e->stats.tuples;
  *num_out = found;
  const uint64_t have = std::min<uint64_t>(found, e->tuple_cap);
  const uint64_t copy = std::min<uint64_t>(have, cap);
  if (copy && out) {
    HIPCHK(hipSetDevice(e->opt.device));
    HIPCHK(hipMemcpy(out, e->tuples, copy * (kMaxQ + 2) * 4, hipMemcpyDefault));
  }
  if (found > e->tuple_cap) return e->fail_msg(DSM_ETRUNC, "%llu tuples found, capacity %llu",
                                               (unsigned long long)found, (unsigned long long)e->tuple_cap);
  return DSM_OK;
}

int dsm_get_stats(const dsm_engine *e, dsm_stats *out) {
  if (!e || !out) return DSM_EINVAL;
  *out = e->stats;
  return DSM_OK;
}

int dsm_get_graph(dsm_engine *e, uint64_t *offsets, uint32_t *neighbours, uint64_t cap, uint32_t *labels,
                  uint64_t *num_entries) {
  if (!e || !offsets || !num_entries) return DSM_EINVAL;
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  const uint32_t n = e->n;
  // packed in the merge scratch, which is idle between updates and has room for
  // the offsets: it is as large as a pool with at least four entries a vertex
  unsigned long long *off = reinterpret_cast<unsigned long long *>(e->scratch.p);
  const size_t sums = csr_sum_words(n + 1ull), head = 2 * (n + 1ull + sums);
  HIPCHK(launch_graph_offsets(n, e->deg.p, off, off + n + 1, e->stream));
  HIPCHK(hipMemcpyAsync(offsets, off, (n + 1ull) * 8, hipMemcpyDeviceToHost, e->stream));
  std::vector<uint8_t> lb(labels ? n : 0);
  if (labels) HIPCHK(hipMemcpyAsync(lb.data(), e->lab.p, n, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  const uint64_t o = offsets[n];
  *num_entries = o;
  for (uint32_t v = 0; labels && v < n; v++) labels[v] = lb[v];
  if (o > cap || !neighbours) return o > cap ? e->fail_msg(DSM_ETRUNC, "neighbour buffer too small") : DSM_OK;
  DevBuf<uint32_t> own;  // where the lists do not fit behind the offsets
  if (head + o > e->scratch_cap) HIPCHK(own.alloc(o));
  uint32_t *lists = own.p ? own.p : e->scratch.p + head;
  HIPCHK(launch_graph_lists(n, off, e->start.p, e->pool.p, o, lists, e->stream));
  HIPCHK(hipMemcpyAsync(neighbours, lists, o * 4, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return DSM_OK;
}

int dsm_get_candidates(dsm_engine *e, uint32_t q, uint32_t u, uint64_t *words) {
  if (!e || !words || q >= e->queries.size() || u >= e->queries[q].n) return DSM_EINVAL;
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  const uint32_t s = e->qsig[q][u];
  HIPCHK(hipMemcpy(words, e->bm.p + (size_t)s * e->words, (size_t)e->words * 8, hipMemcpyDeviceToHost));
  return DSM_OK;
}

uint32_t dsm_cluster_plan(uint32_t num_vertices, uint32_t num_edges, const uint32_t *edge_src,
                          const uint32_t *edge_dst, uint32_t *out, uint32_t cap) {
  if (!edge_src || !edge_dst || num_vertices > (uint32_t)kMaxQ) return 0;
  for (uint32_t i = 0; i < num_edges; i++)
    if (edge_src[i] >= num_vertices || edge_dst[i] >= num_vertices) return 0;
  ClusterPlan P;
  if (build_cluster_plan(num_vertices, num_edges, edge_src, edge_dst, P)) return 0;
  uint32_t w = 0;
  auto put = [&](uint32_t x) {
    if (out && w < cap) out[w] = x;
    w++;
  };
  put(num_vertices);
  uint32_t ncover = 0;
  for (auto &p : P.passes) ncover += p.kind == ClusterPlan::kEncode;
  put(ncover);
  for (auto &p : P.passes)
    if (p.kind == ClusterPlan::kEncode) put(P.clusters[p.arg].members[0]);
  put((uint32_t)P.clusters.size());
  for (auto &c : P.clusters) {
    put(c.valid ? 1 : 0);
    put((uint32_t)c.members.size());
    for (uint32_t u : c.members) put(u);
  }
  put(P.final_cluster);
  for (uint32_t u : P.final_pos) put(u);
  put((uint32_t)P.passes.size());
  for (auto &p : P.passes) {
    put(p.kind);
    put(p.arg);
  }
  return w;
}

int dsm_get_refined_candidates(dsm_engine *e, uint32_t q, uint32_t u, uint64_t *words) {
  if (!e || !words || q >= e->queries.size() || u >= e->queries[q].n) return DSM_EINVAL;
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  const uint32_t r = e->qref[q][u];
  HIPCHK(hipMemcpy(words, e->bm.p + (size_t)r * e->words, (size_t)e->words * 8, hipMemcpyDeviceToHost));
  return DSM_OK;
}

int dsm_get_query_time(dsm_engine *e, double *ms, uint32_t num_queries) {
  if (!e || !ms || num_queries != e->queries.size()) return DSM_EINVAL;
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  std::vector<unsigned long long> t(num_queries);
  HIPCHK(hipMemcpy(t.data(), e->query_busy.p, (size_t)num_queries * 8, hipMemcpyDeviceToHost));
  HIPCHK(hipMemset(e->query_busy.p, 0, (size_t)num_queries * 8));
  for (uint32_t q = 0; q < num_queries; q++) ms[q] = (double)t[q] / (double)e->wall_khz;
  return DSM_OK;
}

int dsm_autotune(dsm_engine *e, const dsm_change *sample, uint32_t k, dsm_tune_report *rep) {
  if (!e || (!sample && k)) return DSM_EINVAL;
  if (e->batch_pending) return e->fail_msg(DSM_EINVAL, "a batch is applied but not matched yet");
  for (uint32_t i = 0; i < k; i++)
    if (sample[i].src >= e->n || sample[i].dst >= e->n)
      return e->fail_msg(DSM_EINVAL, "sample record %u: endpoint out of range", i);
  HIPCHK(hipSetDevice(e->opt.device));
  int rc;
  const uint32_t nq = (uint32_t)e->queries.size();
  e->grid_given = true;  // a trial runs on the grid it stands for, and the one found is kept
  std::vector<uint32_t> s(k), d(k);
  for (uint32_t i = 0; i < k; i++) {
    s[i] = sample[i].src;
    d[i] = sample[i].dst;
  }
  if ((rc = ensure_seed_cap(e, k))) return rc;
  DevBuf<uint32_t> &rb = e->rec_neg;
  if ((rc = upload_records(e, s, d, rb))) return rc;
  // the staging buffer is free again before an update (below) refills it
  HIPCHK(hipStreamSynchronize(e->stream));
  struct Cfg {
    uint32_t wpb, bpc, dmin, lw;
    bool ls, seg;
    uint32_t dev, lb;
    bool pl;
  };
  auto max_bpc = [&](uint32_t wpb) { return dfs_bpc(e, wpb); };
  // With overlap_apply, pipelined rounds run beside the next batch's update
  // (on the second copy of the graph), which competes for the CUs: each trial
  // round then runs beside the update of the first quarter of the sample (the
  // sample being a few batches), applied to the second copy and dropped, and
  // a trial's time is the makespan of both.
  HostDelta load;
  const bool loaded = e->overlap_apply && !e->tuple_cap && k >= 4;
  if (loaded) host_delta(e, sample, k / 4, load);
  // times one sample round under c and checks its counts against the first
  std::vector<unsigned long long> ref_counts;
  uint32_t trials = 0;
  auto timed = [&](const Cfg &c, float &ms) -> int {
    e->dfs_wpb = c.wpb;
    e->dfs_blocks = c.bpc * (uint32_t)e->num_cu;
    e->donate_min = c.dmin;
    e->lane_work = c.lw;
    e->leaf_budget = c.lb;
    e->leaf_sets = c.ls;
    e->leaf_segments = c.seg;
    e->donate_every = c.dev;
    e->bit_probe_last = c.pl;
    if (loaded) HIPCHK(hipEventRecord(e->ev_pre, e->stream));
    e->counts_stale = true;
    int rc2 = run_round(e, rb.p, rb.p + k, k, 0, e->ev[9], e->ev[10], e->ev[11]);
    if (rc2) return rc2;
    if (loaded && (rc2 = overlap_apply(e, load, true, false))) return rc2;
    if ((rc2 = fetch_results(e))) return rc2;
    uint64_t seeds = 0;
    if ((rc2 = check_round(e, &seeds))) return rc2;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[10], e->ev[11]));
    if (loaded) {
      // the makespan of the round and the update beside it: a shape that
      // leaves the update no room on the CUs delays it past the round
      float ua = 0;
      HIPCHK(hipEventElapsedTime(&ua, e->ev[10], e->ev[2]));
      ms = std::max(ms, ua);
    }
    std::vector<unsigned long long> cnt(e->h_counts(), e->h_counts() + 2 * (size_t)nq);
    if (ref_counts.empty()) ref_counts = cnt;
    else if (cnt != ref_counts)
      return e->fail_msg(DSM_EDEVICE, "autotune: launch configurations disagree on the counts");
    return DSM_OK;
  };
  Cfg best{e->dfs_wpb, e->dfs_blocks / (uint32_t)e->num_cu, e->donate_min, e->lane_work, e->leaf_sets,
           e->leaf_segments, e->donate_every, e->leaf_budget, e->bit_probe_last};
  // warm-up: clocks and caches settle before anything is compared
  float best_ms = 1e30f;
  for (int r = 0; r < 4; r++) {
    float t = 0;
    if ((rc = timed(best, t))) return rc;
    if (r >= 2) best_ms = std::min(best_ms, t);
  }
  const float ms0 = best_ms;
  // A candidate is timed in three pairs interleaved with the incumbent (so a
  // drift of the clocks hits both alike) and must beat it by 3% in every pair.
  auto consider = [&](const Cfg &c) -> int {
    float tb = 1e30f, tc = 1e30f;
    bool wins = true;
    for (int r = 0; r < 3; r++) {
      float t = 0, u = 0;
      int rc2 = timed(best, t);
      if (rc2) return rc2;
      tb = std::min(tb, t);
      if ((rc2 = timed(c, u))) return rc2;
      tc = std::min(tc, u);
      wins = wins && u < 0.97f * t;
    }
    trials++;
    if (wins) {
      best = c;
      best_ms = tc;
    } else {
      best_ms = std::min(best_ms, tb);
    }
    return DSM_OK;
  };
  // 1. waves per block (each at its occupancy limit); a tuple engine has one shape
  if (!e->tuple_cap) {
    const Cfg base = best;
    for (uint32_t w : {1u, 2u, 4u, 8u}) {
      if (w == base.wpb || w * dfs_lds_bytes_per_wave(e->max_qn) > 65536) continue;
      Cfg c = base;
      c.wpb = w;
      c.bpc = max_bpc(w);
      if ((rc = consider(c))) return rc;
    }
  }
  // 2. blocks per CU below the occupancy limit
  {
    const Cfg base = best;
    const uint32_t m = max_bpc(base.wpb);
    for (uint32_t b : {m, (m * 3 + 3) / 4, (m + 1) / 2}) {
      if (b == base.bpc || b == 0) continue;
      Cfg c = base;
      c.bpc = b;
      if ((rc = consider(c))) return rc;
    }
  }
  // 3. donation threshold and how often busy waves look for idle ones
  {
    const Cfg base = best;
    for (uint32_t v : {64u, 128u, 256u, 512u, 1024u}) {
      if (v == base.dmin) continue;
      Cfg c = base;
      c.dmin = v;
      if ((rc = consider(c))) return rc;
    }
    const Cfg base2 = best;
    for (uint32_t v : {4u, 8u, 16u, 32u}) {
      if (v == base2.dev) continue;
      Cfg c = base2;
      c.dev = v;
      if ((rc = consider(c))) return rc;
    }
  }
  // 4. leaf sets, 5. lane work
  if (!e->tuple_cap) {
    Cfg c = best;
    c.ls = !best.ls;
    if ((rc = consider(c))) return rc;
    if (best.ls) {
      Cfg c3 = best;
      c3.seg = !best.seg;
      if ((rc = consider(c3))) return rc;
      const Cfg base = best;
      for (uint32_t v : {8u, 16u, 24u, 48u, 64u}) {
        if (v == base.lw) continue;
        Cfg c2 = base;
        c2.lw = v;
        if ((rc = consider(c2))) return rc;
      }
      // 6. leaf budget per window (0xFFFFFFFF: none)
      const Cfg base6 = best;
      for (uint32_t v : {512u, 2048u, 8192u, 32768u, 0xFFFFFFFFu}) {
        if (v == base6.lb) continue;
        Cfg c6 = base6;
        c6.lb = v;
        if ((rc = consider(c6))) return rc;
      }
    }
  }
  // 7. candidate bit before or after the membership tests
  {
    Cfg c = best;
    c.pl = !best.pl;
    if ((rc = consider(c))) return rc;
  }
  // 8. matching order per query. The queries' plans are rebuilt with each
  // order rule in turn (all queries at once: each query's task time is
  // measured on its own), in the order 0..3 then 3..0 so that a drift of the
  // clocks hits every rule alike; a query keeps the rule with the least task
  // time if it beats its current rule by 5%. The new orders are kept only if
  // the sample round is then faster in three interleaved pairs.
  uint32_t order_changed = 0;
  {
    auto use_rules = [&](const std::vector<uint32_t> &rule) -> int {
      for (uint32_t q = 0; q < nq; q++) e->queries[q].order_variant = rule[q];
      build_plans(e);
      HIPCHK(hipMemcpy(e->d_plans.p, e->plans.data(), e->plans.size() * sizeof(Plan), hipMemcpyHostToDevice));
      return DSM_OK;
    };
    auto take_query_ms = [&](std::vector<double> *acc) -> int {
      std::vector<double> ms(nq);
      if (int r2 = dsm_get_query_time(e, ms.data(), nq)) return r2;
      if (acc)
        for (uint32_t q = 0; q < nq; q++) (*acc)[q] += ms[q];
      return DSM_OK;
    };
    std::vector<uint32_t> cur(nq);
    for (uint32_t q = 0; q < nq; q++) cur[q] = e->queries[q].order_variant;
    std::vector<std::vector<double>> qms(kOrderVariants, std::vector<double>(nq, 0.0));
    if ((rc = take_query_ms(nullptr))) return rc;
    for (uint32_t pass = 0; pass < 2; pass++)
      for (uint32_t i = 0; i < kOrderVariants; i++) {
        const uint32_t v = pass ? kOrderVariants - 1 - i : i;
        if ((rc = use_rules(std::vector<uint32_t>(nq, v)))) return rc;
        float t = 0;
        if ((rc = timed(best, t))) return rc;
        if ((rc = take_query_ms(&qms[v]))) return rc;
      }
    std::vector<uint32_t> pick = cur;
    for (uint32_t q = 0; q < nq; q++) {
      double bt = qms[cur[q]][q];
      for (uint32_t v = 0; v < kOrderVariants; v++)
        if (qms[v][q] < 0.95 * qms[cur[q]][q] && qms[v][q] < bt) {
          bt = qms[v][q];
          pick[q] = v;
        }
    }
    if (pick != cur) {
      float t_cur = 0, t_new = 0;
      for (int r = 0; r < 3; r++) {
        float t = 0;
        if ((rc = use_rules(cur)) || (rc = timed(best, t))) return rc;
        t_cur += t;
        if ((rc = use_rules(pick)) || (rc = timed(best, t))) return rc;
        t_new += t;
      }
      if (t_new < t_cur) {
        for (uint32_t q = 0; q < nq; q++) order_changed += pick[q] != cur[q];
      } else if ((rc = use_rules(cur))) {
        return rc;
      }
    } else if ((rc = use_rules(cur))) {
      return rc;
    }
    if ((rc = take_query_ms(nullptr))) return rc;
  }
  // the kept configuration, timed once more
  best_ms = 1e30f;
  for (int r = 0; r < 2; r++) {
    float t = 0;
    if ((rc = timed(best, t))) return rc;
    best_ms = std::min(best_ms, t);
  }
  if (rep) {
    rep->waves_per_block = best.wpb;
    rep->blocks_per_cu = best.bpc;
    rep->donate_min = best.dmin;
    rep->lane_work = best.lw;
    rep->leaf_sets = best.ls ? 1 : 0;
    rep->leaf_segments = best.seg ? 1 : 0;
    rep->donate_every = best.dev;
    rep->leaf_budget = best.lb;
    rep->bit_probe_last = best.pl ? 1 : 0;
    rep->order_changed = order_changed;
    rep->trials = trials;
    rep->ms_initial = ms0;
    rep->ms_best = best_ms;
  }
  return DSM_OK;
}

uint32_t dsm_num_vertices(const dsm_engine *e) { return e ? e->n : 0; }
uint32_t dsm_num_queries(const dsm_engine *e) { return e ? (uint32_t)e->queries.size() : 0; }

}  // extern "C"

// ============================================================ served stream
//
// A request is one update batch. The worker thread keeps a rolling pipeline
// over the submitted requests, in submission order, with the semantics of
// dsm_process_batch for each: request R's negatives are matched in the graph
// before R's update, its positives after it. The positives of the request in
// flight (P, already applied) and the negatives of the next one (R) see the
// same graph, so one DFS launch matches both, each seed tagged with its
// request's count slot. While that launch runs, the host computes R's delta;
// when it ends, P's counts are complete and are published at once, and R's
// update is applied. A request is admitted when it and the one in flight fit
// the memory budget together; one that does not fit even alone is rejected.

#include <chrono>
#include <condition_variable>
#include <deque>
#include <mutex>
#include <thread>
#include <unordered_map>

namespace {

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// One update batch in the rolling pipeline (served stream and
// dsm_process_batches): its records, split into positive and negative seed
// lists, its count slot and, once published, its counts.
struct PipeItem {
  const dsm_change *rec = nullptr;
  uint32_t nrec = 0;
  std::vector<uint32_t> ps, pd, ns, nd;
  uint32_t slot = 0;
  std::vector<uint64_t> pos, neg;
};

void pipe_split(const dsm_engine *e, PipeItem &it) {
  for (uint32_t i = 0; i < it.nrec; i++) {
    const dsm_change &c = it.rec[i];
    if (c.add) {
      it.ps.push_back(c.src);
      it.pd.push_back(c.dst);
    } else if (e->opt.count_negatives) {
      it.ns.push_back(c.src);
      it.nd.push_back(c.dst);
    }
  }
}

struct ServerReq : PipeItem {
  uint64_t id = 0;
  std::vector<dsm_change> ch;
  uint64_t bytes = 0;
  double t_submit = 0, t_start = 0, t_done = 0;
  uint32_t queue_depth = 0, fused = 0;
  int status = 1;  // 1 while pending or in flight
};

}  // namespace

struct dsm_server {
  dsm_engine *e = nullptr;
  uint64_t budget = 0;
  std::mutex mu;
  std::condition_variable cv_work, cv_done;
  std::deque<ServerReq *> pending;
  std::unordered_map<uint64_t, ServerReq *> reqs;
  uint64_t next_id = 1;
  bool stop = false;
  int failed = DSM_OK;  // after a device error every later request fails with it
  std::thread worker;
  PinnedBuf<uint32_t> h_rec;
  DevBuf<uint32_t> d_rec;
  std::string err;
};

namespace {

uint64_t request_bytes(const dsm_engine *e, uint32_t k) {
  // seed table (plan, src, dst, tag per seed) + records on the device + the
  // host-side delta arrays uploaded for the update
  return (uint64_t)k * ((uint64_t)std::max<uint32_t>(e->max_plans_per_key, 1) * 16 + 8 + 48);
}

void publish(dsm_server *sv, ServerReq *r, int status) {
  std::lock_guard<std::mutex> lk(sv->mu);
  r->status = status;
  r->t_done = now_s();
  sv->cv_done.notify_all();
}

// One DFS round over the current graph: the positives of P (if any) and the
// negatives of R (if any); then P's count slot is copied to the host. Waits
// for the round; while it runs, computes R's delta into *d, unless
// `have_delta` says that *d already holds it. With `stats`, the round's work
// counters and time go to the engine's statistics.
// One pipelined round: the positives of P and the negatives of R in one DFS
// launch on the current graph. With `applied` given and overlap_apply on, R's
// update is applied to the second copy of the graph meanwhile and *applied is
// set; otherwise the caller applies it after the round.
int pipe_round(dsm_engine *e, PinnedBuf<uint32_t> &h_rec, DevBuf<uint32_t> &d_rec, PipeItem *P, PipeItem *R,
               HostDelta *d, bool stats, bool *applied, bool have_delta = false) {
  const uint32_t nq = (uint32_t)e->queries.size();
  int rc;
  const uint32_t np = P ? (uint32_t)P->ps.size() : 0u, nn = R ? (uint32_t)R->ns.size() : 0u;
  const bool overlap = applied && R && d && e->overlap_apply;
  if (applied) *applied = false;
  if (overlap) HIPCHK(hipEventRecord(e->ev_pre, e->stream));
  e->counts_stale = false;  // a slot of this round's is cleared instead
  ClearSpan clear{};
  if (R) clear = ClearSpan{nullptr, e->counts() + (size_t)R->slot * nq * 2, nq * 2};
  if (np + nn) {
    if ((rc = ensure_seed_cap(e, np + nn))) return rc;
    HIPCHK(h_rec.ensure(2 * (size_t)(np + nn) + 2));
    HIPCHK(d_rec.ensure(2 * (size_t)(np + nn) + 2));
    uint32_t *h = h_rec.p;
    if (np) {
      std::copy(P->ps.begin(), P->ps.end(), h);
      std::copy(P->pd.begin(), P->pd.end(), h + np);
    }
    if (nn) {
      std::copy(R->ns.begin(), R->ns.end(), h + 2 * np);
      std::copy(R->nd.begin(), R->nd.end(), h + 2 * np + nn);
    }
    SmallCopy up{};
    if (2 * (size_t)(np + nn) <= kSmallCopy) up = {h, d_rec.p, 2 * (np + nn)};
    else HIPCHK(hipMemcpyAsync(d_rec.p, h, 2 * (size_t)(np + nn) * 4, hipMemcpyHostToDevice, e->stream));
    RoundPart parts[2];
    int nparts = 0;
    if (np) parts[nparts++] = RoundPart{d_rec.p, d_rec.p + np, np, (P->slot << 1) | 1u};
    if (nn) parts[nparts++] = RoundPart{d_rec.p + 2 * np, d_rec.p + 2 * np + nn, nn, R->slot << 1};
    if ((rc = dfs_round(e, parts, nparts, stats ? e->ev[9] : nullptr, nullptr, stats ? e->ev[11] : nullptr, up, clear)))
      return rc;
  } else if (R) {
    HIPCHK(launch_ctl_reset(nullptr, nullptr, clear.counts, clear.ncounts, nullptr, 0, {}, e->stream));
  }
  if (P)
    HIPCHK(to_host(e->h_counts() + (size_t)P->slot * nq * 2, e->counts() + (size_t)P->slot * nq * 2, (size_t)nq * 2,
                   e->stream));
  if (R && d && !have_delta) host_delta(e, R->rec, R->nrec, *d);
  if (overlap) {
    if ((rc = overlap_apply(e, *d, stats))) return rc;
    *applied = true;
  }
  HIPCHK(hipStreamSynchronize(e->stream));
  if (np + nn) {
    if (!stats && (rc = round_error(e))) return rc;
    if (stats) {
      uint64_t seeds = 0;
      if ((rc = check_round(e, &seeds))) return rc;
      e->stats.seeds_pos += seeds;
      float ms = 0;
      HIPCHK(hipEventElapsedTime(&ms, e->ev[9], e->ev[11]));
      e->stats.ms_dfs_pos += ms;
    }
  }
  if (P) {
    P->pos.assign(nq, 0);
    P->neg.assign(nq, 0);
    const unsigned long long *c = e->h_counts() + (size_t)P->slot * nq * 2;
    for (uint32_t q = 0; q < nq; q++) {
      P->pos[q] = c[2 * q + 1];
      P->neg[q] = c[2 * q + 0];
    }
  }
  return DSM_OK;
}

int serve_round(dsm_server *sv, ServerReq *P, ServerReq *R, HostDelta *d, bool *applied) {
  return pipe_round(sv->e, sv->h_rec, sv->d_rec, P, R, d, false, applied);
}

void server_loop(dsm_server *sv) {
  dsm_engine *e = sv->e;
  if (hipSetDevice(e->opt.device) != hipSuccess) sv->failed = DSM_EDEVICE;
  ServerReq *P = nullptr;  // applied, positives not yet matched
  for (;;) {
    ServerReq *R = nullptr;
    {
      std::unique_lock<std::mutex> lk(sv->mu);
      if (!P) sv->cv_work.wait(lk, [&] { return sv->stop || !sv->pending.empty(); });
      while (!sv->pending.empty()) {
        ServerReq *c = sv->pending.front();
        const int adm = sv->failed != DSM_OK ? sv->failed : dsm_admit(c->bytes, P ? P->bytes : 0, sv->budget);
        if (adm < 0) {
          // rejected without touching the graph
          sv->pending.pop_front();
          c->status = adm;
          c->t_start = c->t_done = now_s();
          sv->cv_done.notify_all();
          continue;
        }
        if (adm == 0) break;  // waits until the request in flight is done
        sv->pending.pop_front();
        R = c;
        R->queue_depth = (uint32_t)sv->pending.size();
        break;
      }
      if (!P && !R) {
        if (sv->stop && sv->pending.empty()) return;
        continue;
      }
    }
    if (R) {
      R->t_start = now_s();
      R->slot = P ? P->slot ^ 1u : 0u;
      R->fused = P ? 1u : 0u;
      pipe_split(e, *R);
    }
    HostDelta d;
    bool applied = false;
    int rc = serve_round(sv, P, R, R ? &d : nullptr, &applied);
    if (P) publish(sv, P, rc);
    if (rc == DSM_OK && R && !applied) rc = apply_delta_and_refresh(e, d);
    if (rc != DSM_OK) {
      std::lock_guard<std::mutex> lk(sv->mu);
      sv->failed = rc;
      sv->err = e->err;
    }
    if (R && rc != DSM_OK) {
      publish(sv, R, rc);
      R = nullptr;
    }
    P = R;
  }
}

}  // namespace

extern "C" {

int dsm_admit(uint64_t request_bytes, uint64_t in_flight_bytes, uint64_t budget) {
  if (request_bytes > budget) return DSM_EADMIT;
  return in_flight_bytes <= budget - request_bytes ? 1 : 0;
}

uint64_t dsm_estimate_request_bytes(const dsm_engine *e, uint32_t num_changes) {
  return e ? request_bytes(e, num_changes) : 0;
}

int dsm_server_create(dsm_engine *e, const dsm_server_options *opt, dsm_server **out) {
  if (!e || !out) return DSM_EINVAL;
  *out = nullptr;
  if (e->tuple_cap) return e->fail_msg(DSM_EINVAL, "served mode keeps counts only (tuple_capacity must be 0)");
  HIPCHK(hipSetDevice(e->opt.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  // the second copy of the graph is part of the engine, not of the budget
  if (e->overlap_apply)
    if (int rc = reserve_shadow(e)) return rc;
  std::unique_ptr<dsm_server> sv(new dsm_server());
  sv->e = e;
  size_t freeb = 0, totalb = 0;
  HIPCHK(hipMemGetInfo(&freeb, &totalb));
  const double headroom = (opt && opt->hbm_headroom > 0) ? opt->hbm_headroom : 0.30;
  const double reserve = headroom * (double)totalb;
  if (opt && opt->budget_bytes) sv->budget = opt->budget_bytes;
  else sv->budget = (double)freeb > reserve ? (uint64_t)((double)freeb - reserve) : 0;
  dsm_server *p = sv.get();
  p->worker = std::thread(server_loop, p);
  *out = sv.release();
  return DSM_OK;
}

int dsm_server_submit(dsm_server *sv, const dsm_change *changes, uint32_t num_changes, uint64_t *id) {
  if (!sv || (!changes && num_changes) || !id) return DSM_EINVAL;
  const uint32_t n = sv->e->n;
  for (uint32_t i = 0; i < num_changes; i++)
    if (changes[i].src >= n || changes[i].dst >= n) return DSM_EINVAL;
  ServerReq *r = new ServerReq();
  r->ch.assign(changes, changes + num_changes);
  r->rec = r->ch.data();
  r->nrec = num_changes;
  r->bytes = request_bytes(sv->e, num_changes);
  r->t_submit = now_s();
  {
    std::lock_guard<std::mutex> lk(sv->mu);
    r->id = sv->next_id++;
    sv->reqs[r->id] = r;
    sv->pending.push_back(r);
    *id = r->id;
  }
  sv->cv_work.notify_one();
  return DSM_OK;
}

int dsm_server_wait(dsm_server *sv, uint64_t id, dsm_request_info *info, uint64_t *pos, uint64_t *neg) {
  if (!sv) return DSM_EINVAL;
  ServerReq *r;
  {
    std::unique_lock<std::mutex> lk(sv->mu);
    auto it = sv->reqs.find(id);
    if (it == sv->reqs.end()) return DSM_EINVAL;
    r = it->second;
    sv->cv_done.wait(lk, [&] { return r->status != 1; });
    sv->reqs.erase(it);
  }
  const uint32_t nq = (uint32_t)sv->e->queries.size();
  if (info) {
    info->id = r->id;
    info->status = r->status;
    info->t_submit = r->t_submit;
    info->t_start = r->t_start;
    info->t_done = r->t_done;
    info->queue_depth = r->queue_depth;
    info->fused = r->fused;
    info->num_changes = (uint32_t)r->ch.size();
  }
  for (uint32_t q = 0; q < nq; q++) {
    if (pos) pos[q] = r->status == DSM_OK ? r->pos[q] : 0;
    if (neg) neg[q] = r->status == DSM_OK ? r->neg[q] : 0;
  }
  const int st = r->status;
  delete r;
  return st;
}

const char *dsm_server_error(const dsm_server *sv) { return sv ? sv->err.c_str() : ""; }

int dsm_process_batches(dsm_engine *e, const dsm_change *changes, const uint32_t *batch_offsets,
                        uint32_t num_batches, uint64_t *pos, uint64_t *neg, double *done_s) {
  if (!e || !batch_offsets || (!changes && batch_offsets[num_batches]) || !pos || !neg) return DSM_EINVAL;
  if (e->tuple_cap) return e->fail_msg(DSM_EINVAL, "pipelined batches keep counts only (tuple_capacity must be 0)");
  if (e->batch_pending) return e->fail_msg(DSM_EINVAL, "a batch is applied but not matched yet");
  for (uint32_t b = 0; b < num_batches; b++)
    if (batch_offsets[b + 1] < batch_offsets[b]) return e->fail_msg(DSM_EINVAL, "batch offsets decrease");
  for (uint32_t i = 0; i < batch_offsets[num_batches]; i++)
    if (changes[i].src >= e->n || changes[i].dst >= e->n)
      return e->fail_msg(DSM_EINVAL, "change %u: endpoint out of range (%u,%u) for %u vertices", i,
                         changes[i].src, changes[i].dst, e->n);
  HIPCHK(hipSetDevice(e->opt.device));
  e->stats = dsm_stats{};
  const uint32_t nq = (uint32_t)e->queries.size();
  std::vector<PipeItem> items(num_batches);
  for (uint32_t b = 0; b < num_batches; b++) {
    items[b].rec = changes + batch_offsets[b];
    items[b].nrec = batch_offsets[b + 1] - batch_offsets[b];
    pipe_split(e, items[b]);
  }
  auto publish_item = [&](uint32_t b) {
    for (uint32_t q = 0; q < nq; q++) {
      pos[(size_t)b * nq + q] = items[b].pos[q];
      neg[(size_t)b * nq + q] = items[b].neg[q];
    }
    if (done_s) done_s[b] = std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
  };
  int rc;
  bool apply_timed = false;
  auto take_apply_time = [&]() -> int {
    if (!apply_timed) return DSM_OK;
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[0], e->ev[2]));
    e->stats.ms_apply += ms;
    apply_timed = false;
    return DSM_OK;
  };
  // A batch's host delta (its records as per-vertex insert and delete lists)
  // depends on its records alone. A worker thread computes them in batch
  // order, ahead of the rounds, while this thread waits for the GPU; a round
  // then enqueues its update right behind its DFS launch instead of after
  // sorting its batch (at 32,768 records, a few ms per batch). The worker
  // stays at most kDeltasAhead batches ahead of the rounds, so the deltas
  // held at once stay bounded however many batches the call takes.
  constexpr uint32_t kDeltasAhead = 2;
  std::vector<HostDelta> deltas(num_batches);
  std::mutex dmu;
  std::condition_variable ready_cv, taken_cv;
  uint32_t dready = 0, dtaken = 0;
  bool dstop = false;
  std::thread dworker([&] {
    for (uint32_t b = 0; b < num_batches; b++) {
      {
        std::unique_lock<std::mutex> lk(dmu);
        taken_cv.wait(lk, [&] { return dstop || b < dtaken + kDeltasAhead; });
        if (dstop) return;
      }
      host_delta(e, items[b].rec, items[b].nrec, deltas[b]);
      {
        std::lock_guard<std::mutex> lk(dmu);
        dready = b + 1;
      }
      ready_cv.notify_one();
    }
  });
  struct JoinWorker {
    std::thread &t;
    std::mutex &mu;
    std::condition_variable &cv;
    bool &stop;
    ~JoinWorker() {
      {
        std::lock_guard<std::mutex> lk(mu);
        stop = true;
      }
      cv.notify_one();
      t.join();
    }
  } join_worker{dworker, dmu, taken_cv, dstop};
  PipeItem *P = nullptr;
  for (uint32_t b = 0; b < num_batches; b++) {
    PipeItem *R = &items[b];
    R->slot = P ? P->slot ^ 1u : 0u;
    {
      std::unique_lock<std::mutex> lk(dmu);
      ready_cv.wait(lk, [&] { return dready > b; });
      dtaken = b + 1;
    }
    taken_cv.notify_one();
    HostDelta d = std::move(deltas[b]);
    bool applied = false;
    if ((rc = pipe_round(e, e->pipe_h_rec, e->pipe_d_rec, P, R, &d, true, &applied, true))) return rc;
    if ((rc = take_apply_time())) return rc;
    if (P) publish_item(b - 1);
    if (!applied) {
      HIPCHK(hipEventRecord(e->ev[0], e->stream));
      if ((rc = apply_delta_and_refresh(e, d, nullptr, e->ev[2]))) return rc;
      apply_timed = true;
    }
    P = R;
  }
  if (P) {
    if ((rc = pipe_round(e, e->pipe_h_rec, e->pipe_d_rec, P, nullptr, nullptr, true, nullptr))) return rc;
    if ((rc = take_apply_time())) return rc;
    publish_item(num_batches - 1);
  }
  e->stats.pool_entries_used = e->h_actl.p->pool_used;
  e->stats.pool_entries_capacity = e->pool_cap;
  return DSM_OK;
}

void dsm_server_destroy(dsm_server *sv) {
  if (!sv) return;
  {
    std::lock_guard<std::mutex> lk(sv->mu);
    sv->stop = true;
  }
  sv->cv_work.notify_all();
  if (sv->worker.joinable()) sv->worker.join();
  for (auto &kv : sv->reqs) delete kv.second;
  delete sv;
}

}  // extern "C"
