// HIP kernels of the cluster-encoding candidate refinement (gfx950, wave64).
//
// The reference runs one kernel per cluster with a warp per candidate of the
// cluster's core and a cudaDeviceSynchronize after each (encodeKernel,
// mergeKernel, combineMultipleClustersKernel, filter.cu:615-934, driven by
// encode(), filter.cu:936-1177), over vertex-major 32-bit encoding words
// (filter.cu:1546). Here every position is a bitmap row of its own beside the
// LDF/NLF rows, so a query vertex's refined candidates are one row the DFS
// reads directly (no compact pass), and one launch runs the same pass step of
// every standing query:
//
//   k_cluster_init   zero the position rows, load each core's candidate list
//                    (the LDF/NLF row) into its alive row
//   k_cluster_pass   a wave per (query pass, 64 bitmap words): each lane owns
//                    one 64-vertex word of the core's alive row, tests the
//                    pass's core condition for all 64 vertices with one load
//                    per condition row, writes the core and alive words, then
//                    the wave reads the lists of 64 candidates at a time as one
//                    (of a list longer than 64 entries only the label buckets
//                    of the pass's targets, from the label-sorted copy) and
//                    sets or clears the targets' bits; buckets of more than
//                    kClusterChunk entries are queued in chunks
//   k_cluster_heavy  a wave per such chunk
//
// A pass only reads rows of earlier clusters and only writes its own
// cluster's rows and its core's alive row, and the passes of one step belong
// to different queries, so the work items of a launch are independent. Every
// bit update is an atomic read-modify-write on its 64-bit word (the
// reference's plain read-modify-write of a core word, filter.cu:765, could
// drop a neighbouring bit set concurrently); a load first skips updates that
// would change nothing.
#include <algorithm>

#include "dsm_device.h"
#include "dsm_internal.h"

namespace dsm {
namespace {

constexpr int kClusterWaves = 4;

// A commit or merge of the update that the refinement follows found no room: some
// lists have moved while their label-sorted copies wait to be built, so none is
// walked. The refinement is launched again once there is room.
__device__ __forceinline__ bool held_up(const ApplyCtl *actl) { return actl->overflow | actl->merge_overflow; }

// The pass's targets at neighbours w[u] of candidates (lane-parallel: every lane its
// own, those with `in`): the targets of the neighbour's label (every condition row
// implies the target's label, and a combine into an existing cluster holds no bit of
// another label to clear). lab[u] is that label, or, from a label-sorted list, its
// bucket for every u. Encode, merge and new combines set the target's bit when its
// condition rows all hold w; combines into an existing cluster clear it when they do
// not. A target costs one read per condition row and one of its own word, for all U
// neighbours together. All lanes of the wave call it.
template <int U>
__device__ __forceinline__ void visit(const ClusterArgs &a, const ClusterOp &op, uint32_t kind, const uint8_t *of,
                                      const uint32_t (&w)[U], const uint32_t (&lab)[U], const bool (&in)[U]) {
  for (uint32_t t = 0; t < op.ntarget; t++) {
    bool mine[U], cond[U], any = false;
#pragma unroll
    for (int u = 0; u < U; u++) {
      mine[u] = cond[u] = in[u] && lab[u] == of[t];
      any |= mine[u];
    }
    if (ballot(any) == 0) continue;
    const uint32_t o = op.toff[t], c = op.tcnt[t];
    for (uint32_t k = 0; k < c; k++) {
      const uint64_t *row = a.bm + (size_t)a.crow[o + k] * a.words;
      uint64_t x[U];
#pragma unroll
      for (int u = 0; u < U; u++) x[u] = cond[u] ? ld_relaxed(&row[w[u] >> 6]) : 0;
#pragma unroll
      for (int u = 0; u < U; u++) cond[u] = (x[u] >> (w[u] & 63)) & 1;
    }
    unsigned long long *row = (unsigned long long *)a.bm + (size_t)(op.core + 1 + t) * a.words;
    const bool keep = kind == kOpCombineKeep;
    uint64_t x[U];
#pragma unroll
    for (int u = 0; u < U; u++) x[u] = mine[u] && cond[u] != keep ? ld_relaxed(&row[w[u] >> 6]) : 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint64_t bit = 1ull << (w[u] & 63);
      if (!mine[u] || cond[u] == keep || ((x[u] & bit) != 0) != keep) continue;
      if (keep) atomicAnd(&row[w[u] >> 6], (unsigned long long)~bit);
      else atomicOr(&row[w[u] >> 6], (unsigned long long)bit);
    }
  }
}

// A wave's arrays for reading many lists as one.
struct WaveLists {
  uint32_t pre[65], from[64];
};

// The entries of the lanes' lists, `len` of them from list[from], as one array, four
// a lane at a time: f(entries, which of them are).
template <typename F>
__device__ __forceinline__ void each_entry(WaveLists &wl, const uint32_t *list, uint32_t from, uint32_t len, F f) {
  const uint32_t lane = lane_id();
  wave_sync();  // the previous lists' arrays are no longer read
  if (lane == 0) wl.pre[0] = 0;
  wl.pre[lane + 1] = wave_incl_sum(len);
  wl.from[lane] = from;
  wave_sync();
  const uint32_t total = wl.pre[64];
  for (uint32_t e = 0; e < total; e += 256) {
    uint32_t k[4], o[4], w[4];
    bool in[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      in[u] = e + u * 64 + lane < total;
      k[u] = min(e + u * 64 + lane, total - 1);
    }
    ranges_of(wl.pre, k, o);
#pragma unroll
    for (int u = 0; u < 4; u++) w[u] = list[wl.from[o[u]] + (k[u] - wl.pre[o[u]])];
    f(w, in);
  }
}

// The neighbours of the lanes' candidates v (those with `valid`) that the targets
// of pass j can use. A list of more than kLabelSorted entries is read only in the
// label buckets of the targets (its label-sorted copy); a bucket of more than
// kClusterChunk entries is queued in chunks for k_cluster_heavy.
__device__ __forceinline__ void walk_candidates(const ClusterArgs &a, const ClusterOp &op, uint32_t kind, uint32_t j,
                                                uint32_t v, bool valid, WaveLists &wl) {
  const uint32_t st = valid ? a.g.start[v] : 0u, dg = valid ? a.g.deg[v] : 0u;
  each_entry(wl, a.g.pool, st, dg <= kLabelSorted ? dg : 0u, [&](const uint32_t(&w)[4], const bool(&in)[4]) {
    uint32_t lab[4];
#pragma unroll
    for (int u = 0; u < 4; u++) lab[u] = a.g.lab[w[u]];
    visit<4>(a, op, kind, op.tlab, w, lab, in);
  });
  if (ballot(dg > kLabelSorted) == 0) return;
  const uint32_t *row = a.g.loff + (size_t)v * (a.g.nbuckets + 1);
  for (uint32_t k = 0; k < op.nlix; k++) {
    const uint32_t li = op.lix[k];
    uint32_t b0 = 0, b1 = 0;
    if (dg > kLabelSorted) {
      b0 = row[li];
      b1 = row[li + 1];
    }
    const bool heavy = b1 - b0 > kClusterChunk;
    if (ballot(heavy)) {
      const uint32_t nch = heavy ? (b1 - b0 + kClusterChunk - 1) / kClusterChunk : 0u;
      uint32_t all, first = 0;
      const uint32_t before = wave_excl_sum(nch, &all);
      if (lane_id() == 0) first = atomicAdd(&a.ctl[0], all);
      first = bcast(first) + before;
      for (uint32_t c = 0; c < nch; c++)
        if (first + c < a.heavy_cap) a.heavy[first + c] = ClusterHeavy{j, v, b0 + c * kClusterChunk, li};
      // sized by the host so that this cannot happen
      if (heavy && first + nch > a.heavy_cap) atomicAdd(&a.actl->chunks_dropped, 1u);
    }
    each_entry(wl, a.g.lpool, st + b0, heavy ? 0u : b1 - b0, [&](const uint32_t(&w)[4], const bool(&in)[4]) {
      const uint32_t lab[4] = {li, li, li, li};
      visit<4>(a, op, kind, op.tlix, w, lab, in);
    });
  }
}

// The position of the n-th (from 0) set bit of x, which has more than n.
__device__ __forceinline__ uint32_t nth_bit(uint64_t x, uint32_t n) {
  uint32_t at = 0;
#pragma unroll
  for (uint32_t w = 32; w; w >>= 1) {
    const uint32_t c = (uint32_t)__popcll(x & ((1ull << w) - 1));
    if (n >= c) {
      n -= c;
      at += w;
      x >>= w;
    }
  }
  return at;
}

__global__ __launch_bounds__(256) void k_cluster_init(uint64_t *bm, uint32_t words, uint32_t first_row,
                                                      uint32_t nrows, uint64_t *alive, const uint32_t *alive_src,
                                                      uint32_t nalive_src, uint32_t *ctl, uint32_t nctl,
                                                      const ApplyCtl *actl) {
  if (held_up(actl)) return;
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
  const size_t zero = (size_t)nrows * words, copy = (size_t)nalive_src * words;
  uint64_t *z = bm + (size_t)first_row * words;
  for (size_t i = tid; i < zero; i += stride) z[i] = 0;
  for (size_t i = tid; i < copy; i += stride) {
    const size_t r = i / words, wd = i - r * words;
    alive[(size_t)alive_src[2 * r] * words + wd] = bm[(size_t)alive_src[2 * r + 1] * words + wd];
  }
  for (size_t i = tid; i < nctl; i += stride) ctl[i] = 0;
}

// Bound by the chain of reads from a candidate to its neighbours' condition rows. A
// candidate after the other, its neighbours on the lanes, took 69 us a step for 16
// queries on 120,000 vertices; 21 us now.
__global__ __launch_bounds__(kClusterWaves * 64) void k_cluster_pass(ClusterArgs a) {
  __shared__ uint64_t s_aw[kClusterWaves][64];
  __shared__ uint32_t s_pre[kClusterWaves][65];
  __shared__ WaveLists s_lists[kClusterWaves];
  const uint32_t lane = lane_id(), wv = bcast(threadIdx.x >> 6);
  const uint32_t wave = bcast((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
  if (held_up(a.actl)) return;
  const uint32_t groups = (a.words + 63) >> 6;
  const uint64_t units = (uint64_t)a.nops * groups;
  for (uint64_t u = wave; u < units; u += nwaves) {
    const uint32_t j = bcast((uint32_t)(u / groups)), grp = bcast((uint32_t)(u - (uint64_t)j * groups));
    const ClusterOp &op = a.ops[j];
    const uint32_t kind = bcast(op.kind);
    const uint32_t wd = grp * 64 + lane;
    uint64_t aw = 0;
    if (wd < a.words) aw = a.alive[(size_t)op.alive * a.words + wd];
    // core condition, one word per lane: the vertices of this word that hold
    // every check row keep their place in the core's list
    if (aw) {
      uint64_t *core = &a.bm[(size_t)op.core * a.words + wd];
      if (kind == kOpEncode) {
        *core |= aw;
      } else {
        uint64_t pass = aw;
        for (uint32_t k = 0; k < op.ncheck && pass; k++) pass &= a.bm[(size_t)a.crow[op.check_off + k] * a.words + wd];
        if (kind == kOpCombineKeep) *core &= ~(aw & ~pass);
        else *core |= pass;
        a.alive[(size_t)op.alive * a.words + wd] = pass;
      }
    }
    // neighbours of every candidate the pass started with, 64 candidates at a time
    wave_sync();  // the previous unit's arrays are no longer read
    s_aw[wv][lane] = aw;
    if (lane == 0) s_pre[wv][0] = 0;
    s_pre[wv][lane + 1] = wave_incl_sum((uint32_t)__popcll(aw));
    wave_sync();
    const uint32_t total = s_pre[wv][64];
    for (uint32_t c = 0; c < total; c += 64) {
      const uint32_t k[1] = {min(c + lane, total - 1)};
      uint32_t l[1];
      ranges_of(s_pre[wv], k, l);
      const uint32_t v = (grp * 64 + l[0]) * 64 + nth_bit(s_aw[wv][l[0]], k[0] - s_pre[wv][l[0]]);
      walk_candidates(a, op, kind, j, v, c + lane < total, s_lists[wv]);
    }
  }
}

// The queued chunks, dealt out in turn: a wave per chunk. (With the chunks claimed
// from a counter the 4,096 waves' claims took 55 us, also when there were none; 4 us
// now.)
__global__ __launch_bounds__(kClusterWaves * 64) void k_cluster_heavy(ClusterArgs a) {
  const uint32_t lane = lane_id();
  if (held_up(a.actl)) return;
  const uint32_t total = min(bcast(a.ctl[0]), a.heavy_cap);
  for (uint32_t e = bcast((blockIdx.x * blockDim.x + threadIdx.x) >> 6); e < total; e += (gridDim.x * blockDim.x) >> 6) {
    const ClusterHeavy h = a.heavy[e];
    const uint32_t j = bcast(h.op), v = bcast(h.v), lo = bcast(h.lo), li = bcast(h.li);
    const ClusterOp &op = a.ops[j];
    const uint32_t kind = bcast(op.kind);
    const uint32_t st = a.g.start[v];
    const uint32_t b1 = a.g.loff[(size_t)v * (a.g.nbuckets + 1) + li + 1];
    const uint32_t hi = min(b1, lo + kClusterChunk);
    const uint32_t *L = a.g.lpool + st;
    for (uint32_t i = lo; i < hi; i += 256) {
      uint32_t w[4];
      bool in[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        in[u] = i + u * 64 + lane < hi;
        w[u] = L[min(i + u * 64 + lane, hi - 1)];
      }
      const uint32_t lab[4] = {li, li, li, li};
      visit<4>(a, op, kind, op.tlix, w, lab, in);
    }
  }
}

}  // namespace

hipError_t launch_cluster_init(uint64_t *bm, uint32_t words, uint32_t first_row, uint32_t nrows, uint64_t *alive,
                               const uint32_t *alive_src, uint32_t nalive_src, uint32_t *ctl, uint32_t nctl,
                               const ApplyCtl *actl, hipStream_t s) {
  const size_t work = std::max<size_t>((size_t)nrows * words, (size_t)nalive_src * words);
  const uint32_t blocks = (uint32_t)std::min<size_t>(std::max<size_t>((work + 255) / 256, 1), 4096);
  hipLaunchKernelGGL(k_cluster_init, dim3(blocks), dim3(256), 0, s, bm, words, first_row, nrows, alive, alive_src,
                     nalive_src, ctl, nctl, actl);
  return hipGetLastError();
}

hipError_t launch_cluster_pass(const ClusterArgs &a, uint32_t max_blocks, hipStream_t s) {
  const uint64_t units = (uint64_t)a.nops * ((a.words + 63) / 64);
  const uint32_t blocks =
      (uint32_t)std::min<uint64_t>(std::max<uint64_t>((units + kClusterWaves - 1) / kClusterWaves, 1), max_blocks);
  hipLaunchKernelGGL(k_cluster_pass, dim3(blocks), dim3(kClusterWaves * 64), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_cluster_heavy(const ClusterArgs &a, uint32_t blocks, hipStream_t s) {
  hipLaunchKernelGGL(k_cluster_heavy, dim3(std::max<uint32_t>(blocks, 1)), dim3(kClusterWaves * 64), 0, s, a);
  return hipGetLastError();
}

}  // namespace dsm
