// HIP kernels of the MI355X continuous subgraph matching engine (gfx950,
// wave64). Integer work only; no MFMA.
//
//   k_apply_plan / k_apply_rank / k_apply_merge / k_apply_commit
//                                   in-place batch update of the slack CSR
//                                   (the reference rebuilds the whole graph on
//                                   the host, cpuGraph.cpp:521-607, and
//                                   re-uploads it, io.cu:279-302)
//   k_relabel / k_relabel_marks     label changes of the update rule
//                                   (cpuGraph.cpp:564) + dirty marking
//   k_lbuild_pick / k_lbuild / k_lbuild_starts / k_lbuild_place
//                                   label-sorted copies of lists longer than
//                                   64 entries, rebuilt for the dirty set
//   k_filter_full / k_filter_light
//                                   LDF/NLF candidate bitmaps
//                                   (filter.cu:394-566, compact filter.cu:1692)
//   k_update_small                  all of the above for a small update, by one block
//   k_seed                          device edge seeding (main.cu:268-329;
//                                   replaces the host ResTable and join.cu)
//   k_dfs                           persistent wave64 DFS with per-wave LDS
//                                   stacks, work donation and shared leaf sets
//                                   (gpu_match.cu:96-876 restated for CDNA)
#include <algorithm>
#include <cstddef>

#include "dsm_device.h"
#include "dsm_internal.h"

namespace dsm {
namespace {

constexpr int kApplyWaves = 4;

// A commit or merge of this update found no room: the kernels after it wait for
// the host, which makes room, tries again and launches them anew.
// ONE: in the one-block update (k_update_small), whose own atomics wrote the words.
template <bool ONE = false, typename T>
__device__ __forceinline__ T ctl_word(const T &w) {
  return ONE ? ld_relaxed(&w) : w;
}
template <bool ONE = false>
__device__ __forceinline__ bool held_up(const ApplyCtl *actl) {
  return ctl_word<ONE>(actl->overflow) | ctl_word<ONE>(actl->merge_overflow);
}

__device__ __forceinline__ bool bit_of(const uint64_t *bm, uint32_t words, uint32_t sig, uint32_t v) {
  return (bm[(size_t)sig * words + (v >> 6)] >> (v & 63)) & 1ull;
}

// all 8 byte fields of x >= those of y (fields hold 0..127)
__device__ __forceinline__ bool ge_bytes(uint64_t x, uint64_t y) {
  constexpr uint64_t H = 0x8080808080808080ull;
  return (((x | H) - y) & H) == H;
}

// Marks x dirty in the update being applied. A byte a vertex, so that a mark is a
// plain store (every marker stores the same 1): bits took an atomic each, and the
// marks of 19,000 relabelled vertices' neighbours queued up for the few lines that
// hold the bits of 500,000 vertices (157 us, a third of it now). The dirty list is
// made from the marks once all are in (k_dirty_compact).
__device__ __forceinline__ void mark_dirty(const DirtyArgs &d, uint32_t x) { d.marks[x] = 1; }

// The caller's place among the block's c entries each, taken from *count with one
// add for the block: adds of every wave to one counter follow each other at some
// 20 ns. sums holds a word per wave and one more; all threads call it together.
template <typename T>
__device__ __forceinline__ T block_take(T c, T *count, T *sums) {
  const uint32_t wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  T incl = c;
  if constexpr (sizeof(T) == 4) {
    incl = wave_incl_sum(c);
  } else {
    for (int o = 1; o < 64; o <<= 1) {
      const T y = __shfl_up(incl, o);
      if (lane_id() >= (uint32_t)o) incl += y;
    }
  }
  __syncthreads();  // the previous call's sums are no longer read
  if (lane_id() == 63) sums[wv] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    T all = 0;
    for (uint32_t w = 0; w < nw; w++) {
      const T y = sums[w];
      sums[w] = all;
      all += y;
    }
    sums[nw] = all ? atomicAdd(count, all) : (T)0;
  }
  __syncthreads();
  return sums[nw] + sums[wv] + incl - c;
}

// The dirty list from the marks, which are cleared: 16 vertices a thread, a block
// prefix sum and one counter add per block; the list comes out in id order within
// each block's vertices. Only vertices with a label some query uses are listed:
// no seed, DFS level or refilter reads the label-sorted copy or the candidate bits
// of any other vertex, and one that takes such a label later is marked by its own
// relabel, so a stale copy never gets read.
constexpr uint32_t kCompactBlock = 512;
template <bool ONE>
__device__ __forceinline__ void compact_dirty(DevGraph g, DirtyArgs d) {
  __shared__ uint32_t s_sum[kCompactBlock / 64 + 1];
  const uint32_t ngroups = (g.n + 15) / 16;
  if (held_up<ONE>(d.actl)) return;
  for (uint32_t w0 = blockIdx.x * kCompactBlock; w0 < ngroups; w0 += gridDim.x * kCompactBlock) {
    const uint32_t wi = w0 + threadIdx.x;
    uint4 *at = reinterpret_cast<uint4 *>(d.marks) + wi;
    uint4 m = wi < ngroups ? *at : uint4{0, 0, 0, 0};
    uint32_t take = 0;  // bit k: vertex 16 wi + k is listed
    if (m.x | m.y | m.z | m.w) {
      *at = uint4{0, 0, 0, 0};
      const uint4 l = reinterpret_cast<const uint4 *>(g.lab)[wi];
      const uint32_t mk[4] = {m.x, m.y, m.z, m.w}, lb[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
      for (uint32_t k = 0; k < 16; k++) {
        const uint32_t sh = k % 4 * 8;
        if ((mk[k / 4] >> sh & 0xFF) && (lb[k / 4] >> sh & 0xFF) != kNoLabel) take |= 1u << k;
      }
    }
    uint32_t p = block_take((uint32_t)__popc(take), &d.actl->ndirty, s_sum);
    while (take) {
      const uint32_t k = (uint32_t)__builtin_ctz(take);
      take &= take - 1;
      if (p < d.list_cap) d.list[p] = wi * 16u + k;
      p++;
    }
  }
}
__global__ __launch_bounds__(kCompactBlock) void k_dirty_compact(DevGraph g, DirtyArgs d) {
  compact_dirty<false>(g, d);
}

// The block's part in a SmallCopy, 8 bytes a thread at a time (both sides are
// aligned to that), eight in flight.
__device__ __forceinline__ void small_copy(const SmallCopy &c) {
  const uint2 *from = reinterpret_cast<const uint2 *>(c.from);
  uint2 *to = reinterpret_cast<uint2 *>(c.to);
  const uint32_t pairs = c.words / 2;
#pragma unroll 8
  for (uint32_t i = threadIdx.x; i < pairs; i += blockDim.x) to[i] = from[i];
  if (threadIdx.x == 0 && c.words % 2) c.to[c.words - 1] = c.from[c.words - 1];
}

__global__ __launch_bounds__(256) void k_small_copy(SmallCopy c) { small_copy(c); }

__global__ __launch_bounds__(256) void k_array_copies(ArrayCopies c) {
  const size_t tid = (size_t)blockIdx.x * 256 + threadIdx.x, nth = (size_t)gridDim.x * 256;
  for (uint32_t k = 0; k < c.n; k++) {
    const uint4 *from = static_cast<const uint4 *>(c.from[k]);
    uint4 *to = static_cast<uint4 *>(c.to[k]);
    const size_t quads = c.bytes[k] / 16, words = c.bytes[k] / 4;
#pragma unroll 4
    for (size_t i = tid; i < quads; i += nth) to[i] = from[i];
    const size_t w = quads * 4 + tid;
    if (w < words) static_cast<uint32_t *>(c.to[k])[w] = static_cast<const uint32_t *>(c.from[k])[w];
  }
}

// ------------------------------------------------------------------ apply

constexpr uint32_t kBlockList = 65536;

// The lists of a *_big kernel: those of at most kBlockList entries sit at the
// front of its array (nblock of them), a block each; the longer ones at the
// back (nhuge, from index cap - 1 down), each split over every thread of the
// grid. f(entry, first, stride) gets the thread's first index into the list
// and the stride; both are multiples of 64 apart from the lane, so the lanes of
// a wave step through the list together.
template <typename F>
__device__ __forceinline__ void for_big_lists(const uint32_t *arr, uint32_t cap, uint32_t nblock, uint32_t nhuge,
                                              F f) {
  for (uint32_t r = blockIdx.x; r < nblock; r += gridDim.x) f(arr[r], threadIdx.x, blockDim.x);
  for (uint32_t r = 0; r < nhuge; r++)
    f(arr[cap - 1 - r], blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// Queues entry v of a list of len entries on a *_big kernel's array: longer
// than kBlockList at the back, else at the front.
__device__ __forceinline__ void queue_big(uint32_t *arr, uint32_t cap, uint32_t *nblock, uint32_t *nhuge,
                                          uint32_t len, uint32_t v) {
  if (len > kBlockList) arr[cap - 1 - atomicAdd(nhuge, 1u)] = v;
  else arr[atomicAdd(nblock, 1u)] = v;
}

// Copies from[0, len) to to[0, len) (disjoint); the caller's threads are
// first, first + stride, ... (stride >= 4). When both ranges share their
// alignment modulo 16 bytes (the same offset of a pool in either copy of the
// graph), the bulk moves in 16-byte pieces, four in flight per thread, with
// fewer than four entries copied singly at each end; otherwise entry by
// entry, four in flight per thread.
__device__ __forceinline__ void copy_range(const uint32_t *__restrict__ from, uint32_t *__restrict__ to,
                                           uint32_t first, uint32_t stride, uint32_t len) {
  if ((((uintptr_t)from ^ (uintptr_t)to) & 15u) != 0) {
    uint32_t j = first;
    for (; j + 3 * stride < len; j += 4 * stride) {
      const uint32_t a = from[j], b = from[j + stride], c = from[j + 2 * stride], e = from[j + 3 * stride];
      to[j] = a;
      to[j + stride] = b;
      to[j + 2 * stride] = c;
      to[j + 3 * stride] = e;
    }
    for (; j < len; j += stride) to[j] = from[j];
    return;
  }
  const uint32_t lead = (uint32_t)((16u - ((uintptr_t)from & 15u)) & 15u) >> 2;
  const uint32_t head = lead < len ? lead : len;
  if (first < head) to[first] = from[first];
  const uint32_t nv = (len - head) >> 2;
  const uint4 *__restrict__ fv = reinterpret_cast<const uint4 *>(from + head);
  uint4 *__restrict__ tv = reinterpret_cast<uint4 *>(to + head);
  uint32_t j = first;
  for (; j + 3 * stride < nv; j += 4 * stride) {
    const uint4 a = fv[j], b = fv[j + stride], c = fv[j + 2 * stride], e = fv[j + 3 * stride];
    tv[j] = a;
    tv[j + stride] = b;
    tv[j + 2 * stride] = c;
    tv[j + 3 * stride] = e;
  }
  for (; j < nv; j += stride) tv[j] = fv[j];
  const uint32_t done = head + 4 * nv;
  if (first < len - done) to[done + first] = from[done + first];
}

// An update of the lists, new list = (A \ D) u I per touched vertex, in four
// kernels. I and D are sorted and hold at most kMaxVertexChanges entries each;
// every key has a single final operation, so I and D are disjoint.
//
//   k_apply_plan    a lane per vertex: room in the scratch for its merged list and
//                   its pieces of kApplySeg entries, one counter add per wave
//   k_apply_rank    a wave per vertex: where its changes fall in the old list, its
//                   new degree and, when it outgrows its slot, a new one; writes
//                   the new inserts to their places
//   k_apply_merge   a wave per piece of the old lists: copies it, shifted by the
//                   changes before it
//   k_apply_commit  a wave per piece of the new lists: back into the slots of the
//                   lists that stay in place; a lane sets the vertex's record
//
// The lists are long and their changes few (500,000 vertices, 8 M edges, batches
// of 32,768 records: 31,000 lists of 1,100 entries in the mean, two changes each),
// so the pieces nearly all are plain copies; what counts is that they are many and
// alike, and that no counter is added to once per vertex. With a wave per list (a
// block or the grid for long ones), changes searched for every entry and a
// counter add per list, merge and commit of such a batch took 870 us.

// Deals out the lanes' lists in pieces: a lane's list `id` has ns of them, queued
// as (id, piece | tag); one counter add for the wave. Returns where the lane's
// first one went. All lanes must be active.
__device__ __forceinline__ uint32_t deal_pieces(uint2 *q, uint32_t *count, uint32_t id, uint32_t ns, uint32_t tag) {
  uint32_t all;
  const uint32_t before = wave_excl_sum(ns, &all);
  uint32_t at = 0;
  if (all && lane_id() == 0) at = atomicAdd(count, all);
  at = bcast(at) + before;
  for (uint32_t k = 0; k < ns; k++) q[at + k] = uint2{id, k | tag};
  return at;
}

// The number of p[0, n) below x, for the whole wave; p ascends.
__device__ __forceinline__ uint32_t wave_count_below(const uint32_t *p, uint32_t n, uint32_t x) {
  if (n <= 64) return (uint32_t)__popcll(ballot(lane_id() < n && p[min(lane_id(), n - 1)] < x));
  return lower_bound(p, n, x);
}

constexpr uint32_t kPlanBlock = 512;
template <bool ONE>
__device__ __forceinline__ void plan_lists(DevGraph g, BatchDev b, unsigned long long scratch_cap, ApplyCtl *actl) {
  __shared__ unsigned long long s_len[kPlanBlock / 64 + 1];
  __shared__ uint32_t s_segs[kPlanBlock / 64 + 1], s_most;
  if (threadIdx.x == 0) s_most = 0;
  for (uint32_t t0 = blockIdx.x * kPlanBlock; t0 < b.ntouched; t0 += gridDim.x * kPlanBlock) {
    const uint32_t t = t0 + threadIdx.x;
    uint32_t len = 0;  // of the merged list, at most
    if (t < b.ntouched) len = g.deg[b.tv[t]] + b.ioff[t + 1] - b.ioff[t];
    const uint32_t ns = t < b.ntouched ? max(1u, (len + kApplySeg - 1) / kApplySeg) : 0u;
    // (the sum of a block's lists may pass 32 bits)
    const unsigned long long so = block_take((unsigned long long)len, &actl->scratch_used, s_len);
    const uint32_t at = block_take(ns, &actl->nsegs, s_segs);
    atomicMax(&s_most, len);
    if (t < b.ntouched) {
      b.soff[t] = so;
      for (uint32_t k = 0; k < ns; k++) b.segs[at + k] = uint2{t, k};
    }
    // sized by the host so that this cannot happen
    if (so + len > scratch_cap) atomicAdd(&actl->merge_overflow, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_most > ld_relaxed(&actl->max_deg)) atomicMax(&actl->max_deg, s_most);
}
__global__ __launch_bounds__(kPlanBlock) void k_apply_plan(DevGraph g, BatchDev b, unsigned long long scratch_cap, ApplyCtl *actl) {
  plan_lists<false>(g, b, scratch_cap, actl);
}

// A slot for t's merged list of nd entries: its own, a new one from the pool's
// bump pointer, or none.
__device__ __forceinline__ uint32_t take_slot(const DevGraph &g, const BatchDev &b, uint32_t t, uint32_t x, uint32_t nd,
                                              unsigned long long pool_cap, ApplyCtl *actl, uint32_t fits,
                                              uint32_t moves) {
  if (nd <= g.cap[x]) {
    b.dst[t] = g.start[x];
    return fits;
  }
  const uint32_t newcap = nd + nd / 4 + 8;
  const unsigned long long base = atomicAdd(&actl->pool_used, (unsigned long long)newcap);
  if (base + newcap > pool_cap) {
    atomicAdd(&actl->overflow, 1u);
    return kNoRoom;
  }
  atomicAdd(&actl->relocated, 1u);
  b.dst[t] = (uint32_t)base;
  return moves;
}

template <bool ONE, uint32_t WAVES, uint32_t CHANGES>
__device__ __forceinline__ void rank_changes(DevGraph g, BatchDev b, uint32_t *scratch, unsigned long long pool_cap, ApplyCtl *actl) {
  __shared__ uint32_t s_rd[WAVES][CHANGES];
  if (ctl_word<ONE>(actl->merge_overflow)) return;
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  uint32_t *rd = s_rd[wv];
  for (uint32_t t = blockIdx.x * WAVES + wv; t < b.ntouched; t += gridDim.x * WAVES) {
    const uint32_t x = b.tv[t];
    const uint32_t *A = g.pool + g.start[x];
    const uint32_t na = g.deg[x];
    const uint32_t i0 = b.ioff[t], ni = b.ioff[t + 1] - i0;
    const uint32_t d0 = b.doff[t], nd = b.doff[t + 1] - d0;
    // changes 0 .. ni-1 are the inserts, the rest the deletes
    uint32_t nnew = 0, nhit = 0, key = 0, r = 0;
    bool fresh = false;
    wave_sync();  // the previous vertex's positions are no longer read
    for (uint32_t c = 0; c < ni + nd; c += 64) {
      const uint32_t j = c + lane;
      const bool ins = j < ni, del = !ins && j < ni + nd;
      key = ins ? b.ins[i0 + j] : del ? b.del[d0 + j - ni] : 0u;
      if (ni + nd <= 2) {
        // the whole wave searches for the one or two keys
        uint32_t r0, r1, loads = 0;
        bounds2(A, na, __builtin_amdgcn_readlane(key, 0), __builtin_amdgcn_readlane(key, 1), r0, r1, loads);
        r = lane == 0 ? r0 : r1;
      } else if (ins || del) {
        r = lower_bound(A, na, key);
      }
      const bool there = (ins || del) && r < na && A[r] == key;
      fresh = ins && !there;
      const uint64_t mi = ballot(fresh), md = ballot(del && there);
      if (fresh) b.ri[i0 + nnew + mbcnt(mi)] = r;
      if (del && there) {
        const uint32_t k = nhit + mbcnt(md);
        b.rd[d0 + k] = r;
        rd[k] = r;
      }
      nnew += (uint32_t)__popcll(mi);
      nhit += (uint32_t)__popcll(md);
    }
    wave_sync();
    const uint32_t ndeg = na - nhit + nnew;
    uint32_t state = 0, dst = 0;
    if (lane == 0) {
      state = take_slot(g, b, t, x, ndeg, pool_cap, actl, kInPlace, kDirect);
      if (state == kDirect) dst = b.dst[t];
      b.ndeg[t] = ndeg;
      b.nnew[t] = nnew;
      b.state[t] = state;
    }
    state = bcast(state);
    dst = bcast(dst);
    // the new inserts to their places, now that all deletes are known
    uint32_t *out = state == kDirect ? g.pool + dst : scratch + b.soff[t];
    for (uint32_t c = 0, seen = 0; c < ni; c += 64) {
      if (ni + nd > 64) {
        const uint32_t j = c + lane;
        key = j < ni ? b.ins[i0 + j] : 0u;
        r = j < ni ? lower_bound(A, na, key) : 0u;
        fresh = j < ni && !(r < na && A[r] == key);
      }
      const uint64_t m = ballot(fresh);
      if (fresh) out[r - lower_bound(rd, nhit, r) + seen + mbcnt(m)] = key;
      seen += (uint32_t)__popcll(m);
    }
  }
}
__global__ __launch_bounds__(kApplyWaves * 64) void k_apply_rank(DevGraph g, BatchDev b, uint32_t *scratch, unsigned long long pool_cap, ApplyCtl *actl) {
  rank_changes<false, kApplyWaves, kMaxVertexChanges>(g, b, scratch, pool_cap, actl);
}

template <bool ONE>
__device__ __forceinline__ void merge_lists(DevGraph g, BatchDev b, uint32_t *scratch, const ApplyCtl *actl) {
  if (ctl_word<ONE>(actl->merge_overflow)) return;
  const uint32_t lane = lane_id(), nsegs = ctl_word<ONE>(actl->nsegs);
  for (uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < nsegs; i += (gridDim.x * blockDim.x) >> 6) {
    const uint2 sg = b.segs[i];
    const uint32_t t = bcast(sg.x), s0 = bcast(sg.y) * kApplySeg;
    const uint32_t x = b.tv[t];
    const uint32_t na = g.deg[x];
    if (s0 >= na) continue;
    const uint32_t s1 = min(s0 + kApplySeg, na);
    const uint32_t nnew = b.nnew[t], nhit = na + nnew - b.ndeg[t];
    const uint32_t *ri = b.ri + b.ioff[t], *rd = b.rd + b.doff[t];
    const uint32_t *A = g.pool + g.start[x];
    uint32_t *out = b.state[t] == kDirect ? g.pool + b.dst[t] : scratch + b.soff[t];
    // new inserts at or before the piece's first and last entry, deletes before
    // its first entry and its end
    const uint32_t q0 = wave_count_below(ri, nnew, s0 + 1), q1 = wave_count_below(ri, nnew, s1);
    const uint32_t p0 = wave_count_below(rd, nhit, s0), p1 = wave_count_below(rd, nhit, s1);
    if (q0 == q1 && p0 == p1) {
      copy_range(A + s0, out + s0 + q0 - p0, lane, 64, s1 - s0);
      continue;
    }
    for (uint32_t j = s0 + lane; j < s1; j += 64) {
      const uint32_t a = A[j];
      const uint32_t p = p0 + lower_bound(rd + p0, p1 - p0, j);
      if (p < p1 && rd[p] == j) continue;
      const uint32_t q = q0 + lower_bound(ri + q0, q1 - q0, j + 1);
      out[j - p + q] = a;
    }
  }
}
__global__ __launch_bounds__(256) void k_apply_merge(DevGraph g, BatchDev b, uint32_t *scratch, const ApplyCtl *actl) {
  merge_lists<false>(g, b, scratch, actl);
}

// With `again`, the commits that found no room the first time.
template <bool ONE>
__device__ __forceinline__ void commit_lists(DevGraph g, BatchDev b, const uint32_t *scratch, const ApplyCtl *actl, DirtyArgs d, int again) {
  if (ctl_word<ONE>(actl->merge_overflow)) return;
  const uint32_t lane = lane_id(), nsegs = ctl_word<ONE>(actl->nsegs);
  for (uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < nsegs; i += (gridDim.x * blockDim.x) >> 6) {
    const uint2 sg = b.segs[i];
    const uint32_t t = bcast(sg.x), s0 = bcast(sg.y) * kApplySeg;
    const uint32_t state = b.state[t], nd = b.ndeg[t], dst = b.dst[t];
    if (again ? state != kRetried : state == kNoRoom) continue;
    if (state != kDirect && s0 < nd)
      copy_range(scratch + b.soff[t] + s0, g.pool + dst + s0, lane, 64, min(kApplySeg, nd - s0));
    if (s0 == 0 && lane == 0) {
      const uint32_t x = b.tv[t];
      if (g.start[x] != dst) {
        g.start[x] = dst;
        g.cap[x] = nd + nd / 4 + 8;
      }
      g.deg[x] = nd;
      mark_dirty(d, x);
    }
  }
}
__global__ __launch_bounds__(256) void k_apply_commit(DevGraph g, BatchDev b, const uint32_t *scratch, const ApplyCtl *actl, DirtyArgs d, int again) {
  commit_lists<false>(g, b, scratch, actl, d, again);
}

// After the pool has grown: slots for the merged lists that found none.
__global__ __launch_bounds__(256) void k_apply_slots(DevGraph g, BatchDev b, unsigned long long pool_cap,
                                                     ApplyCtl *actl) {
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < b.ntouched; t += gridDim.x * blockDim.x) {
    const uint32_t was = b.state[t];
    uint32_t state = kDone;
    if (was == kNoRoom) state = take_slot(g, b, t, b.tv[t], b.ndeg[t], pool_cap, actl, kRetried, kRetried);
    b.state[t] = state;
  }
}

// The start of an update: its status from another graph copy's, its counters
// cleared.
template <bool ONE>
__device__ __forceinline__ void begin_update(ApplyCtl *actl, const ApplyCtl *from, uint32_t *bctl) {
  const auto put = [](auto &w, auto x) {
    if (ONE) __hip_atomic_store(&w, (std::remove_reference_t<decltype(w)>)x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else w = x;
  };
  if (from) {
    actl->pool_used = from->pool_used;
    actl->max_deg = from->max_deg;
  }
  put(actl->scratch_used, 0);
  put(actl->overflow, 0);
  put(actl->merge_overflow, 0);
  put(actl->relocated, 0);
  put(actl->relabeled, 0);
  put(actl->ndirty, 0);
  put(actl->filter_entries, 0);
  put(actl->filter_bits, 0);
  put(actl->nsegs, 0);
  put(actl->nrelabel_segs, 0);
  put(actl->chunks_dropped, 0);
  for (int i = 0; i < 4; i++) {
    put(actl->sync_queued[i], 0);
    put(bctl[i], 0);
  }
}

__global__ __launch_bounds__(256) void k_update_begin(ApplyCtl *actl, const ApplyCtl *from, uint32_t *bctl,
                                                       SmallCopy up) {
  small_copy(up);
  if (threadIdx.x == 0) begin_update<false>(actl, from, bctl);
}

__global__ __launch_bounds__(256) void k_round_begin(ApplyCtl *actl, SmallCopy up) {
  small_copy(up);
  if (threadIdx.x != 0) return;
  actl->scratch_used = 0;
  actl->nsegs = 0;
}

// The relabels, a lane each: set the label; when it changed, mark the vertex
// dirty and deal out its (post-update) list in pieces for k_relabel_marks, with
// its old label.
template <bool ONE>
__device__ __forceinline__ void relabel(DevGraph g, BatchDev b, DirtyArgs d) {
  if (held_up<ONE>(d.actl)) return;
  for (uint32_t r0 = (blockIdx.x * blockDim.x + threadIdx.x) & ~63u; r0 < b.nrelabel; r0 += gridDim.x * blockDim.x) {
    const uint32_t r = r0 + lane_id();
    uint32_t x = 0, old = 0, L = 0;
    bool changed = false;
    if (r < b.nrelabel) {
      x = b.rl_v[r];
      L = b.rl_l[r];
      old = g.lab[x];
      changed = old != L;
    }
    uint32_t ns = 0;
    if (changed) {
      g.lab[x] = (uint8_t)L;
      mark_dirty(d, x);
      ns = max(1u, (g.deg[x] + kApplySeg - 1) / kApplySeg);
    }
    const uint32_t n = (uint32_t)__popcll(ballot(changed));
    if (n && lane_id() == 0) atomicAdd(&d.actl->relabeled, n);
    deal_pieces(b.segs, &d.actl->nrelabel_segs, x, ns, old << 24);
  }
}
__global__ __launch_bounds__(256) void k_relabel(DevGraph g, BatchDev b, DirtyArgs d) {
  relabel<false>(g, b, d);
}

// A wave per piece of a relabelled vertex's list: its neighbours' neighbour-label
// counts changed, so they are marked dirty; with the first piece the vertex's bits
// go from every bitmap of its old label.
template <bool ONE>
__device__ __forceinline__ void relabel_marks(DevGraph g, BatchDev b, FilterTables ft, DirtyArgs d) {
  const uint32_t lane = lane_id(), nsegs = ctl_word<ONE>(d.actl->nrelabel_segs);
  for (uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < nsegs; i += (gridDim.x * blockDim.x) >> 6) {
    const uint2 sg = b.segs[i];
    const uint32_t x = bcast(sg.x), s0 = bcast(sg.y & 0xFFFFFFu) * kApplySeg, old = bcast(sg.y >> 24);
    if (s0 == 0 && old != kNoLabel) {
      const uint64_t clr = ~(1ull << (x & 63));
      for (uint32_t s = ft.sig_lo[old] + lane; s < ft.sig_hi[old]; s += 64)
        atomicAnd((unsigned long long *)&ft.bm[(size_t)s * ft.words + (x >> 6)], (unsigned long long)clr);
    }
    const uint32_t *A = g.pool + g.start[x];
    const uint32_t s1 = min(s0 + kApplySeg, g.deg[x]);
    constexpr uint32_t kU = 4;  // entries a lane in flight
    for (uint32_t j0 = s0; j0 < s1; j0 += 64 * kU) {
      uint32_t w[kU];
#pragma unroll
      for (uint32_t u = 0; u < kU; u++) w[u] = A[min(j0 + u * 64 + lane, s1 - 1)];
#pragma unroll
      for (uint32_t u = 0; u < kU; u++) mark_dirty(d, w[u]);
    }
  }
}
__global__ __launch_bounds__(256) void k_relabel_marks(DevGraph g, BatchDev b, FilterTables ft, DirtyArgs d) {
  relabel_marks<false>(g, b, ft, d);
}

// ----------------------------------------------------------------- filter

__device__ __forceinline__ bool sig_pass(const SigReq &r, uint32_t deg, const uint64_t *c) {
  return deg >= r.deg && ge_bytes(c[0], r.nlc[0]) && ge_bytes(c[1], r.nlc[1]) &&
         ge_bytes(c[2], r.nlc[2]) && ge_bytes(c[3], r.nlc[3]);
}

// Whole-graph pass, one wave per 64-vertex group: the group's adjacency lists
// are scanned as one logical array (lanes balanced across vertices), label
// counts accumulate in LDS, then every bitmap word of the group is written
// with one ballot.
__global__ __launch_bounds__(256) void k_filter_full(DevGraph g, FilterTables ft) {
  __shared__ uint32_t s_cnt[4][64][kMaxRel + 1];
  __shared__ uint32_t s_pre[4][65];
  __shared__ uint32_t s_st[4][64];
  __shared__ uint8_t s_lmap[256];
  for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) s_lmap[i] = ft.lmap[i];
  __syncthreads();
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  const uint32_t ngroups = (g.n + 63) / 64;
  for (uint32_t grp = blockIdx.x * 4 + wv; grp < ngroups; grp += gridDim.x * 4) {
    const uint32_t v = grp * 64 + lane;
    const bool valid = v < g.n;
    const uint32_t L = valid ? g.lab[v] : kNoLabel;
    const bool has = L != kNoLabel && ft.sig_lo[L] < ft.sig_hi[L];
    const uint32_t dv = valid ? g.deg[v] : 0;
    const uint32_t d = has ? dv : 0;
    s_st[wv][lane] = valid ? g.start[v] : 0;
    for (int l = 0; l <= kMaxRel; l++) s_cnt[wv][lane][l] = 0;
    // inclusive scan of d
    uint32_t incl = d;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off);
      if (lane >= (uint32_t)off) incl += y;
    }
    s_pre[wv][lane + 1] = incl;
    if (lane == 0) s_pre[wv][0] = 0;
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    wave_sync();
    for (uint32_t e = lane; e < total; e += 64) {
      // owner: last k with s_pre[k] <= e
      uint32_t lo = 0, n = 64;
      while (n > 1) {
        const uint32_t half = n >> 1;
        lo = (s_pre[wv][lo + half] <= e) ? lo + half : lo;
        n -= half;
      }
      const uint32_t w = g.pool[s_st[wv][lo] + (e - s_pre[wv][lo])];
      const uint32_t li = s_lmap[g.lab[w]];
      if (li != 0xFF) atomicAdd(&s_cnt[wv][lo][li], 1u);
    }
    wave_sync();
    uint64_t c[4] = {0, 0, 0, 0};
    for (int l = 0; l < kMaxRel; l++) {
      const uint64_t x = s_cnt[wv][lane][l] < 15 ? s_cnt[wv][lane][l] : 15;
      c[l >> 3] |= x << ((l & 7) * 8);
    }
    for (uint32_t s = 0; s < ft.nsig; s++) {
      const SigReq r = ft.sigs[s];
      const bool pass = has && L == r.label && sig_pass(r, dv, c);
      const uint64_t word = ballot(pass);
      if (lane == 0) ft.bm[(size_t)s * ft.words + grp] = word;
    }
    wave_sync();
  }
}

// Sets v's bit in its bitmap word w, which read `cur` before: only this lane
// changes this bit in this kernel.
__device__ __forceinline__ void set_bit_from(uint64_t *w, uint64_t cur, uint32_t v, bool on) {
  const uint64_t bit = 1ull << (v & 63);
  if (((cur & bit) != 0) == on) return;
  if (on) atomicOr((unsigned long long *)w, (unsigned long long)bit);
  else atomicAnd((unsigned long long *)w, (unsigned long long)~bit);
}

// The dirty vertices, up to 64 to a wave, but those with a label-sorted copy, which
// were filtered from its bucket sizes (filter_buckets). The lists of a wave's vertices are read as one array, as many lanes
// to a list as it has entries, and so are their (vertex, signature) pairs, four
// entries and two pairs a lane in flight. Bound by the scattered label and bitmap
// reads. With a lane per vertex, its list and its signatures one after the other,
// 25 us for 4,900 dirty vertices of 100,000 (the longest chain of a wave).
template <bool ONE, uint32_t WAVES>
__device__ __forceinline__ void filter_light(DevGraph g, FilterTables ft, DirtyArgs d) {
  // counts of the wave's vertices: a byte per label (at most kLabelSorted), 32 of them
  // (a 64-bit word of padding keeps the vertices apart in the banks)
  __shared__ uint64_t s_cnt[WAVES][64][kMaxRel / 8 + 1];
  __shared__ uint32_t s_pre[WAVES][65], s_from[WAVES][64], s_v[WAVES][64], s_deg[WAVES][64];
  __shared__ unsigned long long s_sum[2];
  __shared__ uint8_t s_lmap[256];
  for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) s_lmap[i] = ft.lmap[i];
  __syncthreads();
  if (held_up<ONE>(d.actl)) return;
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  const uint32_t nd = min(ctl_word<ONE>(d.actl->ndirty), d.list_cap);
  uint32_t *pre = s_pre[wv], *from = s_from[wv];
  unsigned long long entries = 0;  // list entries of the vertices this lane re-filters
  uint32_t bits = 0;               // candidate bits they receive (one per signature of the label)
  if (lane == 0) pre[0] = 0;
  if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
  __syncthreads();
  // fewer vertices a wave where there are waves enough: shorter chains
  uint32_t per = 64;
  while (per > 8 && nd <= per / 2 * gridDim.x * WAVES) per >>= 1;
  for (uint32_t i0 = (blockIdx.x * WAVES + wv) * per; i0 < nd; i0 += gridDim.x * WAVES * per) {
    const uint32_t i = i0 + lane;
    uint32_t v = 0, L = kNoLabel, dv = 0, lo = 0, ns = 0;
    if (lane < per && i < nd) {
      v = d.list[i];
      L = g.lab[v];
    }
    if (L != kNoLabel) {
      lo = ft.sig_lo[L];
      ns = ft.sig_hi[L] - lo;
    }
    if (ns) {
      dv = g.deg[v];
      entries += dv;
      bits += ns;
    }
    if (dv > kLabelSorted) dv = ns = 0;
    wave_sync();  // the previous vertices' arrays are no longer read
    pre[lane + 1] = wave_incl_sum(dv);
    from[lane] = ns ? g.start[v] : 0;
    s_v[wv][lane] = v;
    s_deg[wv][lane] = dv;
    for (int k = 0; k < kMaxRel / 8; k++) s_cnt[wv][lane][k] = 0;
    wave_sync();
    const uint32_t total = pre[64];
    constexpr int kU = 4;  // entries a lane in flight
    for (uint32_t e = 0; e < total; e += 64 * kU) {
      uint32_t k[kU], o[kU], w[kU];
#pragma unroll
      for (int u = 0; u < kU; u++) k[u] = min(e + u * 64 + lane, total - 1);
      ranges_of(pre, k, o);
#pragma unroll
      for (int u = 0; u < kU; u++) w[u] = g.pool[from[o[u]] + (k[u] - pre[o[u]])];
#pragma unroll
      for (int u = 0; u < kU; u++) w[u] = s_lmap[g.lab[w[u]]];
#pragma unroll
      for (int u = 0; u < kU; u++)
        if (e + u * 64 + lane < total && w[u] != 0xFF)
          atomicAdd(reinterpret_cast<uint32_t *>(s_cnt[wv][o[u]]) + (w[u] >> 2), 1u << (w[u] & 3) * 8);
    }
    // the pairs take the lists' place in the arrays
    wave_sync();
    pre[lane + 1] = wave_incl_sum(ns);
    from[lane] = lo;
    wave_sync();
    const uint32_t pairs = pre[64];
    for (uint32_t e = 0; e < pairs; e += 128) {
      uint32_t k[2], o[2];
      uint64_t *word[2], cur[2];
      bool pass[2];
#pragma unroll
      for (int u = 0; u < 2; u++) k[u] = min(e + u * 64 + lane, pairs - 1);
      ranges_of(pre, k, o);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const uint32_t s = from[o[u]] + (k[u] - pre[o[u]]);
        word[u] = &ft.bm[(size_t)s * ft.words + (s_v[wv][o[u]] >> 6)];
        cur[u] = ld_relaxed(word[u]);
        pass[u] = sig_pass(ft.sigs[s], s_deg[wv][o[u]], s_cnt[wv][o[u]]);
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
        if (e + u * 64 + lane < pairs) set_bit_from(word[u], cur[u], s_v[wv][o[u]], pass[u]);
    }
  }
  if (entries) atomicAdd(&s_sum[0], entries);
  if (bits) atomicAdd(&s_sum[1], (unsigned long long)bits);
  __syncthreads();
  if (threadIdx.x == 0 && s_sum[0]) atomicAdd(&d.actl->filter_entries, s_sum[0]);
  if (threadIdx.x == 1 && s_sum[1]) atomicAdd(&d.actl->filter_bits, (uint32_t)s_sum[1]);
}
__global__ __launch_bounds__(256) void k_filter_light(DevGraph g, FilterTables ft, DirtyArgs d) {
  filter_light<false, 4>(g, ft, d);
}

// ---------------------------------------------------- label-sorted copies

// Lanes of the wave whose bucket equals this lane's (among valid lanes): one
// ballot per bit of the bucket index, so a chunk with many distinct buckets
// costs the same as one with a single bucket.
__device__ __forceinline__ uint64_t bucket_peers(uint32_t b, bool valid, uint32_t bits) {
  uint64_t m = ballot(valid);
  for (uint32_t i = 0; i < bits; i++) {
    const bool set = (b >> i) & 1;
    const uint64_t bi = ballot(valid && set);
    m &= set ? bi : ~bi;
  }
  return m;
}

__device__ __forceinline__ uint32_t bucket_of(const DevGraph &g, const uint8_t *s_lmap, uint32_t x) {
  const uint32_t b = s_lmap[g.lab[x]];
  return b == 0xFF ? g.nbuckets - 1 : b;
}

// Adds the bucket histogram of A[lo, hi) to cnt (per-wave LDS counters; the
// lowest lane of each peer group adds the group's size).
__device__ __forceinline__ void bucket_count(const DevGraph &g, const uint8_t *s_lmap, const uint32_t *A,
                                             uint32_t lo, uint32_t hi, uint32_t bits, uint32_t *cnt,
                                             uint8_t *bk_out) {
  const uint32_t lane = lane_id();
  // four chunks at a time: their entries, then their label reads, are all in
  // flight before the first chunk's counts are taken
  constexpr uint32_t kU = 4;
  for (uint32_t c0 = lo; c0 < hi; c0 += 64 * kU) {
    uint32_t x[kU], b[kU];
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t j = c0 + u * 64 + lane;
      x[u] = j < hi ? A[j] : 0u;
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t j = c0 + u * 64 + lane;
      b[u] = j < hi ? bucket_of(g, s_lmap, x[u]) : 0u;
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t j = c0 + u * 64 + lane;
      const bool valid = j < hi;
      if (valid && bk_out) bk_out[j] = (uint8_t)b[u];
      const uint64_t pm = bucket_peers(b[u], valid, bits);
      if (valid && mbcnt(pm) == 0) cnt[b[u]] += (uint32_t)__popcll(pm);
      wave_sync();
    }
  }
}

// Scatters A[lo, hi) into out by bucket, cnt[b] holding the next position of
// bucket b; id order is kept inside each bucket. Four chunks' entries and
// buckets are loaded before the first chunk is placed.
__device__ __forceinline__ void bucket_scatter(const DevGraph &g, const uint8_t *s_lmap, const uint32_t *A,
                                               uint32_t lo, uint32_t hi, uint32_t bits, uint32_t *cnt,
                                               uint32_t *out, const uint8_t *bk_in) {
  const uint32_t lane = lane_id();
  constexpr uint32_t kU = 4;
  for (uint32_t c0 = lo; c0 < hi; c0 += 64 * kU) {
    uint32_t x[kU], b[kU];
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t j = c0 + u * 64 + lane;
      x[u] = j < hi ? A[j] : 0u;
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t j = c0 + u * 64 + lane;
      b[u] = j < hi ? (bk_in ? (uint32_t)bk_in[j] : bucket_of(g, s_lmap, x[u])) : 0u;
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const bool valid = c0 + u * 64 + lane < hi;
      const uint64_t pm = bucket_peers(b[u], valid, bits);
      const uint32_t rank = mbcnt(pm);
      const uint32_t base = valid ? cnt[b[u]] : 0u;
      wave_sync();
      if (valid) {
        out[base + rank] = x[u];
        if (rank == 0) cnt[b[u]] = base + (uint32_t)__popcll(pm);
      }
      wave_sync();
    }
  }
}


// The candidate bits of a dirty vertex with a label-sorted copy: its neighbour
// count of query label li is the size of bucket li, so no list is read again. One
// wave; `size` is the lane's bucket's, of nb (the last one holds the other labels);
// pack is the wave's.
__device__ __forceinline__ void filter_buckets(const DevGraph &g, const FilterTables &ft, uint32_t v, uint32_t d,
                                               uint32_t size, uint32_t nb, uint64_t *pack) {
  const uint32_t lane = lane_id(), L = g.lab[v];
  if (L == kNoLabel) return;
  if (lane < kMaxRel) reinterpret_cast<uint8_t *>(pack)[lane] = (uint8_t)(lane + 1 < nb ? min(size, 15u) : 0u);
  wave_sync();
  for (uint32_t s = ft.sig_lo[L] + lane; s < ft.sig_hi[L]; s += 64) {
    uint64_t *word = &ft.bm[(size_t)s * ft.words + (v >> 6)];
    const uint64_t cur = ld_relaxed(word);
    set_bit_from(word, cur, v, sig_pass(ft.sigs[s], d, pack));
  }
  wave_sync();
}

// The label-sorted copy of v (degree d, at most 64 U) by one wave, which holds the
// whole list in registers: each entry's place among its bucket's, the buckets'
// starts, then the entries to their places (in id order inside a bucket). Returns
// the size of the lane's bucket. Bound by the chain of reads (list, labels) and the
// ballots per entry: with the list read and its buckets matched twice 62 us for the
// 12,000 such lists of a 32,768-record batch.
template <uint32_t U>
__device__ __forceinline__ uint32_t build_one(const DevGraph &g, const uint8_t *s_lmap, uint32_t v, uint32_t d,
                                              uint32_t nb, uint32_t bits, uint32_t *cnt) {
  const uint32_t lane = lane_id(), st = g.start[v];
  const uint32_t *A = g.pool + st;
  uint32_t *row = g.loff + (size_t)v * (nb + 1);
  if (lane < nb) cnt[lane] = 0;
  uint32_t x[U], b[U];
#pragma unroll
  for (uint32_t u = 0; u < U; u++) x[u] = u * 64 < d ? A[min(u * 64 + lane, d - 1)] : 0u;
#pragma unroll
  for (uint32_t u = 0; u < U; u++) b[u] = u * 64 < d ? bucket_of(g, s_lmap, x[u]) : 0u;
  wave_sync();
#pragma unroll
  for (uint32_t u = 0; u < U; u++) {
    if (u * 64 >= d) break;
    const bool valid = u * 64 + lane < d;
    const uint64_t pm = bucket_peers(b[u], valid, bits);
    const uint32_t rank = mbcnt(pm), before = cnt[b[u]];
    wave_sync();
    if (valid && rank == 0) cnt[b[u]] = before + (uint32_t)__popcll(pm);
    wave_sync();
    b[u] |= (before + rank) << 8;
  }
  // bucket starts: an exclusive scan with a lane per bucket (nb <= kMaxRel + 1 < 64)
  uint32_t total;
  const uint32_t c = lane < nb ? cnt[lane] : 0u;
  const uint32_t first = wave_excl_sum(c, &total);
  if (lane < nb) row[lane] = cnt[lane] = first;
  if (lane == 0) row[nb] = total;
  wave_sync();
  uint32_t *out = g.lpool + st;
#pragma unroll
  for (uint32_t u = 0; u < U; u++)
    if (u * 64 + lane < d) out[cnt[b[u] & 0xFF] + (b[u] >> 8)] = x[u];
  wave_sync();
  return c;
}

// Entries per piece of a long list: kBuildSeg, more where the list would have over
// kBuildPieces pieces; a multiple of 64.
__device__ __forceinline__ uint32_t build_piece(uint32_t d) {
  return max(kBuildSeg, ((d + kBuildPieces - 1) / kBuildPieces + 63) & ~63u);
}

// The listed vertices (or all), four a lane: those of degree in (kLabelSorted,
// kBuildSeg] to hs.mid, longer ones to hs.big and in pieces to hs.pieces.
// Vertices whose label no query uses are skipped (never read, see
// k_dirty_compact); a full build leaves their groups empty.
template <bool ONE, uint32_t WAVES>
__device__ __forceinline__ void pick_builds(DevGraph g, const uint32_t *list, const uint32_t *count, SortedBuild hs) {
  __shared__ uint32_t s_sum[WAVES + 1];
  const uint32_t nb = g.nbuckets;
  if (hs.actl && held_up<ONE>(hs.actl)) return;
  const uint32_t total = list ? min(ctl_word<ONE>(*count), g.n) : g.n;
  constexpr uint32_t kU = 4;
  for (uint32_t base = blockIdx.x * (WAVES * 64) * kU; base < total; base += gridDim.x * (WAVES * 64) * kU) {
    uint32_t v[kU], d[kU], l[kU], nmid = 0, nbig = 0, npieces = 0;
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      const uint32_t t = min(base + u * (WAVES * 64) + threadIdx.x, total - 1);
      v[u] = list ? list[t] : t;
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      d[u] = base + u * (WAVES * 64) + threadIdx.x < total ? g.deg[v[u]] : 0u;
      l[u] = g.lab[v[u]];
    }
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      if (d[u] <= kLabelSorted) continue;
      if (l[u] == kNoLabel) {
        if (!list)
          for (uint32_t k = 0; k <= nb; k++) g.loff[(size_t)v[u] * (nb + 1) + k] = 0;
        d[u] = 0;
      } else if (d[u] <= kBuildSeg) {
        nmid++;
      } else {
        const uint32_t sz = build_piece(d[u]);
        nbig++;
        npieces += (d[u] + sz - 1) / sz;
      }
    }
    uint32_t at = block_take(nmid, &hs.ctl[0], s_sum);
#pragma unroll
    for (uint32_t u = 0; u < kU; u++)
      if (d[u] > kLabelSorted && d[u] <= kBuildSeg) hs.mid[at++] = v[u];
    if (!__syncthreads_or(nbig != 0)) continue;
    at = block_take(nbig, &hs.ctl[1], s_sum);
    uint32_t first = block_take(npieces, &hs.ctl[2], s_sum);
#pragma unroll
    for (uint32_t u = 0; u < kU; u++) {
      if (d[u] <= kBuildSeg) continue;
      const uint32_t sz = build_piece(d[u]), np = (d[u] + sz - 1) / sz;
      hs.big[at++] = uint2{v[u], first};
      for (uint32_t k = 0; k < np; k++) hs.pieces[first + k] = uint2{v[u], k};
      first += np;
    }
  }
}
__global__ __launch_bounds__(256) void k_lbuild_pick(DevGraph g, const uint32_t *list, const uint32_t *count, SortedBuild hs) {
  pick_builds<false, 4>(g, list, count, hs);
}

// A wave per piece of a long list: its bucket counts; then a wave per short list:
// its label-sorted copy and, if asked, its vertex's candidate bits.
template <bool ONE, uint32_t WAVES>
__device__ __forceinline__ void sort_lists(DevGraph g, FilterTables ft, SortedBuild hs, bool filter) {
  __shared__ uint8_t s_lmap[256];
  __shared__ uint32_t s_cnt[WAVES][kMaxRel + 2];
  __shared__ uint64_t s_pack[WAVES][kMaxRel / 8];
  for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) s_lmap[i] = ft.lmap[i];
  __syncthreads();
  const uint32_t wv = bcast(threadIdx.x >> 6), lane = lane_id();
  const uint32_t nb = g.nbuckets;
  const uint32_t bits = 32u - (uint32_t)__builtin_clz(nb > 1 ? nb - 1 : 1u);
  const uint32_t npieces = ctl_word<ONE>(hs.ctl[2]), total = npieces + ctl_word<ONE>(hs.ctl[0]);
  uint32_t *cnt = s_cnt[wv];
  for (uint32_t t = blockIdx.x * WAVES + wv; t < total; t += gridDim.x * WAVES) {
    if (t >= npieces) {
      const uint32_t v = bcast(hs.mid[t - npieces]), d = bcast(g.deg[v]);
      const uint32_t size = d <= 256 ? build_one<4>(g, s_lmap, v, d, nb, bits, cnt)
                                     : build_one<kBuildSeg / 64>(g, s_lmap, v, d, nb, bits, cnt);
      if (filter) filter_buckets(g, ft, v, d, size, nb, s_pack[wv]);
      continue;
    }
    const uint2 pc = hs.pieces[t];
    const uint32_t v = bcast(pc.x), d = g.deg[v], sz = build_piece(d);
    const uint32_t lo = bcast(pc.y) * sz, hi = min(lo + sz, d);
    if (lane < nb) cnt[lane] = 0;
    wave_sync();
    bucket_count(g, s_lmap, g.pool + g.start[v], lo, hi, bits, cnt,
                 hs.bucket_bytes ? hs.bucket_bytes + g.start[v] : nullptr);
    if (lane < nb) hs.hist[(size_t)t * (kMaxRel + 2) + lane] = cnt[lane];
    wave_sync();
  }
}
__global__ __launch_bounds__(256) void k_lbuild(DevGraph g, FilterTables ft, SortedBuild hs, bool filter) {
  sort_lists<false, 4>(g, ft, hs, filter);
}

// A wave per long list, a lane per bucket (nb <= kMaxRel + 1 < 64): the buckets'
// starts, and each piece's start inside every bucket in place of its counts; if
// asked, its vertex's candidate bits.
__global__ __launch_bounds__(256) void k_lbuild_starts(DevGraph g, FilterTables ft, SortedBuild hs, bool filter) {
  __shared__ uint64_t s_pack[4][kMaxRel / 8];
  const uint32_t lane = lane_id(), nb = g.nbuckets, nbig = hs.ctl[1];
  for (uint32_t t = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; t < nbig; t += (gridDim.x * blockDim.x) >> 6) {
    const uint2 bg = hs.big[t];
    const uint32_t v = bcast(bg.x), d = g.deg[v], sz = build_piece(d), np = (d + sz - 1) / sz;
    uint32_t *hist = hs.hist + (size_t)bcast(bg.y) * (kMaxRel + 2) + lane;
    uint32_t sum = 0, total;
    if (lane < nb)
#pragma unroll 8
      for (uint32_t p = 0; p < np; p++) sum += hist[(size_t)p * (kMaxRel + 2)];
    uint32_t run = wave_excl_sum(sum, &total);
    uint32_t *row = g.loff + (size_t)v * (nb + 1);
    if (lane < nb) {
      row[lane] = run;
#pragma unroll 8
      for (uint32_t p = 0; p < np; p++) {
        const uint32_t c = hist[(size_t)p * (kMaxRel + 2)];
        hist[(size_t)p * (kMaxRel + 2)] = run;
        run += c;
      }
    }
    if (lane == 0) row[nb] = total;
    if (filter) filter_buckets(g, ft, v, d, sum, nb, s_pack[threadIdx.x >> 6]);
  }
}

// A wave per piece of a long list: its entries to their buckets, in id order.
__global__ __launch_bounds__(256) void k_lbuild_place(DevGraph g, const uint8_t *lmap, SortedBuild hs) {
  __shared__ uint8_t s_lmap[256];
  __shared__ uint32_t s_cnt[4][kMaxRel + 2];
  for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x) s_lmap[i] = lmap[i];
  __syncthreads();
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  const uint32_t nb = g.nbuckets;
  const uint32_t bits = 32u - (uint32_t)__builtin_clz(nb > 1 ? nb - 1 : 1u);
  const uint32_t npieces = hs.ctl[2];
  uint32_t *cnt = s_cnt[wv];
  for (uint32_t t = blockIdx.x * 4 + wv; t < npieces; t += gridDim.x * 4) {
    const uint2 pc = hs.pieces[t];
    const uint32_t v = bcast(pc.x), d = g.deg[v], sz = build_piece(d);
    const uint32_t lo = bcast(pc.y) * sz, hi = min(lo + sz, d);
    if (lane < nb) cnt[lane] = hs.hist[(size_t)t * (kMaxRel + 2) + lane];
    wave_sync();
    bucket_scatter(g, s_lmap, g.pool + g.start[v], lo, hi, bits, cnt, g.lpool + g.start[v],
                   hs.bucket_bytes ? hs.bucket_bytes + g.start[v] : nullptr);
    wave_sync();
  }
}

// A whole update by one block, its phases a block barrier apart instead of a launch: one
// record on lists of 30 entries takes it 18.5 us, and the call 81 where the ten kernels,
// most of whose time lies between them, made it 105. Lists of at most kBuildSeg entries
// (no pieces), at most kSmallChanges changes. It ends with the update's status in pinned
// host memory.
constexpr uint32_t kOneWaves = 8;
static_assert(kOneWaves * 64 == kPlanBlock && kOneWaves * 64 == kCompactBlock, "the phases' strides");
__global__ __launch_bounds__(kOneWaves * 64) void k_update_small(DevGraph g, BatchDev b, FilterTables ft, DirtyArgs d,
                                                                 SortedBuild hs, uint32_t *scratch,
                                                                 unsigned long long scratch_cap,
                                                                 unsigned long long pool_cap, bool sorted, SmallCopy up,
                                                                 uint32_t *status) {
  ApplyCtl *actl = d.actl;
  // a phase's stores and counter adds have been taken before the next begins
  const auto next = [] {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
  small_copy(up);
  if (threadIdx.x == 0) begin_update<true>(actl, nullptr, hs.ctl);
  next();
  plan_lists<true>(g, b, scratch_cap, actl);
  next();
  rank_changes<true, kOneWaves, kSmallChanges>(g, b, scratch, pool_cap, actl);
  next();
  merge_lists<true>(g, b, scratch, actl);
  next();
  commit_lists<true>(g, b, scratch, actl, d, 0);
  next();
  if (b.nrelabel) {
    relabel<true>(g, b, d);
    next();
    relabel_marks<true>(g, b, ft, d);
    next();
  }
  compact_dirty<true>(g, d);
  next();
  if (sorted) {
    pick_builds<true, kOneWaves>(g, d.list, &actl->ndirty, hs);
    next();
    sort_lists<true, kOneWaves>(g, ft, hs, true);
    next();
  }
  filter_light<true, kOneWaves>(g, ft, d);
  next();
  if (threadIdx.x < sizeof(ApplyCtl) / 4) status[threadIdx.x] = ld_relaxed(reinterpret_cast<uint32_t *>(actl) + threadIdx.x);
}

__global__ void k_build_reset(SortedBuild hs) {
  if (threadIdx.x < 4) hs.ctl[threadIdx.x] = 0;
}

// ------------------------------------------------------------------- seed

// Records of a wave: few where there are waves enough for all.
__host__ __device__ inline uint32_t seed_share(uint32_t records) { return records <= 8192 ? 16 : 64; }

// Which of the records `need` (bits) name an edge of the graph: d in N(s), the
// direction the DFS also tests. 16 lanes search a list, four lists at a time, so a
// list of 4,096 entries takes three reads one after the other instead of twelve.
__device__ __forceinline__ uint64_t edges_there(const DevGraph &g, uint64_t need, const uint32_t *rs,
                                                const uint32_t *rd) {
  const uint32_t j = lane_id() & 15, group = lane_id() >> 4;
  uint64_t there = 0;
  while (need) {
    uint32_t r[4];
    for (int k = 0; k < 4; k++) {
      r[k] = need ? (uint32_t)__builtin_ctzll(need) : 64u;
      need &= need - 1;  // (0 stays 0)
    }
    const uint32_t mine = group == 0 ? r[0] : group == 1 ? r[1] : group == 2 ? r[2] : r[3];
    const uint32_t s = mine < 64 ? rs[mine] : 0u, d = mine < 64 ? rd[mine] : 0u;
    const uint32_t *A = g.pool + g.start[s];
    uint32_t lo = 0, hi = mine < 64 ? g.deg[s] : 0u;  // d is in A[lo, hi), if at all
    while (ballot(hi - lo > 16)) {
      const uint32_t n = hi - lo, at = lo + (uint32_t)((uint64_t)n * (j + 1) / 17);
      const bool below = n > 16 && A[at] <= d;
      const uint32_t c = (uint32_t)__popcll(ballot(below) >> (group * 16) & 0xFFFF);
      if (n > 16) {
        if (c < 16) hi = lo + (uint32_t)((uint64_t)n * (c + 1) / 17);
        if (c) lo += (uint32_t)((uint64_t)n * c / 17);
      }
    }
    const uint64_t hit = ballot(lo + j < hi && A[lo + j] == d);
    for (int k = 0; k < 4; k++)
      if (r[k] < 64 && (hit >> (k * 16) & 0xFFFF)) there |= 1ull << r[k];
  }
  return there;
}

// For each record (s,d) every plan whose seeded query edge (u0,u1) has
// s in C(u0) and d in C(u1) becomes a DFS root, provided (s,d) is an edge of
// the graph being matched.
//
// A wave takes seed_share records, a lane each as far as their plans (a table by
// label pair); then the (record, plan) pairs lie on the lanes. Pairs whose ends are
// candidates wait in the wave's queue for the look at the record's edge; the seeds
// take one counter add per queue. Bound by the chain of reads from a record to its
// edge: with a lane per record, two binary searches for its plans, one for its edge
// and its plans one after the other, 52 us for 1,024 records and 16 refined queries
// (7 now) and 88 us for 4,096 records and 64 queries beside an update (17 now).
constexpr uint32_t kSeedQueue = 256;
__global__ __launch_bounds__(256) void k_seed(SeedArgs a) {
  __shared__ uint32_t s_pre[4][65], s_plan[4][64], s_rs[4][64], s_rd[4][64], s_tag[4][64], s_q[4][kSeedQueue];
  __shared__ uint8_t s_qr[4][kSeedQueue];
  const uint32_t lane = lane_id(), wv = bcast(threadIdx.x >> 6);
  const uint32_t total = a.nrec[0] + a.nrec[1], share = seed_share(total);
  uint32_t *pre = s_pre[wv], *q = s_q[wv];
  uint8_t *qr = s_qr[wv];
  for (uint32_t i0 = bcast(blockIdx.x * 4 + wv) * share; i0 < total; i0 += gridDim.x * 4 * share) {
    const uint32_t i = i0 + lane;
    uint32_t s = 0, d = 0, tag = 0;
    bool ok = lane < share && i < total;
    if (ok) {
      const uint32_t which = i < a.nrec[0] ? 0u : 1u, r = which ? i - a.nrec[0] : i;
      s = a.rs[which][r];
      d = a.rd[which][r];
      tag = a.tag[which];
      ok = s != d && s < a.g.n && d < a.g.n;
    }
    uint2 plans{0, 0};  // the first, how many
    if (ok) {
      const uint32_t ls = a.lmap[a.g.lab[s]], ld = a.lmap[a.g.lab[d]];
      if (ls < kMaxRel && ld < kMaxRel) plans = a.plan_of[ls * kMaxRel + ld];
    }
    wave_sync();  // the previous records' arrays are no longer read
    if (lane == 0) pre[0] = 0;
    pre[lane + 1] = wave_incl_sum(plans.y);
    s_plan[wv][lane] = plans.x;
    s_rs[wv][lane] = s;
    s_rd[wv][lane] = d;
    s_tag[wv][lane] = tag;
    wave_sync();
    const uint32_t pairs = pre[64];
    uint32_t nq = 0;
    uint64_t met = 0, looked = 0, there = 0;  // records with a queued pair, looked at, with their edge
    for (uint32_t e = 0; e < pairs; e += 64) {
      const uint32_t k[1] = {min(e + lane, pairs - 1)};
      uint32_t o[1];
      ranges_of(pre, k, o);
      const uint32_t p = s_plan[wv][o[0]] + (k[0] - pre[o[0]]);
      const Plan &pl = a.plans[p];
      const uint32_t g0 = pl.sig[0], g1 = pl.sig[1];
      const bool c0 = bit_of(a.bm, a.words, g0, s_rs[wv][o[0]]), c1 = bit_of(a.bm, a.words, g1, s_rd[wv][o[0]]);
      const bool pass = e + lane < pairs && c0 && c1;
      const uint64_t m = ballot(pass);
      if (pass) {
        q[nq + mbcnt(m)] = p;
        qr[nq + mbcnt(m)] = (uint8_t)o[0];
      }
      nq += (uint32_t)__popcll(m);
      met |= (uint64_t)wave_or(pass && o[0] >= 32 ? 1u << (o[0] - 32) : 0u) << 32 |
             wave_or(pass && o[0] < 32 ? 1u << o[0] : 0u);
      if (nq == 0 || (nq <= kSeedQueue - 64 && e + 64 < pairs)) continue;
      // the queue's seeds
      wave_sync();
      there |= edges_there(a.g, met & ~looked, s_rs[wv], s_rd[wv]);
      looked |= met;
      uint32_t n = 0;
      for (uint32_t x = 0; x < nq; x += 64)
        n += (uint32_t)__popcll(ballot(x + lane < nq && (there >> qr[min(x + lane, nq - 1)] & 1)));
      uint32_t base = 0;
      if (n && lane == 0) {
        base = atomicAdd(&a.ctl->nseeds.v, n);
        if (base + n > a.seed_cap) atomicAdd(&a.ctl->seed_overflow.v, n);
      }
      base = bcast(base);
      if (base + n > a.seed_cap) n = 0;
      for (uint32_t x = 0; n && x < nq; x += 64) {
        const uint32_t y = min(x + lane, nq - 1), rec = qr[y];
        const bool out = x + lane < nq && (there >> rec & 1);
        const uint64_t mo = ballot(out);
        if (out) {
          const uint32_t at = base + mbcnt(mo);
          a.seed_plan[at] = q[y];
          a.seed_s[at] = s_rs[wv][rec];
          a.seed_d[at] = s_rd[wv][rec];
          a.seed_tag[at] = s_tag[wv][rec];
        }
        base += (uint32_t)__popcll(mo);
      }
      nq = 0;
      wave_sync();
    }
  }
}

__global__ __launch_bounds__(256) void k_ctl_reset(DfsCtl *ctl, unsigned long long *tuple_count,
                                                    unsigned long long *counts, uint32_t ncounts, IdleWord *idle,
                                                    uint32_t nidle, SmallCopy up) {
  small_copy(up);
  for (uint32_t i = threadIdx.x; counts && i < ncounts; i += blockDim.x) counts[i] = 0;
  for (uint32_t i = threadIdx.x; i < nidle; i += blockDim.x) idle[i].v = 0;
  if (ctl && threadIdx.x < kSeedHeads) ctl->seed_head[threadIdx.x].v = 0;
  if (threadIdx.x == 0) {
    if (tuple_count) *tuple_count = 0;
    if (ctl) {
      ctl->nseeds.v = 0;
      ctl->seed_overflow.v = 0;
      ctl->donated.v = 0;
      ctl->abort.v = 0;
    }
  }
}

// -------------------------------------------------------------------- DFS

// Per-wave DFS state, in dynamic LDS: a fixed header, a window buffer for the
// cooperative intersections and, for each chunk level 2 .. n-2, 64 candidates
// with their prefetched list start and degree. Sized to the engine's largest
// query, so small queries keep high occupancy.
struct WaveHdr {
  uint32_t f[kMaxQ];         // data vertex of each position
  uint32_t fs[kMaxQ];        // its list start
  uint32_t fd[kMaxQ];        // its degree
  uint32_t srcj[kMaxQ];      // backward position whose list drives the scan
  uint32_t pos[kMaxQ];       // next source index
  uint32_t end[kMaxQ];       // one past the last source index
  uint32_t cn[kMaxQ];        // chunk size
  uint32_t ci[kMaxQ];        // next chunk entry
  uint32_t cbase[kMaxQ];     // source index of the chunk's first lane
  uint64_t cmask[kMaxQ];     // lanes of the chunk that passed (k-th set bit = cand[k])
  const uint32_t *src[kMaxQ]; // the list (or label bucket) the level scans
  uint16_t sig[kMaxQ];
  uint16_t back[kMaxQ];
  uint16_t inj[kMaxQ];
  uint8_t qv[kMaxQ];
  uint8_t lix[kMaxQ];
  uint32_t n, query, plan, tag;
  uint32_t donated;          // tasks the wave has handed out
  uint64_t since;            // when it began
  uint32_t fstate, fn;       // leaf set F of the current positions 0..n-3 (see leaf_count)
};
constexpr uint32_t kFCap = 1024;   // largest leaf set F kept in LDS as whole ids
constexpr uint32_t kFScan = 2048;  // longest list it is computed from
// Membership in F goes through a table beside it, of one of two kinds.
// - Up to kFHash entries: a hash set of the ids, kFBuckets buckets of four, a full
//   bucket going on to the next. One 16-byte read settles almost every id (F has
//   21 entries in the mean on the 64-query stream, and a bucket a third of one).
// - More: F indexed by id range: bucket b = id >> DfsArgs::fshift (fshift makes the
//   graph's ids fit kFIdx buckets), fidx[b] = first entry of F at or past the
//   bucket. A test reads two offsets and searches the bucket's few entries.
//   Filling the buckets between two entries is a loop per entry, as long as F is
//   short, which is why the short sets, nearly all of them, take the hash set.
// A set of more than kFCap entries lies in the same words as the low halves of its
// ids, two a word: the bucket gives the rest, where an id has at most 16 bits below its
// bucket's (up to 2^25 vertices; in larger graphs such a set is not kept).
constexpr uint32_t kFIdx = 512;
constexpr uint32_t kFHash = 128;
constexpr uint32_t kFBuckets = 64;
constexpr uint32_t kFEmpty = 0xFFFFFFFFu;
// One level above the leaf, the candidates of a 64-entry window count their
// leaf images inline until their summed scan or search work passes
// DfsArgs::leaf_budget entries; the candidate that passes it descends to the
// leaf level instead, where the scan can be split with idle waves (an inline
// count cannot), and the window resumes after it.
// states of the leaf set F
constexpr uint32_t kFStale = 0;  // not computed for the current positions
constexpr uint32_t kFReady = 1;  // fbuf[0, fn) holds F, ftab its table
constexpr uint32_t kFLarge = 2;  // the shortest fixed list exceeds kFScan, or F kFCap unhalved: per-candidate descent
constexpr uint32_t kFNone = 3;   // the leaf's only backward neighbour is position n-2

struct WaveMem {
  WaveHdr *h;
  uint32_t *win;    // [kWin]
  uint32_t *cand;   // [levels][64]
  uint32_t *cst;    // [levels][64] list start of each candidate
  uint32_t *cdg;    // [levels][64] degree of each candidate
  uint32_t *fbuf;   // [kFCap] leaf set F, ascending (past kFCap entries, halves: [2 kFCap])
  uint32_t *ftab;   // F's table: kFBuckets x 4 ids, or kFIdx + 1 16-bit bucket offsets into fbuf
};
constexpr uint32_t kFTabBytes = ((kFIdx + 1) * 2 + 15) / 16 * 16;
static_assert(kFScan <= 2 * kFCap, "every set in halves fits");
static_assert(kFBuckets * 16 <= kFTabBytes && kFBuckets == 64, "the hash set fits the table, a bucket per lane");

__host__ __device__ constexpr uint32_t wave_lds_bytes(uint32_t chunk_levels) {
  return (uint32_t)((sizeof(WaveHdr) + 15) / 16 * 16) + kWin * 4 + kFCap * 4 + chunk_levels * 64 * 12 + kFTabBytes;
}

// 4 B per entry of the full lists of the positions in `mask`: what a merge
// intersection over those lists reads (the work measure of the expansion).
// Lane j's share: position j's list.
__device__ __forceinline__ uint32_t list_bytes(const WaveHdr &S, uint32_t mask) {
  const uint32_t lane = lane_id();
  return lane < (uint32_t)kMaxQ && (mask >> lane & 1) ? 4u * S.fd[lane] : 0u;
}

// Among the lists of the positions in `mask`, the one with the fewest entries
// of label index li: for a vertex of degree > kLabelSorted, its label bucket in
// the label-sorted copy; otherwise the whole list. Lane j examines position j;
// a minimum over lanes 0 .. 15 picks the shortest, lowest position on ties. Wave-uniform
// results; an empty mask gives length 0.
__device__ __forceinline__ void pick_source(const WaveHdr &S, const DevGraph &g, uint32_t mask, uint32_t li,
                                            const uint32_t *&src, uint32_t &len, uint32_t &j) {
  const uint32_t lane = lane_id();
  uint32_t n = 0xFFFFFFFFu, off = 0, sorted = 0;
  if (mask >> (lane & 31) & 1 && lane < (uint32_t)kMaxQ) {
    n = S.fd[lane];
    off = S.fs[lane];
    if (n > kLabelSorted) {
      const uint32_t *row = g.loff + (size_t)S.f[lane] * (g.nbuckets + 1);
      const uint32_t b0 = row[li], b1 = row[li + 1];
      n = b1 - b0;
      off += b0;
      sorted = 1;
    }
  }
  len = row0_min(n);
  j = 0;
  if (len == 0xFFFFFFFFu) len = 0;
  else j = (uint32_t)__builtin_ctzll(ballot(lane < (uint32_t)kMaxQ && n == len));
  const uint32_t boff = __builtin_amdgcn_readlane(off, j);
  const uint32_t bsorted = __builtin_amdgcn_readlane(sorted, j);
  src = (bsorted ? g.lpool : g.pool) + boff;
}

// Sets up level l to scan source indices [lo, min(hi, length)) of the shortest
// backward list (pick_source); no backward neighbour leaves it empty.
__device__ __forceinline__ void init_level(WaveHdr &S, const DevGraph &g, uint32_t l, uint32_t lo, uint32_t hi) {
  const uint32_t *src;
  uint32_t best, bj;
  pick_source(S, g, S.back[l], S.lix[l], src, best, bj);
  wave_sync();
  if (lane_id() == 0) {
    S.srcj[l] = bj;
    S.src[l] = src;
    S.pos[l] = lo;
    S.end[l] = hi < best ? hi : best;
    S.cn[l] = 0;
    S.ci[l] = 0;
  }
  wave_sync();
}

// Tests source entries [p, min(p + 64, e)) of `src`, one per lane: the
// candidate bit of signature `sig`, injectivity against the positions in
// `inj` and membership in the list of every position in `oth`. The bit is
// probed first (it narrows the membership windows) or, with bit_probe_last,
// only for the entries that passed the membership tests (the bitmap words are
// scattered reads; the windows are contiguous). The source chunk is sorted, so the entries still
// alive span [wmin, wmax]; the wave finds that window of the other list
// cooperatively (bounds2) and, when it holds at most kWin entries, stages it
// in LDS for the lanes' searches.
__device__ __forceinline__ bool test_entries(const WaveMem &M, const DfsArgs &a, const uint32_t *src, uint32_t oth,
                                             uint32_t inj, uint32_t sig, uint32_t p, uint32_t e, uint32_t &w,
                                             uint32_t &loads) {
  WaveHdr &S = *M.h;
  const uint32_t lane = lane_id();
  const uint32_t i = p + lane;
  bool ok = i < e;
  w = ok ? src[i] : 0xFFFFFFFFu;
  if (!a.bit_probe_last) ok = ok && bit_of(a.bm, a.words, sig, w);
  while (inj) {
    const uint32_t j = __builtin_ctz(inj);
    inj &= inj - 1;
    ok = ok && S.f[j] != w;
  }
  while (oth) {
    const uint32_t j = __builtin_ctz(oth);
    oth &= oth - 1;
    if (ballot(ok) == 0) break;
    ok = window_member(a.g.pool + S.fs[j], S.fd[j], w, ok, M.win, loads);
  }
  if (a.bit_probe_last) ok = ok && bit_of(a.bm, a.words, sig, w);
  return ok;
}

// The level's own chunk test: source = its chosen list, membership in the
// other backward lists, injectivity and signature of level l.
__device__ __forceinline__ bool test_chunk(const WaveMem &M, const DfsArgs &a, uint32_t l, uint32_t p,
                                           uint32_t e, uint32_t &w, uint32_t &loads) {
  const WaveHdr &S = *M.h;
  return test_entries(M, a, S.src[l], S.back[l] & ~(1u << S.srcj[l]), S.inj[l], S.sig[l], p, e, w, loads);
}

// An id's first bucket in the hash set of a short leaf set.
__device__ __forceinline__ uint32_t f_hash(uint32_t y) { return (y * 0x9E3779B1u) >> 26; }

// Leaf set F for positions 0..n-3 (leaf = n-1): the images the leaf may take
// judging only by its backward neighbours other than position n-2, i.e. the
// entries of the intersection of their lists (label bucket of the shortest)
// that carry the leaf's signature bit and differ from the earlier images of
// its label. F is sorted. Sets fstate: kFReady (F in fbuf), kFLarge (shortest
// such list longer than kFScan, or F than kFCap with ids too long for halves) or kFNone
// (no such neighbour). A set found to pass kFCap is computed anew, in halves, with its
// bucket offsets: squares over lists of 1,900 entries (12,000 vertices) take 8.4 ms for 8
// records and 79 for 256 with a descent per candidate instead, 3.4 and 29 in halves.
__device__ __forceinline__ void compute_leaf_set(const WaveMem &M, const DfsArgs &a, uint32_t leaf, uint32_t &scanned,
                                 uint32_t &loads) {
  WaveHdr &S = *M.h;
  const uint32_t lane = lane_id();
  const uint32_t pv = leaf - 1;
  const uint32_t bp = S.back[leaf] & ~(1u << pv);
  uint32_t state = kFReady, cnt = 0;
  uint16_t *fidx = reinterpret_cast<uint16_t *>(M.ftab);
  const uint32_t sh = a.fshift;
  bool halves = false;
  uint32_t open = 0;  // of halves: the first bucket without an offset
  if (bp == 0) {
    state = kFNone;
  } else {
    const uint32_t *src;
    uint32_t len, j;
    pick_source(S, a.g, bp, S.lix[leaf], src, len, j);
    if (len > kFScan) {
      state = kFLarge;
    } else {
      const uint32_t oth = bp & ~(1u << j);
      const uint32_t inj = S.inj[leaf] & ~(1u << pv);
      const uint32_t sig = S.sig[leaf];
      for (uint32_t p = 0; p < len; p += 64) {
        uint32_t w;
        const bool ok = test_entries(M, a, src, oth, inj, sig, p, len, w, loads);
        scanned += p + lane < len ? 1u : 0u;
        const uint64_t m = ballot(ok);
        if (!halves && cnt + (uint32_t)__popcll(m) > kFCap) {
          if (sh > 16) {
            state = kFLarge;
            break;
          }
          halves = true;
          cnt = 0;
          p = 0u - 64;
          continue;
        }
        const uint32_t at = cnt + mbcnt(m);
        if (!halves) {
          if (ok) M.fbuf[at] = w;
        } else if (m) {
          // entry `at` opens every bucket after its predecessor's up to its own
          const uint32_t b = w >> sh;
          const uint64_t below = m & ((1ull << lane) - 1);
          const uint32_t before = __shfl(b, below ? 63 - __builtin_clzll(below) : 0) + 1;
          if (ok) {
            for (uint32_t k = below ? before : open; k <= b; k++) fidx[k] = (uint16_t)at;
            reinterpret_cast<uint16_t *>(M.fbuf)[at] = (uint16_t)w;
          }
          open = __builtin_amdgcn_readlane(b, 63 - __builtin_clzll(m)) + 1;
        }
        cnt += (uint32_t)__popcll(m);
      }
    }
  }
  wave_sync();
  if (halves) {
    for (uint32_t k = open + lane; k <= kFIdx; k += 64) fidx[k] = (uint16_t)cnt;
  } else if (state == kFReady && cnt <= kFHash) {
    reinterpret_cast<uint4 *>(M.ftab)[lane] = uint4{kFEmpty, kFEmpty, kFEmpty, kFEmpty};
    wave_sync();
    for (uint32_t i = lane; i < cnt; i += 64) {
      const uint32_t y = M.fbuf[i];
      uint32_t at = f_hash(y) * 4;
      while (atomicCAS(&M.ftab[at], kFEmpty, y) != kFEmpty) at = (at + 1) % (kFBuckets * 4);
    }
  } else if (state == kFReady) {
    // bucket offsets: entry i opens every bucket after its predecessor's up
    // to its own; buckets past the last entry start at cnt
    for (uint32_t i = lane; i < cnt; i += 64) {
      const uint32_t b = M.fbuf[i] >> sh;
      const uint32_t pb = i ? (M.fbuf[i - 1] >> sh) + 1 : 0u;
      for (uint32_t k = pb; k <= b; k++) fidx[k] = (uint16_t)i;
    }
    const uint32_t last = (M.fbuf[cnt - 1] >> sh) + 1;
    for (uint32_t k = last + lane; k <= kFIdx; k += 64) fidx[k] = (uint16_t)cnt;
  }
  wave_sync();
  if (lane == 0) {
    S.fstate = state;
    S.fn = cnt;
  }
  wave_sync();
}

// Looks a lane's id y up in bucket h of the hash set. Returns true when that
// settles it: the bucket holds y (found) or is not full.
__device__ __forceinline__ bool f_look(const uint4 &t, uint32_t y, bool &found) {
  found = t.x == y || t.y == y || t.z == y || t.w == y;
  return found || t.w == kFEmpty;
}

// y in F of more than kFHash entries, which are whole ids or, past kFCap, halves.
template <typename T>
__device__ __forceinline__ bool in_leaf_range(const WaveMem &M, const DfsArgs &a, uint32_t y) {
  const uint16_t *fidx = reinterpret_cast<const uint16_t *>(M.ftab);
  const uint32_t b = y >> a.fshift;
  const uint32_t lo = fidx[b], hi = fidx[b + 1];
  return lds_contains(reinterpret_cast<const T *>(M.fbuf) + lo, hi - lo, (T)y);
}

// y in F (state kFReady, fn entries), through F's table.
__device__ __forceinline__ bool in_leaf_set(const WaveMem &M, const DfsArgs &a, uint32_t fn, uint32_t y) {
  if (fn <= kFHash) {
    bool found;
    for (uint32_t h = f_hash(y); !f_look(reinterpret_cast<const uint4 *>(M.ftab)[h], y, found);) h = (h + 1) % kFBuckets;
    return found;
  }
  return fn <= kFCap ? in_leaf_range<uint32_t>(M, a, y) : in_leaf_range<uint16_t>(M, a, y);
}

// Entry k of F.
__device__ __forceinline__ uint32_t f_entry(const WaveMem &M, const DfsArgs &a, uint32_t fn, uint32_t k) {
  if (fn <= kFCap) return M.fbuf[k];
  const uint16_t *fidx = reinterpret_cast<const uint16_t *>(M.ftab);
  uint32_t b = 0;  // the last bucket that starts at or before k, and so holds it
  for (uint32_t half = kFIdx / 2; half; half >>= 1) b = fidx[b + half] <= k ? b + half : b;
  return b << a.fshift | (reinterpret_cast<const uint16_t *>(M.fbuf)[k] & ((1u << a.fshift) - 1));
}

// Leaf images of the partial match whose position n-2 holds w (this lane's
// candidate), given F. With the leaf not adjacent to position n-2 the count is
// |F|. Otherwise it scans w's list (its label bucket when sorted copies exist):
// with F, the entries that lie in F; with no other backward neighbour
// (kFNone), the entries that carry the leaf's signature and differ from the
// earlier images of its label. Injectivity against w itself applies when the
// leaf has w's label. The lanes' scans are shared by the wave
// (leaf_scan_segments); a list much longer than F is left to leaf_count_wave,
// which searches F's elements in it. Without leaf_segments a lane scans a list
// of up to a.lane_work entries itself and leaves longer ones to the wave.

struct LeafList {
  const uint32_t *L;
  uint32_t len;
  bool by_f;  // search F's elements in L instead of scanning L
};

// Reads of one search for each of F's elements in a list of len entries.
__device__ __forceinline__ uint32_t search_reads(uint32_t len) { return 33u - (uint32_t)__builtin_clz(len | 1u); }

// F's elements are searched in the list when that is fewer dependent steps for
// the wave: a search takes search_reads(len) of them for up to 256 elements (four
// a lane), a scan one for 256 entries, which come in whole lines. The line lies
// at kScanPerStep entries a step.
constexpr uint32_t kScanPerStep = 128;
__device__ __forceinline__ bool search_f(uint32_t fn, uint32_t len) {
  return len > kScanPerStep * search_reads(len) * ((fn + 255) / 256);
}

// A leaf level's constants, read once per scan.
struct LeafRule {
  uint32_t st, fn, sig, inj;
  bool injw;
};
__device__ __forceinline__ LeafRule leaf_rule(const WaveHdr &S, uint32_t leaf) {
  const uint32_t inj = S.inj[leaf];
  return LeafRule{S.fstate, S.fn, S.sig[leaf], inj & ~(1u << (leaf - 1)), (bool)(inj >> (leaf - 1) & 1)};
}

// Whether y is a leaf image; w is the image of position n-2 it belongs to.
__device__ __forceinline__ bool leaf_accept_one(const WaveMem &M, const DfsArgs &a, const LeafRule &r, uint32_t w,
                                                uint32_t y) {
  if (r.injw && y == w) return false;
  if (r.st == kFReady) return in_leaf_set(M, a, r.fn, y);
  if (!bit_of(a.bm, a.words, r.sig, y)) return false;
  uint32_t m = r.inj;
  while (m) {
    const uint32_t j = __builtin_ctz(m);
    m &= m - 1;
    if (M.h->f[j] == y) return false;
  }
  return true;
}

// How many of a lane's K entries y are leaf images; w is the image of position
// n-2 each belongs to, ok the entries that exist.
template <int K>
__device__ __forceinline__ uint32_t leaf_accept(const WaveMem &M, const DfsArgs &a, const LeafRule &r,
                                                const uint32_t (&w)[K], const uint32_t (&y)[K], bool (&ok)[K]) {
  const WaveHdr &S = *M.h;
  uint32_t c = 0;
  if (r.st == kFReady) {
    if (r.fn <= kFHash) {
      uint4 t[K];
#pragma unroll
      for (int u = 0; u < K; u++) t[u] = reinterpret_cast<const uint4 *>(M.ftab)[f_hash(y[u])];
#pragma unroll
      for (int u = 0; u < K; u++) {
        bool found;
        if (!f_look(t[u], y[u], found)) found = in_leaf_set(M, a, r.fn, y[u]);
        c += ok[u] && found && !(r.injw && y[u] == w[u]) ? 1u : 0u;
      }
    } else if (r.fn <= kFCap) {
#pragma unroll
      for (int u = 0; u < K; u++)
        c += ok[u] && !(r.injw && y[u] == w[u]) && in_leaf_range<uint32_t>(M, a, y[u]) ? 1u : 0u;
    } else {
#pragma unroll
      for (int u = 0; u < K; u++)
        c += ok[u] && !(r.injw && y[u] == w[u]) && in_leaf_range<uint16_t>(M, a, y[u]) ? 1u : 0u;
    }
    return c;
  }
  uint64_t bw[K];
#pragma unroll
  for (int u = 0; u < K; u++) bw[u] = a.bm[(size_t)r.sig * a.words + (ok[u] ? y[u] >> 6 : 0u)];
#pragma unroll
  for (int u = 0; u < K; u++) ok[u] = ok[u] && (bw[u] >> (y[u] & 63) & 1) && !(r.injw && y[u] == w[u]);
  uint32_t m = r.inj;
  while (m) {
    const uint32_t j = __builtin_ctz(m);
    m &= m - 1;
    const uint32_t f = S.f[j];
#pragma unroll
    for (int u = 0; u < K; u++) ok[u] = ok[u] && f != y[u];
  }
#pragma unroll
  for (int u = 0; u < K; u++) c += ok[u] ? 1u : 0u;
  return c;
}

__device__ __forceinline__ uint32_t leaf_count_lane(const WaveMem &M, const DfsArgs &a, uint32_t leaf, uint32_t w,
                                                    bool &defer, bool &scan, LeafList &out, uint32_t &scanned,
                                                    uint32_t &loads, uint32_t &wdeg) {
  const WaveHdr &S = *M.h;
  const uint32_t pv = leaf - 1;
  const uint32_t back = S.back[leaf];
  const LeafRule r = leaf_rule(S, leaf);
  defer = false;
  if (!((back >> pv) & 1)) {
    uint32_t c = r.fn;
    if (r.injw && in_leaf_set(M, a, r.fn, w)) c--;
    return c;
  }
  // the bucket offsets are read beside the degree that says whether they count
  const uint32_t *row = a.g.loff + (size_t)w * (a.g.nbuckets + 1) + S.lix[leaf];
  const uint32_t ws = a.g.start[w], wd = a.g.deg[w], b0 = row[0], b1 = row[1];
  wdeg = wd;
  out.L = a.g.pool + ws;
  out.len = wd;
  if (wd > kLabelSorted) {
    out.L = a.g.lpool + ws + b0;
    out.len = b1 - b0;
    loads += 2;
  }
  out.by_f = r.st == kFReady && search_f(r.fn, out.len);
  if (out.by_f || (!a.leaf_segments && out.len > a.lane_work)) {
    defer = true;
    return 0;
  }
  if (a.leaf_segments) {
    scan = true;
    return 0;
  }
  uint32_t c = 0;
  for (uint32_t k = 0; k < out.len; k++) c += leaf_accept_one(M, a, r, w, out.L[k]) ? 1u : 0u;
  scanned += out.len;
  return c;
}

// The lists of the lanes with `has`, scanned as one segmented array: entry k
// of the concatenation is read by lane k mod 64. Short lists thus share each
// 64-entry step instead of keeping their lanes in a serial loop, and
// consecutive entries of a list are read by consecutive lanes. Four steps are
// taken at a time, their reads in flight together. The lists that are not empty
// sit in the window buffer (where its entry 0 would be, and w); the list of an
// entry is the number of list starts at or before it, from the starts' bits, which
// are set there for 2,048 entries at a time. Returns this lane's share of the count (the task sums the
// wave).
//
// Bound by the latency of the reads and of the LDS steps between them: a step of
// 64 entries took 2,460 cycles one at a time, with the list found by a binary
// search over shuffles, and was 27% of the search (1M vertices, 64 queries). With
// it, the hash sets, searches four at a time and the DPP scans, the waves' time
// on tasks fell from 19.4 to 12.5 s per launch at 2,048 waves. With the starts' bits
// put together from the lanes by two wave-wide ors a step, not set in LDS, the launch
// takes 2% longer. Fetching the next
// four steps ahead of the tests takes 14 more registers and gave 2%; the update
// beside the round then waits for room, so it is not done.
constexpr uint32_t kStartBits = 64 * 32;
__device__ __forceinline__ uint32_t leaf_scan_segments(const WaveMem &M, const DfsArgs &a, uint32_t leaf, uint32_t w,
                                                       bool has, const LeafList &ll, uint32_t &scanned) {
  constexpr int K = 4;
  const uint32_t lane = lane_id();
  const uint32_t n = has ? ll.len : 0u;
  const uint64_t lists = ballot(n > 0);
  if (lists == 0) return 0;
  uint32_t total;
  const uint32_t excl = wave_excl_sum(n, &total);
  const LeafRule r = leaf_rule(*M.h, leaf);
  // [64]: x, y a list's entry 0; z its w; the w words hold the bits of the starts
  uint4 *seg = reinterpret_cast<uint4 *>(M.win);
  wave_sync();
  if (n > 0) {
    const unsigned long long p = (unsigned long long)ll.L - 4ull * excl;
    seg[mbcnt(lists)] = uint4{(uint32_t)p, (uint32_t)(p >> 32), w, 0};
  }
  uint32_t c = 0;
  for (uint32_t part = 0; part < total; part += kStartBits) {
    // bit k: a list starts at entry part + k + 1
    wave_sync();
    seg[lane].w = 0;
    wave_sync();
    const uint32_t bit = excl - 1 - part;
    if (n > 0 && excl > part && bit < kStartBits) atomicOr(&seg[bit >> 5].w, 1u << (bit & 31));
    wave_sync();
    uint32_t before = (uint32_t)__popcll(ballot(n > 0 && excl > 0 && excl <= part));
    for (uint32_t at = 0; at < kStartBits && part + at < total; at += 64 * K) {
      uint32_t wo[K], y[K];
      uint64_t starts[K];
      bool ok[K];
#pragma unroll
      for (int u = 0; u < K; u++)
        starts[u] = (uint64_t)seg[at / 32 + 2 * u + 1].w << 32 | seg[at / 32 + 2 * u].w;
#pragma unroll
      for (int u = 0; u < K; u++) {
        const uint32_t k = part + at + 64 * u + lane;
        const uint4 s = seg[before + mbcnt(starts[u])];
        before += (uint32_t)__popcll(bcast64(starts[u]));
        const uint32_t *L = reinterpret_cast<const uint32_t *>((unsigned long long)s.y << 32 | s.x);
        wo[u] = s.z;
        ok[u] = k < total;
        y[u] = L[ok[u] ? k : total - 1];
      }
      c += leaf_accept(M, a, r, wo, y, ok);
    }
  }
  scanned += n;
  wave_sync();  // the window buffer is free again
  return c;
}

// The deferred lanes' lists, one after another, 256 F elements (or list entries)
// at a time across the wave; returns this lane's share of the count.
__device__ __forceinline__ uint32_t leaf_count_wave(const WaveMem &M, const DfsArgs &a, uint32_t leaf, uint32_t w,
                                                    bool defer, const LeafList &ll, uint32_t &scanned,
                                                    uint32_t &loads) {
  constexpr int K = 4;
  const uint32_t lane = lane_id();
  uint32_t c = 0;
  uint64_t dm = ballot(defer);
  if (dm == 0) return 0;
  const LeafRule r = leaf_rule(*M.h, leaf);
  const uint32_t llo = (uint32_t)(unsigned long long)ll.L, lhi = (uint32_t)((unsigned long long)ll.L >> 32);
  while (dm) {
    const uint32_t src = (uint32_t)__builtin_ctzll(dm);
    dm &= dm - 1;
    const uint32_t *L = reinterpret_cast<const uint32_t *>(
        (unsigned long long)__builtin_amdgcn_readlane(lhi, src) << 32 | (uint32_t)__builtin_amdgcn_readlane(llo, src));
    const uint32_t len = __builtin_amdgcn_readlane(ll.len, src);
    const uint32_t ww = __builtin_amdgcn_readlane(w, src);
    const bool by_f = __builtin_amdgcn_readlane((uint32_t)ll.by_f, src) != 0;
    if (by_f) {
      for (uint32_t k0 = 0; k0 < r.fn; k0 += 64 * K) {
        uint32_t x[K];
        bool in[K];
#pragma unroll
        for (int u = 0; u < K; u++) x[u] = k0 + 64 * u + lane < r.fn ? f_entry(M, a, r.fn, k0 + 64 * u + lane) : 0xFFFFFFFFu;
        contains_each(L, len, x, in);
#pragma unroll
        for (int u = 0; u < K; u++) c += in[u] && !(r.injw && x[u] == ww) ? 1u : 0u;
      }
      for (uint32_t k = lane; k < r.fn; k += 64) loads += search_reads(len);
    } else {
      for (uint32_t k = lane; k < len; k += 64) {
        c += leaf_accept_one(M, a, r, ww, L[k]) ? 1u : 0u;
        scanned++;
      }
    }
  }
  return c;
}

__device__ __forceinline__ void emit_tuples(const WaveHdr &S, const DfsArgs &a, uint32_t l, uint32_t w, bool ok) {
  const uint64_t m = ballot(ok);
  if (m == 0) return;
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(a.tuple_count, (unsigned long long)__popcll(m));
  base = bcast64(base);
  if (!ok) return;
  const unsigned long long idx = base + mbcnt(m);
  if (idx >= a.tuple_cap) return;
  uint32_t *t = a.tuples + idx * (kMaxQ + 2);
  t[0] = S.query;
  t[1] = S.tag;
  for (uint32_t k = S.n; k < (uint32_t)kMaxQ; k++) t[2 + k] = 0xFFFFFFFFu;
  for (uint32_t j = 0; j < l; j++) t[2 + S.qv[j]] = S.f[j];
  t[2 + S.qv[l]] = w;
}

// Hands ranges of the wave's unscanned work to waiting waves.
//
// Levels shallower than the current one give away work when enough entries
// remain there (fetched-but-unconsumed chunk entries count: their source
// indices are recovered from the chunk mask): two, when the level is two or
// more above the leaf; sixteen one level above it. The level being scanned
// gives away work only when at least donate_min source entries remain. The
// receiver re-fetches and re-filters the donated source range [mid, end).
//
// Up to kDonateBurst ranges go out per call, each half of what is left at the
// shallowest level that still holds enough, so that when most of the grid runs
// dry at once the work spreads in fewer check periods.
//
// Words that the whole grid reads or counts on bound the search once it is
// spread: with one pair of ticket counters, read by every busy wave every eight
// scan steps, 1,024 waves on 128 or on 256 CUs took the same time, 2,048 waves
// 14.0 ms per launch (1M vertices, 64 queries, batches of 4,096) and their time
// on tasks fell by 30% when they looked 32 times less often. With a waiting word
// per 16 waves, each busy wave looking at another one each time, a mailbox per
// wave and work counted in registers, the same launches take 10.1 ms, and
// looking every fourth step costs nothing (9.9 ms).
constexpr uint32_t kDonateBurst = DSM_DONATE_BURST;
constexpr uint32_t kMaxParts = 64;  // shares a seed is cut into at most
constexpr unsigned long long kIdleBits = (1ull << kIdleGroup) - 1;

// A wave among the grid's. Those of the blocks that begin at once (a.crew waves) have the
// first a.cgroups waiting words, the reserve's the rest.
struct Crew {
  uint32_t nwaves;
  uint32_t me;       // this wave
  uint32_t look;     // the waiting word it looks at next
};

// One range to a wave that waits in word g; `word` (lane 0) is what lane 0 last
// saw of it. The claim is a compare-and-swap of the word: its owner is no longer
// waiting from then on, and finds the task in its mailbox. CAP: the round has a limit
// of tasks handed out (a kernel of its own: the look at it in the others, never taken,
// cost the 64-query search 0.8%).
template <bool CAP>
__device__ __forceinline__ bool donate_one(WaveHdr &S, const DfsArgs &a, uint32_t L0, uint32_t l, uint32_t n,
                                           Crew &cr, uint32_t g, unsigned long long &word) {
  uint32_t lv = 0xFFFFFFFFu, mid = 0, keep_cn = 0;
  for (uint32_t k = L0; k <= l; k++) {
    const uint32_t p = S.pos[k], e = S.end[k];
    const uint32_t unf = e > p ? e - p : 0;
    if (k == l) {
      // entries one level above the leaf carry a leaf count each
      const uint32_t dmin = k + 2 == n ? a.donate_min_n2 : a.donate_min;
      if (unf >= dmin) {
        lv = k;
        mid = p + unf / 2;
      }
      break;
    }
    const uint32_t ci = S.ci[k], cn = S.cn[k];
    const uint32_t rem = cn - ci;
    // an entry two or more levels above the leaf roots a subtree worth a
    // hand-off; one level above, only a leaf scan
    const uint32_t need = (k + 3 <= n) ? 2u : 16u;
    if (rem + unf < need) continue;
    if (unf >= 2) {
      lv = k;
      mid = p + unf / 2;
      keep_cn = cn;
      break;
    }
    {
      // split the unconsumed chunk: keep [ci, ci+half), donate from the
      // source index of entry ci+half to the end of the range
      const uint32_t half = (rem + unf) / 2;
      const uint32_t kth = ci + half;
      if (half == 0 || kth >= cn) continue;
      uint64_t m = S.cmask[k];
      for (uint32_t i = 0; i < kth; i++) m &= m - 1;
      lv = k;
      mid = S.cbase[k] + (uint32_t)__builtin_ctzll(m);
      keep_cn = kth;
      break;
    }
  }
  if (lv == 0xFFFFFFFFu) return false;
  // a place under the limit first, which goes back if no wave is waiting, as does one past it
  if constexpr (CAP) {
    uint32_t room = 0;
    if (lane_id() == 0 && ld_relaxed(&a.ctl->donated.v) < a.donate_cap) {
      room = atomicAdd(&a.ctl->donated.v, 1u) < a.donate_cap;
      if (!room) atomicSub(&a.ctl->donated.v, 1u);
    }
    if (!bcast(room)) return false;
  }
  const uint32_t e = S.end[lv];
  uint32_t who = 0xFFFFFFFFu;
  if (lane_id() == 0) {
    while (word & kIdleBits) {
      const uint32_t b = (uint32_t)__builtin_ctzll(word);
      const unsigned long long next = (word & ~(1ull << b)) + (1ull << 32);
      const unsigned long long was = atomicCAS(&a.idle[g].v, word, next);
      if (was == word) {
        who = g < a.cgroups ? b * a.cgroups + g : a.crew + b * (a.ngroups - a.cgroups) + g - a.cgroups;
        word = next;
        break;
      }
      word = was;
    }
  }
  who = bcast(who);
  if (who == 0xFFFFFFFFu) {
    if (CAP && lane_id() == 0) atomicSub(&a.ctl->donated.v, 1u);
    return false;
  }
  const uint32_t lane = lane_id();
  uint32_t pay = 0;
  if (lane == 0) pay = S.plan;
  else if (lane == 1) pay = lv;
  else if (lane == 2) pay = mid;
  else if (lane == 3) pay = e;
  else if (lane < 4u + kMaxQ) pay = S.f[lane - 4];
  else if (lane == 4u + kMaxQ) pay = S.tag;
  if (lane < (uint32_t)kTaskWords) reinterpret_cast<uint32_t *>(&a.mail[who])[lane] = pay;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  if (lane == 0) {
    atomicAdd(&a.mail[who].mail, 1u);
    // the donor keeps source indices below mid; after a split inside the
    // chunk, mid <= pos, so nothing is left to fetch at this level and a later
    // split there donates [mid', mid) only
    if (lv != l && keep_cn != S.cn[lv]) S.cn[lv] = keep_cn;
    S.end[lv] = mid;
    S.donated++;
  }
  wave_sync();
  return true;
}

template <bool CAP>
__device__ __forceinline__ void try_donate(WaveHdr &S, const DfsArgs &a, uint32_t L0, uint32_t l, uint32_t n, Crew &cr) {
  const uint32_t g = cr.look;
  // the reserve's words too once it has joined
  const bool last = g + 1 == a.cgroups ? a.cgroups == a.ngroups || wall_clock64() - bcast64(S.since) < a.join_after
                                       : g + 1 == a.ngroups;
  cr.look = last ? 0u : g + 1;
  unsigned long long word = 0;
  if (lane_id() == 0) word = ld_relaxed(&a.idle[g].v);
  const uint32_t waiting = bcast((uint32_t)__popcll(word & kIdleBits));
  for (uint32_t k = 0; k < waiting && k < kDonateBurst; k++)
    if (!donate_one<CAP>(S, a, L0, l, n, cr, g, word)) break;
}

// Where wave `me` marks that it has started and that it waits.
struct IdlePlace {
  uint32_t word, bit;
};
__device__ __forceinline__ IdlePlace idle_place(const DfsArgs &a, uint32_t me) {
  const bool crew = me < a.crew;
  const uint32_t w = crew ? me : me - a.crew, words = crew ? a.cgroups : a.ngroups - a.cgroups;
  return IdlePlace{(crew ? 0u : a.cgroups) + w % words, w / words};
}

// No started wave has work: every waiting word has all its started waves
// waiting, twice in a row with no claim between. Work can only come from a
// busy wave, so nothing is left then, apart from waves that start later, which
// bring a seed of their own and finish it alone.
__device__ __forceinline__ bool all_waiting(const DfsArgs &a) {
  uint32_t claims = 0;
  for (int pass = 0; pass < 2; pass++) {
    wave_sync();  // keeps the passes apart; the words are read past the caches
    uint32_t c = 0;
    bool all = true;
    for (uint32_t g = lane_id(); g < a.ngroups; g += 64) {
      const unsigned long long v = ld_relaxed(&a.idle[g].v);
      all = all && (v & kIdleBits) == (v >> kIdleGroup & kIdleBits);
      c += (uint32_t)(v >> 32);
    }
    if (pass == 1) all = all && c == claims;
    claims = c;
    if (ballot(!all)) return false;
  }
  return true;
}

// A wave out of work: marks itself waiting in its word and polls its mailbox.
// Returns true with a task in it, false when the launch is over (or aborted).
// The wave whose mark completes its word looks at all of them, and when no wave
// has work it tells every mailbox to stop. A wave that stops takes its mark
// back first; if a busy wave claimed it in the meantime (one that started late,
// after the others had been told to stop), it takes that task instead.
__device__ __forceinline__ bool wait_for_task(const DfsArgs &a, const Crew &cr, uint32_t &seen) {
  const uint32_t lane = lane_id();
  const IdlePlace at = idle_place(a, cr.me);
  unsigned long long *word = &a.idle[at.word].v;
  const uint32_t b = at.bit;
  const unsigned long long bits = 1ull << b | 1ull << (b + kIdleGroup);
  uint32_t full = 0;
  if (lane == 0) {
    const unsigned long long v = atomicOr(word, bits) | bits;
    full = (v & kIdleBits) == (v >> kIdleGroup & kIdleBits);
  }
  bool look = bcast(full) != 0;
  Mailbox *mb = &a.mail[cr.me];
  const uint64_t since = wall_clock64();
  for (uint32_t naps = 0;; naps++) {
    if (look && all_waiting(a))
      for (uint32_t w = lane; w < cr.nwaves; w += 64)
        __hip_atomic_store(&a.mail[w].stop, a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    look = false;
    // relaxed poll: an acquire here would invalidate the CU's L1 on every poll
    // of every waiting wave; the acquire fence follows a hit instead
    unsigned long long ms = 0;
    if (lane == 0) ms = ld_relaxed(reinterpret_cast<unsigned long long *>(&mb->mail));
    ms = bcast64(ms);
    if ((uint32_t)ms != seen) {
      seen = (uint32_t)ms;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      return true;
    }
    if ((uint32_t)(ms >> 32) == a.epoch) {
      uint32_t mine = 0;
      if (lane == 0) mine = (uint32_t)(atomicAnd(word, ~bits) >> b) & 1u;
      if (bcast(mine)) return false;
    }
    if ((naps & 63) == 63) {
      // the abort flag and the watchdog; one wave per word looks at the words again
      look = b == 0;
      uint32_t out = 0;
      if (lane == 0) {
        out = ld_relaxed(&a.ctl->abort.v);
        if (!out && wall_clock64() - since > a.watchdog) {
          st_release(&a.ctl->abort.v, 1u);
          out = 1;
        }
      }
      if (bcast(out)) return false;
    }
    const uint32_t reps = (1u << (naps < 4 ? naps : 4u)) < a.poll_max ? (1u << (naps < 4 ? naps : 4u)) : a.poll_max;
    for (uint32_t r = 0; r < reps; r++) __builtin_amdgcn_s_sleep(8);
  }
}

// A block of the reserve (whose waves come after the first a.crew): waits until the round is over
// (false) or has lasted long enough to be worth its waves (true). It joins as a block does
// that starts late, which the words above allow for: it takes what seeds are left and then
// waits for tasks. Its first wave watches its mailbox for the round's end, the others wait
// at the barrier.
__device__ __forceinline__ bool reserve_joins(const DfsArgs &a, uint32_t total, uint32_t me, uint64_t since) {
  __shared__ uint32_t s_joins;
  if (total == 0) return false;  // nobody will say that the round is over
  if (threadIdx.x < 64) {
    uint32_t joins = 0;
    for (;;) {
      uint32_t stop = 0;
      if (lane_id() == 0) stop = ld_relaxed(&a.mail[me].stop);
      if (bcast(stop) == a.epoch) break;
      joins = wall_clock64() - since >= a.join_after;
      if (joins) break;
      for (uint32_t r = 0; r < 4; r++) __builtin_amdgcn_s_sleep(8);
    }
    if (lane_id() == 0) s_joins = joins;
  }
  __syncthreads();
  return s_joins != 0;
}

// Bound by latency: dependent scattered reads and LDS steps, on few waves. What
// counts is how many waves fit. Registers: the wave's index is made uniform, so
// that its LDS addresses live in scalar registers (135 -> 96 vector registers; at
// most 128 leave room for the 16-wave blocks of an update beside three blocks
// per CU, which otherwise wait for the round to end). LDS: 10.3 KB a wave with a
// leaf set of 1,024 entries, three blocks of four waves per CU beside an update;
// 14.3 KB, two blocks, with 2,048. Per launch (1M vertices, 64 queries, batches
// of 4,096, beside the update): 8.1 ms at two blocks, 6.1 at three, 5.9 at four
// (a 512-entry leaf set), where the update falls behind; 5.6 at three with hash
// sets for the short leaf sets.
template <int WPB, bool TUP, bool CAP>
__global__ __launch_bounds__(WPB * 64, 4) void k_dfs(DfsArgs a, uint32_t chunk_levels) {
  extern __shared__ __align__(16) uint8_t s_dyn[];
  const uint32_t lane = lane_id();
  const uint32_t wv = bcast(threadIdx.x >> 6);
  WaveMem M;
  {
    uint8_t *base = s_dyn + wv * wave_lds_bytes(chunk_levels);
    M.h = reinterpret_cast<WaveHdr *>(base);
    M.win = reinterpret_cast<uint32_t *>(base + (sizeof(WaveHdr) + 15) / 16 * 16);
    M.cand = M.win + kWin;
    M.cst = M.cand + chunk_levels * 64;
    M.cdg = M.cst + chunk_levels * 64;
    M.fbuf = M.cdg + chunk_levels * 64;
    M.ftab = M.fbuf + kFCap;
  }
  WaveHdr &S = *M.h;
  if (lane == 0) {
    S.plan = 0xFFFFFFFFu;
    S.donated = 0;
    S.since = wall_clock64();
  }
  wave_sync();
  // what the block's waves did, for its record
  __shared__ unsigned long long s_rec[WPB][7];
  Crew cr;
  cr.nwaves = gridDim.x * WPB;
  cr.me = blockIdx.x * WPB + wv;
  cr.look = (cr.me + 1) % a.cgroups;
  // a seed table overflow leaves unwritten slots: match nothing, the host
  // reports the error (the table is sized so that it cannot happen)
  const uint32_t nseeds = a.ctl->seed_overflow.v ? 0u : a.ctl->nseeds.v;
  // With fewer seeds than waves, every seed is cut into `parts` shares of its
  // first level's source range, so that the grid starts with work for all
  // instead of spreading it by halves (100,000 vertices, 4 queries, batches of
  // 256, about 30 seeds a launch: 230 -> 96 us, with the waiting words).
  // Shares are claimed, never assigned by wave index: the grid is sized to what
  // the occupancy query says fits, but nothing guarantees that every block is
  // resident at once (an update may run beside the round). They are claimed from
  // kSeedHeads counters, a wave starting at one of its own, so that the grid's
  // first claims do not queue up on one line. With more shares than waves a wave
  // whose counter has run out moves on to one that has not.
  const uint32_t parts = nseeds && nseeds < a.crew ? min(a.crew / nseeds, kMaxParts) : 1u;
  const uint32_t total = nseeds * parts;
  if (cr.me >= a.crew && !reserve_joins(a, total, cr.me, bcast64(S.since))) return;
  uint32_t head = cr.me % kSeedHeads;
  bool seeds_left = total > 0;
  uint32_t seen = 0;  // mail taken so far
  if (lane == 0) {
    seen = ld_relaxed(&a.mail[cr.me].mail);
    if (seeds_left) {
      const IdlePlace at = idle_place(a, cr.me);
      atomicOr(&a.idle[at.word].v, 1ull << (at.bit + kIdleGroup));
    }
  }
  seen = bcast(seen);
  uint64_t busy = 0;            // wall-clock ticks spent on tasks
  uint64_t first_t = 0, last_t = 0;  // start of the first task, end of the last
  if (lane < 7) s_rec[wv][lane] = 0;
  for (;;) {
    uint32_t got = 0, slot = 0;
    if (total == 0) break;
    while (seeds_left) {
      if (lane == 0) slot = head + kSeedHeads * atomicAdd(&a.ctl->seed_head[head].v, 1u);
      slot = bcast(slot);
      if (slot < total) {
        got = 2;
        break;
      }
      uint64_t open = 0;
      if (total > a.crew) {
        const uint32_t h = lane % kSeedHeads;
        open = ballot(lane < kSeedHeads && h + kSeedHeads * ld_relaxed(&a.ctl->seed_head[h].v) < total);
      }
      if (open == 0) seeds_left = false;
      else head = (uint32_t)__builtin_ctzll(open >> head ? open >> head << head : open);
    }
    if (!got) {
      if (!wait_for_task(a, cr, seen)) break;
      got = 1;
    }
    // ---- load the task
    const uint64_t t_task = wall_clock64();
    if (first_t == 0) first_t = t_task;
    uint32_t plan, L0, lo, hi, tag, fw = 0, part = 0;
    if (got == 1) {
      const uint32_t word =
          lane < (uint32_t)kTaskWords ? reinterpret_cast<const uint32_t *>(&a.mail[cr.me])[lane] : 0u;
      plan = __builtin_amdgcn_readlane(word, 0);
      L0 = __builtin_amdgcn_readlane(word, 1);
      lo = __builtin_amdgcn_readlane(word, 2);
      hi = __builtin_amdgcn_readlane(word, 3);
      tag = __builtin_amdgcn_readlane(word, 4 + kMaxQ);
      fw = __shfl(word, (int)((lane + 4) & 63));
    } else {
      part = slot / nseeds;
      slot -= part * nseeds;
      plan = a.seed_plan[slot];
      tag = a.seed_tag[slot];
      L0 = 2;
      lo = 0;
      hi = 0xFFFFFFFFu;
      fw = lane == 0 ? a.seed_s[slot] : a.seed_d[slot];
    }
    if (lane == 0) S.tag = tag;
    if (bcast(S.plan) != plan) {
      const Plan &P = a.plans[plan];
      if (lane < (uint32_t)kMaxQ) {
        S.sig[lane] = P.sig[lane];
        S.back[lane] = P.back[lane];
        S.inj[lane] = P.inj[lane];
        S.qv[lane] = P.qv[lane];
        S.lix[lane] = P.lix[lane];
      }
      if (lane == 0) {
        S.n = P.n;
        S.query = P.query;
        S.plan = plan;
      }
    }
    if (lane < L0) {
      S.f[lane] = fw;
      S.fs[lane] = a.g.start[fw];
      S.fd[lane] = a.g.deg[fw];
    }
    if (lane == 0) S.fstate = kFStale;
    wave_sync();
    const uint32_t n = bcast(S.n);
    uint64_t lcount = 0, mbytes = 0;
    uint32_t scanned = 0, loads = 0;  // per lane: source entries read, search loads
    if (L0 >= n) {
      // complete embedding (two-vertex query seeded by its only edge)
      if (lane == 0 && part == 0) lcount = 1;
      if (TUP) emit_tuples(S, a, n - 1, S.f[n - 1], lane == 0 && part == 0);
    } else {
      // a seed expands its partial match here; a donated task continues one
      // whose expansion the donor counted
      if (got == 2 && part == 0) mbytes += list_bytes(S, S.back[L0]);
      init_level(S, a.g, L0, lo, hi);
      if (got == 2 && parts > 1) {
        // the share of the source range, in pieces of what a hand-off is worth:
        // an entry two or more levels above the leaf, 16 one level above it,
        // a chunk of 64 at the leaf
        const uint32_t piece = L0 + 3 <= n ? 1u : L0 + 2 == n ? 16u : 64u;
        const uint32_t len = bcast(S.end[L0]), np = (len + piece - 1) / piece;
        lo = (uint32_t)((uint64_t)np * part / parts) * piece;
        hi = min((uint32_t)((uint64_t)np * (part + 1) / parts) * piece, len);
        wave_sync();
        if (lane == 0) {
          S.pos[L0] = lo;
          S.end[L0] = hi;
        }
        wave_sync();
      }
      uint32_t l = L0;
      // highest position the leaf set F depends on (-1: none)
      int fdep = -1;
      if (n >= 4) {
        const uint32_t dep = (uint32_t)(S.back[n - 1] | S.inj[n - 1]) & ((1u << (n - 2)) - 1u);
        fdep = dep ? 31 - __builtin_clz(dep) : -1;
      }
      uint32_t tick = 0;
      for (;;) {
        if (l == n - 1) {
          // leaf: count every valid image in the remaining source range
          for (;;) {
            if (++tick >= a.donate_every) {
              tick = 0;
              try_donate<CAP>(S, a, L0, l, n, cr);
            }
            const uint32_t p = bcast(S.pos[l]), e = bcast(S.end[l]);
            if (p >= e) break;
            uint32_t w;
            const bool ok = test_chunk(M, a, l, p, e, w, loads);
            scanned += p + lane < e ? 1u : 0u;
            lcount += ok ? 1u : 0u;
            if (TUP) emit_tuples(S, a, l, w, ok);
            wave_sync();
            if (lane == 0) S.pos[l] = p + 64;
            wave_sync();
          }
          if (l == L0) break;
          l--;
          continue;
        }
        const uint32_t ci = bcast(S.ci[l]), cn = bcast(S.cn[l]);
        if (ci < cn) {
          const uint32_t c = (l - 2) * 64 + ci;
          const uint32_t w = bcast(M.cand[c]);
          const uint32_t ws = bcast(M.cst[c]);
          const uint32_t wd = bcast(M.cdg[c]);
          wave_sync();
          if (lane == 0) {
            S.ci[l] = ci + 1;
            S.f[l] = w;
            S.fs[l] = ws;
            S.fd[l] = wd;
            // F depends only on the positions of the leaf's backward and
            // same-label neighbours other than n-2: it stays valid while
            // deeper positions change
            if ((int)l <= fdep) S.fstate = kFStale;
          }
          wave_sync();
          l++;
          mbytes += list_bytes(S, S.back[l]);
          init_level(S, a.g, l, 0, 0xFFFFFFFFu);
          continue;
        }
        if (!TUP && a.leaf_sets && l + 2 == n && bcast(S.fstate) != kFLarge) {
          // one level above the leaf: each lane counts the leaf images of its
          // own candidate against the shared leaf set F, instead of a descent
          // per candidate
          bool large = false, descend = false;
          for (;;) {
            if (++tick >= a.donate_every) {
              tick = 0;
              try_donate<CAP>(S, a, L0, l, n, cr);
            }
            const uint32_t p = bcast(S.pos[l]), e = bcast(S.end[l]);
            if (p >= e) break;
            uint32_t w;
            const bool ok = test_chunk(M, a, l, p, e, w, loads);
            scanned += p + lane < e ? 1u : 0u;
            if (ballot(ok) == 0) {
              wave_sync();
              if (lane == 0) S.pos[l] = p + 64;
              wave_sync();
              continue;
            }
            if (bcast(S.fstate) == kFStale) compute_leaf_set(M, a, l + 1, scanned, loads);
            // backward lists of the leaf other than position n-2, read by a
            // merge for every candidate of this level
            const uint64_t fixed_leaf_bytes = list_bytes(S, S.back[l + 1] & ~(1u << l));  // this lane's share
            if (bcast(S.fstate) == kFLarge) {
              // this chunk and the rest of the level take the descent path
              large = true;
              break;
            }
            bool defer = false, scan = false;
            LeafList ll{nullptr, 0, false};
            uint32_t wdeg = 0, lc = 0;
            if (ok) lc = leaf_count_lane(M, a, l + 1, w, defer, scan, ll, scanned, loads, wdeg);
            // inline work of the lanes up to this one; the first lane past the
            // budget descends, the lanes after it are tested again later
            uint32_t wk = 0;
            if (scan || defer) wk = ll.by_f ? S.fn * search_reads(ll.len) : ll.len;
            const uint32_t incl = wave_incl_sum(wk);
            const uint64_t dm = ballot(wk > 0 && incl > a.leaf_budget);
            const uint32_t k0 = dm ? (uint32_t)__builtin_ctzll(dm) : 64u;
            if (lane >= k0) {
              lc = 0;
              scan = defer = false;
            } else if (ok) {
              mbytes += 4ull * wdeg;
            }
            mbytes += fixed_leaf_bytes * (uint32_t)__popcll(ballot(ok && lane < k0));
            lcount += lc;
            if (a.leaf_segments) lcount += leaf_scan_segments(M, a, l + 1, w, scan, ll, scanned);
            lcount += leaf_count_wave(M, a, l + 1, w, defer, ll, scanned, loads);
            if (dm) {
              // lane k0's candidate as a one-entry chunk at source index p + k0
              const uint32_t w0 = __builtin_amdgcn_readlane(w, k0);
              wave_sync();
              if (lane == 0) {
                const uint32_t c = (l - 2) * 64;
                M.cand[c] = w0;
                M.cst[c] = a.g.start[w0];
                M.cdg[c] = a.g.deg[w0];
                S.cn[l] = 1;
                S.ci[l] = 0;
                S.cbase[l] = p + k0;
                S.cmask[l] = 1;
                S.pos[l] = p + k0 + 1;
              }
              wave_sync();
              descend = true;
              break;
            }
            wave_sync();
            if (lane == 0) S.pos[l] = p + 64;
            wave_sync();
          }
          if (descend) continue;
          if (!large) {
            if (l == L0) break;
            l--;
            continue;
          }
        }
        if (++tick >= a.donate_every) {
          tick = 0;
          try_donate<CAP>(S, a, L0, l, n, cr);
        }
        const uint32_t p = bcast(S.pos[l]), e = bcast(S.end[l]);
        if (p < e) {
          uint32_t w;
          const bool ok = test_chunk(M, a, l, p, e, w, loads);
          scanned += p + lane < e ? 1u : 0u;
          // prefetch the list of every survivor for the descent
          uint32_t ws = 0, wd = 0;
          if (ok) {
            ws = a.g.start[w];
            wd = a.g.deg[w];
          }
          const uint64_t m = ballot(ok);
          wave_sync();
          if (ok) {
            const uint32_t c = (l - 2) * 64 + mbcnt(m);
            M.cand[c] = w;
            M.cst[c] = ws;
            M.cdg[c] = wd;
          }
          if (lane == 0) {
            S.cn[l] = __popcll(m);
            S.ci[l] = 0;
            S.cbase[l] = p;
            S.cmask[l] = m;
            S.pos[l] = p + 64;
          }
          wave_sync();
          continue;
        }
        if (l == L0) break;
        l--;
      }
    }
    const uint64_t tot = wave_sum(lcount);
    if (lane == 0 && tot) {
      const uint32_t tg = S.tag;
      atomicAdd(&a.counts[((size_t)(tg >> 1) * a.nq + S.query) * 2 + (tg & 1)], (unsigned long long)tot);
    }
    const uint64_t sc = wave_sum(scanned), ld = wave_sum(loads), mb = wave_sum(mbytes);
    if (lane == 0) {
      s_rec[wv][4] += sc;
      s_rec[wv][5] += ld;
      s_rec[wv][6] += mb;
    }
    last_t = wall_clock64();
    busy += last_t - t_task;
    if (a.query_busy && lane == 0) atomicAdd(&a.query_busy[S.query], (unsigned long long)(last_t - t_task));
  }
  // the block's record: the time its waves
  // spent on tasks (not waiting), when their first task started and their last
  // ended, and their work
  if (lane == 0) {
    s_rec[wv][0] = busy;
    s_rec[wv][1] = first_t;
    s_rec[wv][2] = last_t;
    s_rec[wv][3] = S.donated;
  }
  __syncthreads();
  if (wv == 0) {
    // a lane per word of the record, so that it leaves as one write over the bus
    unsigned long long x = 0;
    const unsigned long long field = lane;
    if (field == offsetof(BlockRec, first_min) / 8) x = ~0ull;
    for (int w = 0; w < WPB; w++) {
      const unsigned long long *r = s_rec[w];
      const bool act = r[1] != 0;
      switch (field) {
        case offsetof(BlockRec, active) / 8: x += act; break;
        case offsetof(BlockRec, busy) / 8: x += r[0]; break;
        case offsetof(BlockRec, first_min) / 8: x = act ? min(x, r[1]) : x; break;
        case offsetof(BlockRec, first_sum) / 8: x += r[1]; break;
        case offsetof(BlockRec, last_max) / 8: x = max(x, r[2]); break;
        case offsetof(BlockRec, last_sum) / 8: x += r[2]; break;
        case offsetof(BlockRec, donated) / 8: x += r[3]; break;
        case offsetof(BlockRec, scanned) / 8: x += r[4]; break;
        case offsetof(BlockRec, loads) / 8: x += r[5]; break;
        case offsetof(BlockRec, mbytes) / 8: x += r[6]; break;
      }
    }
    if (field == offsetof(BlockRec, epoch) / 8) x = a.epoch;
    if (field == offsetof(BlockRec, nseeds) / 8) x = a.ctl->nseeds.v;
    if (field == offsetof(BlockRec, seed_overflow) / 8) x = a.ctl->seed_overflow.v;
    if (field == offsetof(BlockRec, abort) / 8) x = ld_relaxed(&a.ctl->abort.v);
    if (lane < sizeof(BlockRec) / 8) reinterpret_cast<unsigned long long *>(&a.rec[blockIdx.x])[lane] = x;
  }
}

// Copies every vertex's live list to its new slot (pool growth/compaction).
__global__ __launch_bounds__(256) void k_pool_move(const uint32_t *old_pool, uint32_t *new_pool,
                                                   const uint32_t *old_start, const uint32_t *new_start,
                                                   const uint32_t *deg, uint32_t n) {
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  for (uint32_t v = blockIdx.x * 4 + wv; v < n; v += gridDim.x * 4) {
    const uint32_t d = deg[v];
    const uint32_t *src = old_pool + old_start[v];
    uint32_t *dst = new_pool + new_start[v];
    for (uint32_t j = lane; j < d; j += 64) dst[j] = src[j];
  }
}

template <int WPB>
int max_blocks(uint32_t chunk_levels) {
  int nb = 0;
  const size_t lds = (size_t)WPB * wave_lds_bytes(chunk_levels);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_dfs<WPB, false, false>, WPB * 64, lds) != hipSuccess) return 1;
  return nb > 0 ? nb : 1;
}

// ------------------------------------------------------ graph copy sync

// Bringing the second copy of the graph up to date before an overlapped
// update: instead of copying the whole graph, only what the previous update
// changed is copied from the up-to-date copy `x` to the stale one `y`: the
// touched vertices' slots, degrees and lists, the relabelled vertices' labels and
// the signature rows (k_catch_up), then, once the update has marked its own dirty
// vertices, the other dirty vertices' label-sorted copies and bucket offsets
// (k_sync_sorted). Lists of up to kSyncWave entries are copied by one wave;
// longer ones are queued (queue_big: a block each up to kBlockList entries, the
// whole grid beyond) for k_sync_big.
__global__ __launch_bounds__(256) void k_catch_up(CatchUp c) {
  const uint32_t lane = lane_id();
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nth = (size_t)gridDim.x * blockDim.x;
  for (size_t t = tid >> 6; t < c.ntouched; t += nth >> 6) {
    const uint32_t v = c.touched[t];
    const uint32_t st = c.x.start[v], d = c.x.deg[v];
    if (lane == 0) {
      c.y.start[v] = st;
      c.y.deg[v] = d;
      c.y.cap[v] = c.x.cap[v];
    }
    if (d <= kSyncWave) copy_range(c.x.pool + st, c.y.pool + st, lane, 64, d);
    else if (lane == 0) queue_big(c.q, c.qcap, &c.actl->sync_queued[0], &c.actl->sync_queued[1], d, v);
  }
  for (size_t r = tid; r < c.nrelabeled; r += nth) {
    const uint32_t v = c.relabeled[r];
    c.y.lab[v] = c.x.lab[v];
  }
  size_t i = tid;
  for (; i + 3 * nth < c.nbm; i += 4 * nth) {
    const uint64_t w0 = c.bm_x[i], w1 = c.bm_x[i + nth], w2 = c.bm_x[i + 2 * nth], w3 = c.bm_x[i + 3 * nth];
    c.bm_y[i] = w0;
    c.bm_y[i + nth] = w1;
    c.bm_y[i + 2 * nth] = w2;
    c.bm_y[i + 3 * nth] = w3;
  }
  for (; i < c.nbm; i += nth) c.bm_y[i] = c.bm_x[i];
}

__global__ __launch_bounds__(256) void k_sync_sorted(DevGraph x, DevGraph y, const uint32_t *list,
                                                     const uint32_t *count, const uint8_t *skip, uint32_t *q,
                                                     uint32_t qcap, ApplyCtl *actl) {
  const uint32_t lane = lane_id();
  if (held_up(actl)) return;
  const uint32_t total = *count < x.n ? *count : x.n;
  for (uint32_t t = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; t < total; t += (gridDim.x * blockDim.x) >> 6) {
    const uint32_t v = list[t];
    if (skip[v]) continue;
    const uint32_t st = x.start[v], d = x.deg[v];
    if (d <= kLabelSorted) continue;
    const uint32_t nb = x.nbuckets + 1;
    if (lane < nb) y.loff[(size_t)v * nb + lane] = x.loff[(size_t)v * nb + lane];
    if (d <= kSyncWave) copy_range(x.lpool + st, y.lpool + st, lane, 64, d);
    else if (lane == 0) queue_big(q, qcap, &actl->sync_queued[2], &actl->sync_queued[3], d, v);
  }
}

__global__ __launch_bounds__(256) void k_sync_big(DevGraph x, const uint32_t *from, uint32_t *to, const uint32_t *q,
                                                  uint32_t qcap, const uint32_t *queued) {
  for_big_lists(q, qcap, queued[0], queued[1], [&](uint32_t v, uint32_t first, uint32_t stride) {
    const uint32_t st = x.start[v];
    copy_range(from + st, to + st, first, stride, x.deg[v]);
  });
}

// Blocks for n items, so many a block.
uint32_t blocks_for(size_t n, uint32_t per_block, uint32_t most) {
  const size_t b = (n + per_block - 1) / per_block;
  return b == 0 ? 1u : b < most ? (uint32_t)b : most;
}

}  // namespace

hipError_t launch_small_copy(const SmallCopy &c, hipStream_t s) {
  if (c.words) hipLaunchKernelGGL(k_small_copy, dim3(1), dim3(256), 0, s, c);
  return hipGetLastError();
}

hipError_t launch_array_copies(const ArrayCopies &c, hipStream_t s) {
  size_t most = 0;
  for (uint32_t k = 0; k < c.n; k++) most = std::max(most, c.bytes[k]);
  if (most) hipLaunchKernelGGL(k_array_copies, dim3(blocks_for(most, 4 * 256 * 16, 4096)), dim3(256), 0, s, c);
  return hipGetLastError();
}

hipError_t launch_update_begin(ApplyCtl *actl, const ApplyCtl *from, uint32_t *bctl, const SmallCopy &up,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_update_begin, dim3(1), dim3(256), 0, s, actl, from, bctl, up);
  return hipGetLastError();
}

hipError_t launch_round_begin(ApplyCtl *actl, const SmallCopy &up, hipStream_t s) {
  hipLaunchKernelGGL(k_round_begin, dim3(1), dim3(256), 0, s, actl, up);
  return hipGetLastError();
}

hipError_t launch_apply(const DevGraph &g, const BatchDev &b, uint32_t *scratch, unsigned long long scratch_cap,
                        unsigned long long pool_cap, ApplyCtl *actl, const DirtyArgs &d, size_t max_segs,
                        hipStream_t s) {
  if (b.ntouched == 0) return hipSuccess;
  const dim3 seg_blocks(blocks_for(max_segs, 4, 4096));
  hipLaunchKernelGGL(k_apply_plan, dim3(blocks_for(b.ntouched, kPlanBlock, 4096)), dim3(kPlanBlock), 0, s, g, b, scratch_cap, actl);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_apply_rank, dim3(blocks_for(b.ntouched, kApplyWaves, 4096)), dim3(kApplyWaves * 64), 0, s, g, b,
                     scratch, pool_cap, actl);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_apply_merge, seg_blocks, dim3(256), 0, s, g, b, scratch, (const ApplyCtl *)actl);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_apply_commit, seg_blocks, dim3(256), 0, s, g, b, (const uint32_t *)scratch,
                     (const ApplyCtl *)actl, d, 0);
  return hipGetLastError();
}

hipError_t launch_commit_again(const DevGraph &g, const BatchDev &b, const uint32_t *scratch,
                               unsigned long long pool_cap, ApplyCtl *actl, const DirtyArgs &d, size_t max_segs,
                               hipStream_t s) {
  if (b.ntouched == 0) return hipSuccess;
  hipLaunchKernelGGL(k_apply_slots, dim3(blocks_for(b.ntouched, 256, 4096)), dim3(256), 0, s, g, b, pool_cap, actl);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_apply_commit, dim3(blocks_for(max_segs, 4, 4096)), dim3(256), 0, s, g, b, scratch,
                     (const ApplyCtl *)actl, d, 1);
  return hipGetLastError();
}

hipError_t launch_dirty_compact(const DevGraph &g, const DirtyArgs &d, hipStream_t s) {
  hipLaunchKernelGGL(k_dirty_compact, dim3(blocks_for(g.n, 16 * kCompactBlock, 4096)), dim3(kCompactBlock), 0, s, g, d);
  return hipGetLastError();
}

hipError_t launch_catch_up(const CatchUp &c, uint32_t longest, hipStream_t s) {
  const uint32_t blocks = std::max(blocks_for(c.ntouched, 4, 4096), std::max(blocks_for(c.nrelabeled, 256, 4096),
                                                                            blocks_for(c.nbm, 1024, 4096)));
  hipLaunchKernelGGL(k_catch_up, dim3(blocks), dim3(256), 0, s, c);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || longest <= kSyncWave) return e;
  hipLaunchKernelGGL(k_sync_big, dim3(1024), dim3(256), 0, s, c.x, (const uint32_t *)c.x.pool, c.y.pool,
                     (const uint32_t *)c.q, c.qcap, (const uint32_t *)&c.actl->sync_queued[0]);
  return hipGetLastError();
}

hipError_t launch_sync_sorted(const DevGraph &x, const DevGraph &y, const uint32_t *dirty, const uint32_t *ndirty,
                              const uint8_t *skip, uint32_t *q, uint32_t qcap, ApplyCtl *actl, uint32_t longest,
                              hipStream_t s) {
  if (longest <= kLabelSorted) return hipSuccess;
  hipLaunchKernelGGL(k_sync_sorted, dim3(blocks_for(x.n, 4, 4096)), dim3(256), 0, s, x, y, dirty, ndirty, skip, q, qcap,
                     actl);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || longest <= kSyncWave) return e;
  hipLaunchKernelGGL(k_sync_big, dim3(1024), dim3(256), 0, s, x, (const uint32_t *)x.lpool, y.lpool,
                     (const uint32_t *)q, qcap, (const uint32_t *)&actl->sync_queued[2]);
  return hipGetLastError();
}

hipError_t launch_relabel(const DevGraph &g, const BatchDev &b, const FilterTables &ft,
                          const DirtyArgs &d, size_t max_segs, hipStream_t s) {
  if (b.nrelabel == 0) return hipSuccess;
  hipLaunchKernelGGL(k_relabel, dim3(blocks_for(b.nrelabel, 256, 4096)), dim3(256), 0, s, g, b, d);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_relabel_marks, dim3(blocks_for(max_segs, 4, 4096)), dim3(256), 0, s, g, b, ft, d);
  return hipGetLastError();
}

hipError_t launch_filter_full(const DevGraph &g, const FilterTables &ft, hipStream_t s) {
  const uint32_t groups = (g.n + 63) / 64;
  const uint32_t blocks = (groups + 3) / 4;
  hipLaunchKernelGGL(k_filter_full, dim3(blocks < 8192 ? blocks : 8192), dim3(256), 0, s, g, ft);
  return hipGetLastError();
}

hipError_t launch_filter_dirty(const DevGraph &g, const FilterTables &ft, const DirtyArgs &d, hipStream_t s) {
  hipLaunchKernelGGL(k_filter_light, dim3(blocks_for(g.n, 256, 1024)), dim3(256), 0, s, g, ft, d);
  return hipGetLastError();
}

hipError_t launch_update_small(const DevGraph &g, const BatchDev &b, const FilterTables &ft, const DirtyArgs &d,
                               const SortedBuild &hs, uint32_t *scratch, unsigned long long scratch_cap,
                               unsigned long long pool_cap, uint32_t longest, const SmallCopy &up, ApplyCtl *status,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_update_small, dim3(1), dim3(kOneWaves * 64), 0, s, g, b, ft, d, hs, scratch, scratch_cap,
                     pool_cap, longest > kLabelSorted, up, reinterpret_cast<uint32_t *>(status));
  return hipGetLastError();
}

hipError_t launch_build_reset(const SortedBuild &hs, hipStream_t s) {
  hipLaunchKernelGGL(k_build_reset, dim3(1), dim3(64), 0, s, hs);
  return hipGetLastError();
}

hipError_t launch_lbuild(const DevGraph &g, const FilterTables &ft, const uint32_t *list, const uint32_t *count,
                         const SortedBuild &hs, uint32_t longest, bool filter, hipStream_t s) {
  if (longest <= kLabelSorted) return hipSuccess;
  hipLaunchKernelGGL(k_lbuild_pick, dim3(blocks_for(g.n, 1024, 2048)), dim3(256), 0, s, g, list, count, hs);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_lbuild, dim3(blocks_for(g.n, 4, 2048)), dim3(256), 0, s, g, ft, hs, filter);
  if ((e = hipGetLastError()) != hipSuccess || longest <= kBuildSeg) return e;
  hipLaunchKernelGGL(k_lbuild_starts, dim3(blocks_for(g.n, 4, 1024)), dim3(256), 0, s, g, ft, hs, filter);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_lbuild_place, dim3(blocks_for(g.n, 4, 2048)), dim3(256), 0, s, g, ft.lmap, hs);
  return hipGetLastError();
}

hipError_t launch_seed(const SeedArgs &a, hipStream_t s) {
  const uint32_t nrec = a.nrec[0] + a.nrec[1];
  if (nrec == 0 || a.nplans == 0) return hipSuccess;
  hipLaunchKernelGGL(k_seed, dim3(blocks_for(nrec, 4 * seed_share(nrec), 4096)), dim3(256), 0, s, a);
  return hipGetLastError();
}

namespace {
template <bool CAP>
hipError_t launch_dfs_shape(const DfsArgs &a, uint32_t blocks, uint32_t waves_per_block, uint32_t cl, hipStream_t s) {
  const size_t per = wave_lds_bytes(cl);
  if (a.tuples) {
    hipLaunchKernelGGL((k_dfs<4, true, CAP>), dim3(blocks), dim3(256), 4 * per, s, a, cl);
    return hipGetLastError();
  }
  switch (waves_per_block) {
    case 1: hipLaunchKernelGGL((k_dfs<1, false, CAP>), dim3(blocks), dim3(64), per, s, a, cl); break;
    case 2: hipLaunchKernelGGL((k_dfs<2, false, CAP>), dim3(blocks), dim3(128), 2 * per, s, a, cl); break;
    case 8: hipLaunchKernelGGL((k_dfs<8, false, CAP>), dim3(blocks), dim3(512), 8 * per, s, a, cl); break;
    default: hipLaunchKernelGGL((k_dfs<4, false, CAP>), dim3(blocks), dim3(256), 4 * per, s, a, cl); break;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_dfs(const DfsArgs &a, uint32_t blocks, uint32_t waves_per_block, uint32_t max_query_vertices,
                      hipStream_t s) {
  const uint32_t cl = max_query_vertices > 3 ? max_query_vertices - 3 : 1;
  if (a.donate_cap != kNoDonateCap) return launch_dfs_shape<true>(a, blocks, waves_per_block, cl, s);
  return launch_dfs_shape<false>(a, blocks, waves_per_block, cl, s);
}

uint32_t dfs_lds_bytes_per_wave(uint32_t max_query_vertices) {
  return wave_lds_bytes(max_query_vertices > 3 ? max_query_vertices - 3 : 1);
}

int dfs_max_blocks_per_cu(uint32_t waves_per_block, uint32_t max_query_vertices) {
  const uint32_t cl = max_query_vertices > 3 ? max_query_vertices - 3 : 1;
  switch (waves_per_block) {
    case 1: return max_blocks<1>(cl);
    case 2: return max_blocks<2>(cl);
    case 8: return max_blocks<8>(cl);
    default: return max_blocks<4>(cl);
  }
}

hipError_t launch_ctl_reset(DfsCtl *ctl, unsigned long long *tuple_count, unsigned long long *counts,
                            uint32_t ncounts, IdleWord *idle, uint32_t nidle, const SmallCopy &up, hipStream_t s) {
  hipLaunchKernelGGL(k_ctl_reset, dim3(1), dim3(256), 0, s, ctl, tuple_count, counts, ncounts, idle, nidle, up);
  return hipGetLastError();
}

hipError_t launch_pool_move(const uint32_t *old_pool, uint32_t *new_pool, const uint32_t *old_start,
                            const uint32_t *new_start, const uint32_t *deg, uint32_t n, hipStream_t s) {
  const uint32_t blocks = (n + 3) / 4;
  hipLaunchKernelGGL(k_pool_move, dim3(blocks < 8192 ? blocks : 8192), dim3(256), 0, s, old_pool, new_pool,
                     old_start, new_start, deg, n);
  return hipGetLastError();
}

}  // namespace dsm
