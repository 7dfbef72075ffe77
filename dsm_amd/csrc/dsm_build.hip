// The data graph's adjacency from its edge list, on the device: every edge becomes
// two 64-bit keys (source, target), a radix sort puts them in order, equal
// neighbours are dropped, and the lists go to their slots in the pool. With the
// lists counted, scattered and sorted by one host core, an engine for 2,000,003
// edges on 200,003 vertices took 82.8 ms to make; it takes 4.4 ms this way, most
// of it allocations and the upload of the edges.
//
//   k_csr_keys                          the keys; the first edge out of range
//   k_radix_count / k_scan_* / k_radix_place
//                                       one stable pass of the sort over 8 bits
//   k_unique_count / k_scan_* / k_unique_place
//                                       equal keys dropped
//   k_csr_rows / k_csr_slots / k_scan_* / k_csr_start
//                                       degrees and slots
//   k_csr_fill                          the lists into the pool
//
// And back again, for a copy of the graph: k_degrees / k_scan_* / k_lists pack the
// lists out of their slots.
#include <algorithm>

#include "dsm_device.h"
#include "dsm_internal.h"

namespace dsm {
namespace {

typedef unsigned long long u64;

// Keys per tile: a block of four waves takes one tile, a wave a contiguous quarter
// of it in chunks of 64. A tile's 4,096 keys spread over 256 digits make runs of 16
// keys (128 bytes) on average, so the placing pass writes whole cache lines.
constexpr uint32_t kTileWaves = 4, kTileChunks = 16, kTile = kTileWaves * kTileChunks * 64;
constexpr uint32_t kDigits = 256;
constexpr uint32_t kScanItems = 8, kScanTile = 256 * kScanItems;

__global__ __launch_bounds__(256) void k_csr_keys(const uint32_t *src, const uint32_t *dst, u64 m, uint32_t n,
                                                  uint32_t bits, u64 *keys, CsrCtl *ctl) {
  for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < m; i += gridDim.x * 256ull) {
    u64 a = src[i], b = dst[i];
    if (a >= n || b >= n) {
      atomicMin(&ctl->bad, i);
      a = b = 0;
    }
    reinterpret_cast<ulonglong2 *>(keys)[i] = ulonglong2{a << bits | b, b << bits | a};
  }
}

__global__ __launch_bounds__(256) void k_radix_count(const u64 *keys, u64 count, uint32_t shift, uint32_t tiles,
                                                     u64 *hist) {
  __shared__ uint32_t s_cnt[kTileWaves][kDigits];
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  const u64 at = (u64)blockIdx.x * kTile + wv * (kTileChunks * 64) + lane;
  for (uint32_t k = lane; k < kDigits; k += 64) s_cnt[wv][k] = 0;
  u64 k[kTileChunks];
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) k[u] = at + u * 64 < count ? keys[at + u * 64] : 0;
  wave_sync();
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++)
    if (at + u * 64 < count) atomicAdd(&s_cnt[wv][(uint32_t)(k[u] >> shift) & (kDigits - 1)], 1u);
  __syncthreads();
  const uint32_t d = threadIdx.x;
  hist[(u64)d * tiles + blockIdx.x] = s_cnt[0][d] + s_cnt[1][d] + s_cnt[2][d] + s_cnt[3][d];
}

// The tile's keys, sorted by digit in LDS, to where the scanned counts say. Bound by
// the reads and writes of the keys; the eight ballots per key come second.
__global__ __launch_bounds__(256) void k_radix_place(const u64 *from, u64 *to, u64 count, uint32_t shift,
                                                     uint32_t tiles, const u64 *hist) {
  __shared__ u64 s_key[kTile], s_base[kDigits];
  __shared__ uint32_t s_cnt[kTileWaves][kDigits], s_sum[kTileWaves];
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  const u64 first = (u64)blockIdx.x * kTile;
  const uint32_t here = (uint32_t)min((u64)kTile, count - first), at = wv * (kTileChunks * 64) + lane;
  for (uint32_t k = lane; k < kDigits; k += 64) s_cnt[wv][k] = 0;
  u64 k[kTileChunks];
  uint32_t r[kTileChunks];
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) k[u] = at + u * 64 < here ? from[first + at + u * 64] : 0;
  wave_sync();
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) {
    const bool valid = at + u * 64 < here;
    const uint32_t d = (uint32_t)(k[u] >> shift) & (kDigits - 1);
    uint64_t peers = ballot(valid);
#pragma unroll
    for (uint32_t b = 0; b < 8; b++) {
      const uint64_t m = ballot(d >> b & 1);
      peers &= d >> b & 1 ? m : ~m;
    }
    const uint32_t rank = mbcnt(peers), before = s_cnt[wv][d];
    wave_sync();
    if (valid && rank == 0) s_cnt[wv][d] = before + (uint32_t)__popcll(peers);
    wave_sync();
    r[u] = before + rank;
  }
  __syncthreads();
  // a thread per digit: where each wave's keys of it start in the tile
  {
    const uint32_t d = threadIdx.x;
    uint32_t c[kTileWaves], all = 0;
    for (uint32_t w = 0; w < kTileWaves; w++) {
      c[w] = s_cnt[w][d];
      all += c[w];
    }
    const uint32_t incl = wave_incl_sum(all);
    if (lane == 63) s_sum[wv] = incl;
    __syncthreads();
    uint32_t start = incl - all;
    for (uint32_t w = 0; w < wv; w++) start += s_sum[w];
    s_base[d] = hist[(u64)d * tiles + blockIdx.x] - start;
    for (uint32_t w = 0; w < kTileWaves; w++) {
      s_cnt[w][d] = start;
      start += c[w];
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++)
    if (at + u * 64 < here) s_key[s_cnt[wv][(uint32_t)(k[u] >> shift) & (kDigits - 1)] + r[u]] = k[u];
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < here; i += 256) {
    const u64 key = s_key[i];
    to[s_base[(uint32_t)(key >> shift) & (kDigits - 1)] + i] = key;
  }
}

__device__ __forceinline__ u64 wave_incl_sum64(u64 x) {
  for (uint32_t o = 1; o < 64; o <<= 1) {
    const u64 y = __shfl_up(x, o);
    if (lane_id() >= o) x += y;
  }
  return x;
}

// An exclusive scan of a[count] in three launches: the tiles' sums, the scan of the
// sums by one block, then the tiles again.
__global__ __launch_bounds__(256) void k_scan_sums(const u64 *a, u64 count, u64 *sums) {
  __shared__ u64 s_sum[4];
  const u64 at = (u64)blockIdx.x * kScanTile + threadIdx.x;
  u64 x = 0;
#pragma unroll
  for (uint32_t u = 0; u < kScanItems; u++) x += at + u * 256 < count ? a[at + u * 256] : 0;
  x = wave_incl_sum64(x);
  if (lane_id() == 63) s_sum[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

__global__ __launch_bounds__(1024) void k_scan_top(u64 *sums, uint32_t tiles, u64 *total) {
  __shared__ u64 s_sum[16];
  u64 run = 0;
  for (uint32_t b = 0; b < tiles; b += 1024) {
    const uint32_t i = b + threadIdx.x;
    const u64 x = i < tiles ? sums[i] : 0, incl = wave_incl_sum64(x);
    __syncthreads();
    if (lane_id() == 63) s_sum[threadIdx.x >> 6] = incl;
    __syncthreads();
    u64 before = run;
    for (uint32_t w = 0; w < 16; w++) {
      if (w < threadIdx.x >> 6) before += s_sum[w];
      run += s_sum[w];
    }
    if (i < tiles) sums[i] = before + incl - x;
  }
  if (threadIdx.x == 0 && total) *total = run;
}

__global__ __launch_bounds__(256) void k_scan_tiles(u64 *a, u64 count, const u64 *sums) {
  __shared__ u64 s_sum[4];
  const u64 at = (u64)blockIdx.x * kScanTile + (u64)threadIdx.x * kScanItems;
  u64 x[kScanItems], sum = 0;
#pragma unroll
  for (uint32_t u = 0; u < kScanItems; u++) {
    x[u] = at + u < count ? a[at + u] : 0;
    sum += x[u];
  }
  const u64 incl = wave_incl_sum64(sum);
  if (lane_id() == 63) s_sum[threadIdx.x >> 6] = incl;
  __syncthreads();
  u64 before = sums[blockIdx.x] + incl - sum;
  for (uint32_t w = 0; w < threadIdx.x >> 6; w++) before += s_sum[w];
#pragma unroll
  for (uint32_t u = 0; u < kScanItems; u++) {
    if (at + u < count) a[at + u] = before;
    before += x[u];
  }
}

// The lanes' keys of a tile that differ from the key before them, per chunk.
__device__ __forceinline__ uint32_t new_keys(const u64 *keys, u64 count, u64 at, u64 (&k)[kTileChunks],
                                             uint64_t (&fresh)[kTileChunks]) {
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) {
    const u64 i = at + u * 64;
    k[u] = i < count ? keys[i] : 0;
    fresh[u] = i < count && (i == 0 || keys[i - 1] != k[u]);
  }
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) {
    fresh[u] = ballot(fresh[u] != 0);
    sum += (uint32_t)__popcll(fresh[u]);
  }
  return sum;
}

__global__ __launch_bounds__(256) void k_unique_count(const u64 *keys, u64 count, u64 *tile_sums) {
  __shared__ uint32_t s_sum[kTileWaves];
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  u64 k[kTileChunks];
  uint64_t fresh[kTileChunks];
  const uint32_t sum = new_keys(keys, count, (u64)blockIdx.x * kTile + wv * (kTileChunks * 64) + lane, k, fresh);
  if (lane == 0) s_sum[wv] = sum;
  __syncthreads();
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

__global__ __launch_bounds__(256) void k_unique_place(const u64 *keys, u64 *to, u64 count, const u64 *tile_sums) {
  __shared__ uint32_t s_sum[kTileWaves];
  const uint32_t wv = threadIdx.x >> 6, lane = lane_id();
  u64 k[kTileChunks];
  uint64_t fresh[kTileChunks];
  const uint32_t sum = new_keys(keys, count, (u64)blockIdx.x * kTile + wv * (kTileChunks * 64) + lane, k, fresh);
  if (lane == 0) s_sum[wv] = sum;
  __syncthreads();
  u64 p = tile_sums[blockIdx.x];
  for (uint32_t w = 0; w < wv; w++) p += s_sum[w];
#pragma unroll
  for (uint32_t u = 0; u < kTileChunks; u++) {
    if (fresh[u] >> lane & 1) to[p + mbcnt(fresh[u])] = k[u];
    p += (uint32_t)__popcll(fresh[u]);
  }
}

// begin[v] and, for now in deg[v], the end of v's keys (vertices without any keep
// deg 0).
__global__ __launch_bounds__(256) void k_csr_rows(const u64 *keys, const CsrCtl *ctl, uint32_t bits, uint32_t *begin,
                                                  uint32_t *deg) {
  const u64 count = ctl->unique;
  for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < count; i += gridDim.x * 256ull) {
    const uint32_t v = (uint32_t)(keys[i] >> bits);
    if (i == 0 || (uint32_t)(keys[i - 1] >> bits) != v) begin[v] = (uint32_t)i;
    if (i + 1 == count || (uint32_t)(keys[i + 1] >> bits) != v) deg[v] = (uint32_t)(i + 1);
  }
}

// Degrees, and slots with a quarter of the degree and four entries to spare.
__global__ __launch_bounds__(256) void k_csr_slots(uint32_t n, const uint32_t *begin, uint32_t *deg, uint32_t *cap,
                                                   u64 *slot, CsrCtl *ctl) {
  __shared__ uint32_t s_most;
  if (threadIdx.x == 0) s_most = 0;
  __syncthreads();
  for (u64 v = blockIdx.x * 256ull + threadIdx.x; v < n; v += gridDim.x * 256ull) {
    const uint32_t end = deg[v], d = end ? end - begin[v] : 0u, c = d + d / 4 + 4;
    deg[v] = d;
    cap[v] = c;
    slot[v] = c;
    atomicMax(&s_most, d);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_most) atomicMax(&ctl->max_deg, s_most);
}

__global__ __launch_bounds__(256) void k_csr_start(uint32_t n, const u64 *slot, uint32_t *start) {
  for (u64 v = blockIdx.x * 256ull + threadIdx.x; v < n; v += gridDim.x * 256ull) start[v] = (uint32_t)slot[v];
}

__global__ __launch_bounds__(256) void k_csr_fill(const u64 *keys, const CsrCtl *ctl, uint32_t bits,
                                                  const uint32_t *begin, const uint32_t *start, uint32_t *pool) {
  const u64 count = ctl->unique, mask = (1ull << bits) - 1;
  for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < count; i += gridDim.x * 256ull) {
    const u64 k = keys[i];
    const uint32_t v = (uint32_t)(k >> bits);
    pool[start[v] + (uint32_t)(i - begin[v])] = (uint32_t)(k & mask);
  }
}

__global__ __launch_bounds__(256) void k_degrees(uint32_t n, const uint32_t *deg, u64 *off) {
  for (u64 v = blockIdx.x * 256ull + threadIdx.x; v <= n; v += gridDim.x * 256ull) off[v] = v < n ? deg[v] : 0;
}

// The lists one after the other, a thread per entry: its vertex is found in the
// offsets. Some 20 us for 2,000,000 entries, whose copy to the host takes 20 times
// as long.
__global__ __launch_bounds__(256) void k_lists(uint32_t n, const u64 *off, const uint32_t *start, const uint32_t *pool,
                                               u64 total, uint32_t *out) {
  for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < total; i += gridDim.x * 256ull) {
    uint32_t lo = 0, hi = n;  // off[lo] <= i < off[hi]
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (off[mid] <= i) lo = mid;
      else hi = mid;
    }
    out[i] = pool[start[lo] + (uint32_t)(i - off[lo])];
  }
}

uint32_t tiles_of(u64 count) { return (uint32_t)((count + kTile - 1) / kTile); }
uint32_t grid_of(u64 items) { return (uint32_t)std::min<u64>(std::max<u64>((items + 255) / 256, 1), 8192); }

hipError_t scan(u64 *a, u64 count, u64 *sums, u64 *total, hipStream_t s) {
  const uint32_t tiles = (uint32_t)((count + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_scan_sums, dim3(tiles), dim3(256), 0, s, a, count, sums);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, sums, tiles, total);
  hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(256), 0, s, a, count, sums);
  return hipGetLastError();
}

}  // namespace

size_t csr_scan_words(size_t count) { return std::max<size_t>((size_t)tiles_of(count) * kDigits, 1); }
size_t csr_sum_words(size_t items) { return (items + kScanTile - 1) / kScanTile + 1; }

hipError_t launch_csr_keys(const uint32_t *src, const uint32_t *dst, size_t m, uint32_t n, uint32_t bits, u64 *keys,
                           CsrCtl *ctl, hipStream_t s) {
  hipLaunchKernelGGL(k_csr_keys, dim3(grid_of(m)), dim3(256), 0, s, src, dst, (u64)m, n, bits, keys, ctl);
  return hipGetLastError();
}

hipError_t launch_radix_pass(const u64 *from, u64 *to, size_t count, uint32_t shift, u64 *hist, u64 *sums,
                             hipStream_t s) {
  const uint32_t tiles = tiles_of(count);
  hipLaunchKernelGGL(k_radix_count, dim3(tiles), dim3(256), 0, s, from, (u64)count, shift, tiles, hist);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || (e = scan(hist, (u64)tiles * kDigits, sums, nullptr, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_radix_place, dim3(tiles), dim3(256), 0, s, from, to, (u64)count, shift, tiles, hist);
  return hipGetLastError();
}

hipError_t launch_csr_unique(const u64 *from, u64 *to, size_t count, u64 *hist, u64 *sums, CsrCtl *ctl,
                             hipStream_t s) {
  const uint32_t tiles = tiles_of(count);
  hipLaunchKernelGGL(k_unique_count, dim3(tiles), dim3(256), 0, s, from, (u64)count, hist);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || (e = scan(hist, tiles, sums, &ctl->unique, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_unique_place, dim3(tiles), dim3(256), 0, s, from, to, (u64)count, hist);
  return hipGetLastError();
}

hipError_t launch_csr_slots(const u64 *keys, size_t count, uint32_t n, uint32_t bits, uint32_t *begin, uint32_t *deg,
                            uint32_t *cap, uint32_t *start, u64 *slot, u64 *sums, CsrCtl *ctl, hipStream_t s) {
  if (count)
    hipLaunchKernelGGL(k_csr_rows, dim3(grid_of(count)), dim3(256), 0, s, keys, ctl, bits, begin, deg);
  hipLaunchKernelGGL(k_csr_slots, dim3(grid_of(n)), dim3(256), 0, s, n, begin, deg, cap, slot, ctl);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || (e = scan(slot, n, sums, &ctl->total, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_csr_start, dim3(grid_of(n)), dim3(256), 0, s, n, slot, start);
  return hipGetLastError();
}

hipError_t launch_csr_fill(const u64 *keys, size_t count, uint32_t bits, const uint32_t *begin, const uint32_t *start,
                           uint32_t *pool, const CsrCtl *ctl, hipStream_t s) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(k_csr_fill, dim3(grid_of(count)), dim3(256), 0, s, keys, ctl, bits, begin, start, pool);
  return hipGetLastError();
}

hipError_t launch_graph_offsets(uint32_t n, const uint32_t *deg, u64 *off, u64 *sums, hipStream_t s) {
  hipLaunchKernelGGL(k_degrees, dim3(grid_of(n + 1ull)), dim3(256), 0, s, n, deg, off);
  hipError_t e = hipGetLastError();
  return e != hipSuccess ? e : scan(off, n + 1ull, sums, nullptr, s);
}

hipError_t launch_graph_lists(uint32_t n, const u64 *off, const uint32_t *start, const uint32_t *pool, size_t total,
                              uint32_t *out, hipStream_t s) {
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(k_lists, dim3(grid_of(total)), dim3(256), 0, s, n, off, start, pool, (u64)total, out);
  return hipGetLastError();
}

}  // namespace dsm
