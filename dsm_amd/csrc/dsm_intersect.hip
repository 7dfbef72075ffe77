// Sorted-set intersection on the device with the DFS's own membership test
// (window_member: a cooperative 32-ary bounds search for the window the 64
// lanes' values span, then LDS-staged or in-place binary searches). The
// reference's counterpart is intersect (gpu_match.cu:21-94), which the DFS
// calls with a lane per element of the first set. dsm_intersect_sorted is the
// entry point; it lets the primitive be checked against a set intersection on
// its own, outside the DFS.
#include <algorithm>
#include <memory>
#include <mutex>
#include <new>

#include "../../include/dsm.h"
#include "dsm_device.h"
#include "dsm_internal.h"

namespace dsm {
namespace {

constexpr int kIntersectWaves = 4;
constexpr uint32_t kBadInput = 0xFFFFFFFFu;  // in place of the result's size: inputs not in order

// *bad = 1 unless both inputs are strictly ascending and end below 0xFFFFFFFF; it
// must be clear. (The host's loop over 5,000,000 entries took half of the 2.0 ms of
// 1,000,000 x 4,000,003; 1.0 ms this way.)
__global__ void k_check_clear(uint32_t *bad) { *bad = 0; }
__global__ __launch_bounds__(256) void k_check_sorted(const uint32_t *A, uint32_t na, const uint32_t *B, uint32_t nb,
                                                      uint32_t *bad) {
  const uint64_t total = (uint64_t)na + nb;
  bool wrong = false;
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < total; i += gridDim.x * 256ull) {
    const bool first = i < na;
    const uint32_t *p = first ? A + i : B + (i - na);
    const bool last = first ? i + 1 == na : i + 1 == total;
    wrong |= last ? *p == 0xFFFFFFFFu : p[0] >= p[1];
  }
  if (ballot(wrong) && lane_id() == 0) *bad = 1;
}

// A wave per 64-entry chunk of A: the chunk's members of B, in order, at
// hits[chunk * 64 ..] and their number at cnt[chunk]; none of it if the inputs are
// bad.
__global__ __launch_bounds__(kIntersectWaves * 64) void k_intersect(const uint32_t *A, uint32_t na, const uint32_t *B,
                                                                    uint32_t nb, uint32_t *hits, uint32_t *cnt,
                                                                    const uint32_t *bad) {
  __shared__ uint32_t win[kIntersectWaves][kWin];
  const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
  const uint32_t nch = (na + 63) / 64;
  if (*bad) return;
  for (uint32_t c = blockIdx.x * kIntersectWaves + wv; c < nch; c += gridDim.x * kIntersectWaves) {
    const uint32_t i = c * 64 + lane;
    const bool in = i < na;
    const uint32_t w = in ? A[i] : 0xFFFFFFFFu;
    uint32_t loads = 0;
    const bool ok = window_member(B, nb, w, in, win[wv], loads);
    const uint64_t m = ballot(ok);
    if (ok) hits[(size_t)c * 64 + mbcnt(m)] = w;
    if (lane == 0) cnt[c] = (uint32_t)__popcll(m);
  }
}

// Exclusive prefix of cnt[0, nch) into off, the total at *total (one block), which
// said before whether the inputs are bad: kBadInput then.
__global__ __launch_bounds__(1024) void k_chunk_offsets(const uint32_t *cnt, uint32_t nch, uint32_t *off,
                                                        uint32_t *total) {
  __shared__ uint32_t s_sum[16];
  uint32_t run = 0;
  const bool bad = *total != 0;
  if (bad) nch = 0;
  __syncthreads();
  for (uint32_t base = 0; base < nch; base += 1024) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t x = i < nch ? cnt[i] : 0u, incl = wave_incl_sum(x);
    __syncthreads();  // the previous sums are no longer read
    if (lane_id() == 63) s_sum[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t before = run;
    for (uint32_t w = 0; w < 16; w++) {
      if (w < threadIdx.x >> 6) before += s_sum[w];
      run += s_sum[w];
    }
    if (i < nch) off[i] = before + incl - x;
  }
  if (threadIdx.x == 0) *total = bad ? kBadInput : run;
}

// Chunk c's members (hits[c * 64 ..], cnt[c] of them) to res[off[c] ..].
__global__ __launch_bounds__(256) void k_chunk_gather(const uint32_t *hits, const uint32_t *cnt,
                                                      const uint32_t *off, uint32_t nch, const uint32_t *total,
                                                      uint32_t *res) {
  const uint32_t lane = lane_id();
  if (*total == kBadInput) return;
  for (uint32_t c = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; c < nch; c += (gridDim.x * blockDim.x) >> 6)
    if (lane < cnt[c]) res[off[c] + lane] = hits[(size_t)c * 64 + lane];
}

// The whole intersection by one block, a wave per chunk, 16 chunks at a time:
// their number to *total, the members to res. For a short A, where the two
// launches and the trip through memory between them cost more than the search.
// With `checked`, *total says before whether the inputs are bad: kBadInput then.
constexpr uint32_t kShortWaves = 16;
__global__ __launch_bounds__(kShortWaves * 64) void k_intersect_short(const uint32_t *A, uint32_t na,
                                                                      const uint32_t *B, uint32_t nb, bool checked,
                                                                      uint32_t *total, uint32_t *res) {
  __shared__ uint32_t win[kShortWaves][kWin], s_cnt[kShortWaves];
  const uint32_t lane = lane_id(), wv = bcast(threadIdx.x >> 6);
  uint32_t run = 0;
  const bool bad = checked && *total != 0;
  if (bad) na = 0;
  __syncthreads();
  for (uint32_t base = 0; base < na; base += kShortWaves * 64) {
    const uint32_t i = base + threadIdx.x;
    const bool in = i < na;
    const uint32_t w = in ? A[i] : 0xFFFFFFFFu;
    uint32_t loads = 0;
    const bool ok = window_member(B, nb, w, in, win[wv], loads);
    const uint64_t m = ballot(ok);
    __syncthreads();  // the previous counts are no longer read
    if (lane == 0) s_cnt[wv] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t at = run;
    for (uint32_t k = 0; k < kShortWaves; k++) {
      if (k < wv) at += s_cnt[k];
      run += s_cnt[k];
    }
    if (ok) res[at + mbcnt(m)] = w;
  }
  if (threadIdx.x == 0) *total = bad ? kBadInput : run;
}

}  // namespace

// Inputs of the intersection entry points: strictly ascending, no 0xFFFFFFFF.
bool sorted_set(const uint32_t *a, uint32_t n) {
  for (uint32_t i = 0; i < n; i++) {
    if (a[i] == 0xFFFFFFFFu) return false;
    if (i && a[i] <= a[i - 1]) return false;
  }
  return true;
}

namespace {

// Calls that are not long. At most kShortA entries of A go to k_intersect_short (two
// rounds of its block); inputs of at most kShortCheck entries together are checked on
// the host. Inputs of at most `staged` entries together go up in one copy, the word that
// says whether they are in order with them, and results of at most half as many come
// back in one copy with their number: a copy costs some 8 us, however small, and the
// release of device memory 25 more once a call has sent eight copies and launches. Of
// more entries, the copy into the staging buffer costs more than that.
// 1,000 x 3,000 entries: 67 us with a copy per array and three launches, 36 with one of
// each. With the device memory allocated, 5,000 x 5,000: 113 us with a copy per array
// and five launches, 68 in six steps; 40,000 x 40,000 116 and 69, 130,000 x 130,000 211
// and 154, 132,000 x 132,000 (unstaged) 187. In the fixed array, without that release:
// 65,000 x 65,000 89 and 82 us, 80,000 x 80,000 96 and 92, 130,000 x 130,000 112 and 123.
constexpr uint32_t kShortA = 2048, kShortCheck = 8192, kStaged = 262144, kStagedFixed = 131072;

// kStaged + 1 words of the calling thread, or null (calls of at most kShortCheck entries
// have theirs on the stack). Kept until the thread ends: fresh pages would cost each call
// more than the copies it saves.
uint32_t *staging() {
  static thread_local std::unique_ptr<uint32_t[]> words;
  if (!words) words.reset(new (std::nothrow) uint32_t[kStaged + 1]);
  return words.get();
}

uint32_t chunks_of(uint32_t na) { return (na + 63) / 64; }

// Words of device memory: a | b | total | result | hits (64 per chunk) | cnt | off
size_t words_of(uint32_t na, uint32_t nb) {
  const size_t nch = chunks_of(na);
  return (size_t)na + nb + nch * 64 + 2 * nch + 1 + std::min(na, nb);
}

// a and b, not empty, intersected in the words_of(na, nb) words at base; kBadInput
// as the size if they are not in order, which the device checks past kShortCheck entries.
hipError_t intersect_in(uint32_t *base, const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb,
                        uint32_t staged, uint32_t *out, uint32_t *num_out) {
  const uint32_t nch = chunks_of(na), most = std::min(na, nb);
  uint32_t *dA = base, *dB = dA + na, *dT = dB + nb, *dR = dT + 1, *dH = dR + most, *dC = dH + (size_t)nch * 64,
           *dO = dC + nch;
  const size_t both = (size_t)na + nb;
  const bool check = both > kShortCheck;
  uint32_t few[kShortCheck + 1];
  uint32_t *buf = !check ? few : most <= staged / 2 ? staging() : nullptr;
  hipError_t e;
  if (buf && both <= staged) {
    std::copy(a, a + na, buf);
    std::copy(b, b + nb, buf + na);
    // the word only where it is looked at: 1,000 x 3,000 entries take 0.8 us longer with it
    const size_t flag = check || na > kShortA;
    buf[both] = 0;
    if ((e = hipMemcpy(dA, buf, (both + flag) * 4, hipMemcpyHostToDevice)) != hipSuccess) return e;
  } else {
    if ((e = hipMemcpy(dA, a, (size_t)na * 4, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(dB, b, (size_t)nb * 4, hipMemcpyHostToDevice)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_check_clear, dim3(1), dim3(1), 0, nullptr, dT);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (check) {
    const uint32_t blocks = (uint32_t)std::min<size_t>(((size_t)na + nb + 255) / 256, 2048);
    hipLaunchKernelGGL(k_check_sorted, dim3(blocks), dim3(256), 0, nullptr, dA, na, dB, nb, dT);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (na <= kShortA) {
    hipLaunchKernelGGL(k_intersect_short, dim3(1), dim3(kShortWaves * 64), 0, nullptr, dA, na, dB, nb, check, dT, dR);
  } else {
    const uint32_t blocks = (nch + kIntersectWaves - 1) / kIntersectWaves;
    hipLaunchKernelGGL(k_intersect, dim3(std::min(blocks, 2048u)), dim3(kIntersectWaves * 64), 0, nullptr, dA, na, dB,
                       nb, dH, dC, dT);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_chunk_offsets, dim3(1), dim3(1024), 0, nullptr, dC, nch, dO, dT);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_chunk_gather, dim3(std::min((nch + 3) / 4, 2048u)), dim3(256), 0, nullptr, dH, dC, dO, nch,
                       dT, dR);
  }
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (buf) {
    if ((e = hipMemcpy(buf, dT, ((size_t)most + 1) * 4, hipMemcpyDeviceToHost)) != hipSuccess) return e;
    *num_out = buf[0];
    if (buf[0] != kBadInput) std::copy(buf + 1, buf + 1 + buf[0], out);
    return hipSuccess;
  }
  uint32_t total = 0;
  if ((e = hipMemcpy(&total, dT, 4, hipMemcpyDeviceToHost)) != hipSuccess) return e;
  if (total && total != kBadInput &&
      (e = hipMemcpy(out, dR, (size_t)total * 4, hipMemcpyDeviceToHost)) != hipSuccess)
    return e;
  *num_out = total;
  return hipSuccess;
}

}  // namespace
}  // namespace dsm

using namespace dsm;

namespace {

int not_sorted(const char *who) {
  set_global_error("%s: inputs must be strictly ascending and below 0xFFFFFFFF", who);
  return DSM_EINVAL;
}

// Arguments that settle the call: DSM_EINVAL, or DSM_OK with *num_out = 0; else 1.
// Inputs that need the device's check are looked at here only if `all`.
int settled(const char *who, const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb, const uint32_t *out,
            uint32_t *num_out, bool all) {
  if (!num_out || (na && !a) || (nb && !b) || (na && nb && !out)) {
    set_global_error("%s: null argument", who);
    return DSM_EINVAL;
  }
  const bool none = na == 0 || nb == 0;
  if ((none || all || (size_t)na + nb <= kShortCheck) && (!sorted_set(a, na) || !sorted_set(b, nb)))
    return not_sorted(who);
  if (!none) return 1;
  *num_out = 0;
  return DSM_OK;
}

// The call's end: what intersect_in (or an allocation before it) gave.
int finished(const char *who, hipError_t e, const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb,
             uint32_t size, uint32_t *num_out) {
  if (e == hipSuccess && size == kBadInput) return not_sorted(who);
  // bad inputs are bad inputs, also where there is no device to say so
  if (e != hipSuccess && (!sorted_set(a, na) || !sorted_set(b, nb))) return not_sorted(who);
  *num_out = e == hipSuccess ? size : 0;
  if (e == hipSuccess) return DSM_OK;
  set_global_error("%s failed: %s", who, hipGetErrorString(e));
  return DSM_EDEVICE;
}

}  // namespace

extern "C" int dsm_intersect_sorted(int device, const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb,
                                    uint32_t *out, uint32_t *num_out) {
  const char *who = "dsm_intersect_sorted";
  if (int rc = settled(who, a, na, b, nb, out, num_out, false); rc <= 0) return rc;
  uint32_t *base = nullptr, size = 0;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = hipMalloc(&base, words_of(na, nb) * 4);
  if (e == hipSuccess) e = intersect_in(base, a, na, b, nb, kStaged, out, &size);
  if (base) (void)hipFree(base);
  return finished(who, e, a, na, b, nb, size, num_out);
}

// ------------------------------------------------------------------------
// dsm_intersect_sorted_noalloc: the same intersection without any device
// allocation, for callers that cannot allocate (code under HIP graph capture,
// tight serving loops). Its device memory is one file-scope array per GPU,
// `scratch`, of kScratchWords words; inputs, per-chunk results, their prefix
// offsets and the compacted output all live in it. The host reaches it through
// the address hipGetSymbolAddress returns for the current device (the array's
// name is only a host-side stand-in). Every call on one GPU shares that GPU's
// array, so calls that overlap on one GPU race; nothing in it needs clearing
// (every word a call reads was written by that call).

namespace dsm {
namespace {

constexpr size_t kScratchWords = size_t(1) << 22;  // 16 MiB per GPU
static __device__ __align__(256) uint32_t scratch[kScratchWords];

constexpr int kMaxDevices = 64;
uint32_t *g_scratch[kMaxDevices] = {};
std::once_flag g_scratch_once[kMaxDevices];
hipError_t g_scratch_rc[kMaxDevices] = {};

// The array's address on `device` (current), looked up once per device.
hipError_t scratch_of(int device, uint32_t **out) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::call_once(g_scratch_once[device], [device]() {
    void *p = nullptr;
    g_scratch_rc[device] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (g_scratch_rc[device] == hipSuccess) g_scratch[device] = static_cast<uint32_t *>(p);
  });
  *out = g_scratch[device];
  return g_scratch_rc[device];
}

}  // namespace
}  // namespace dsm

extern "C" int dsm_intersect_sorted_noalloc(int device, const uint32_t *a, uint32_t na, const uint32_t *b,
                                            uint32_t nb, uint32_t *out, uint32_t *num_out) {
  const char *who = "dsm_intersect_sorted_noalloc";
  const size_t need = words_of(na, nb);
  if (int rc = settled(who, a, na, b, nb, out, num_out, need > kScratchWords); rc <= 0) return rc;
  if (need > kScratchWords) {
    *num_out = 0;
    set_global_error("dsm_intersect_sorted_noalloc: %zu scratch words needed, %zu available (na + nb + 66 per "
                     "64 entries of a + min(na, nb) + 1)", need, kScratchWords);
    return DSM_ELIMIT;
  }
  uint32_t *base = nullptr, size = 0;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = scratch_of(device, &base);
  if (e == hipSuccess) e = intersect_in(base, a, na, b, nb, kStagedFixed, out, &size);
  return finished(who, e, a, na, b, nb, size, num_out);
}
