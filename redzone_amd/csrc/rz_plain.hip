// rz_plain.hip -- Redzone O(k) removal from one list on gfx950.
//
// The removal list R (k entries) pairs with the red zone Z = A[n-k, n): pair i
// moves Z[i] into hole R[i].  Three dependent steps (bodies in
// rz_redzone_dev.hpp):
//
//   1. mark   every R[i] >= n-k kills tail item R[i]-(n-k): one bit in a k-bit
//             tail bitmap (relaxed atomicOr).  Replaces the sentinel write of
//             redzone.hxx:698-707, so no payload value is reserved.
//   2. move   R is cut into slices of L pairs, one workgroup each.  A
//             workgroup loads its R, Z and bitmap words coalesced, classifies
//             every pair with two 64-lane ballots, and ranks the orphans of its
//             slice in i order with one LDS scan per step (redzone.hxx:714-822
//             does two block scans per step on 32-lane warps).  Moves go
//             straight to their holes; dest orphans go to the slice's own part
//             of R, source orphans to the slice's own part of Z.  The slice's
//             bitmap words are cleared after use, so the bitmap is zero again
//             for the next call without a memset.
//   3. pair   every workgroup scans the per-slice orphan counts in LDS and
//             pairs the t-th dest orphan with the t-th source orphan
//             (redzone.hxx:834-934).  Orphans are ordered by slice then by i,
//             so the result is the canonical one for every launch shape.
//
// Launch variants: (0) one kernel per step on the caller's stream, the kernel
// boundary being the grid-wide barrier; (1) one cooperative kernel with
// in-kernel barriers made of relaxed atomics (RemoveFromList_GPUWide's
// structure, redzone.hxx:626-941); (2) the persistent work-queue kernel of
// rz_batch.hip with a single list; (3) one ordered launch, roles by workgroup
// id; (4) mark, then one kernel that moves and pairs orphans through a
// decoupled look-back and per-rank exchange words (rz_move_pair); (6) the same
// in one launch; (7) one launch of independent workgroups for small k
// (rz_direct).
//
// Contract violations (duplicates, out-of-range indices) never cause an
// out-of-bounds access: marks are taken only for indices inside the tail,
// moves only into holes below n-k, and pairing stops at the smaller orphan
// total (a mismatch sets an error bit in the control block).
#include <type_traits>

#include "../../include/redzone_device.h"
#include "rz_fused_dev.hpp"
#include "rz_redzone_dev.hpp"
#include "rz_rules.hpp"

namespace rz {

// The mark step for callers that mark into their own bitmap (rz_mark_removals),
// written with the public producer helper.
__global__ __launch_bounds__(256) void rz_mark_removals_kernel(const int32_t* __restrict__ R, int64_t n, int64_t k,
                                                                uint32_t* __restrict__ bits) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < k; i += (int64_t)gridDim.x * 256ll)
    rz_mark_removal(bits, R[i], n, k);
}

rz_status launch_mark_removals(rz_ctx* ctx, const int32_t* R, int64_t n, int64_t k, uint32_t* bits, hipStream_t s) {
  if (k == 0) return RZ_OK;
  const int64_t g = (k + 1023) / 1024;
  const int64_t cap = (int64_t)ctx->cu_count * 8;
  hipLaunchKernelGGL(rz_mark_removals_kernel, dim3((uint32_t)(g < cap ? g : cap)), dim3(256), 0, s, R, n, k, bits);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

template <bool STATS>
__global__ __launch_bounds__(256) void rz_mark_tail(const int32_t* __restrict__ R, uint32_t k, uint32_t sZ,
                                                     uint32_t* __restrict__ bits, uint64_t* __restrict__ stat_tail) {
  mark_body<STATS>(R, k, k, sZ, bits, stat_tail, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u);
}

// Sorted removal list: the removals that fall in the red zone are R's suffix.
// Workgroup w takes the chunk R[w*C, (w+1)*C) and leaves at once when the
// chunk's last entry is below the red zone, so only the suffix is read.
constexpr uint32_t kSortedChunk = 4096;
__global__ __launch_bounds__(256) void rz_mark_tail_sorted(const int32_t* __restrict__ R, uint32_t k, uint32_t sZ,
                                                            uint32_t* __restrict__ bits) {
  const uint32_t lo = blockIdx.x * kSortedChunk;
  const uint32_t hi = min(lo + kSortedChunk, k);
  if ((uint32_t)R[hi - 1] < sZ) return;  // uniform across the workgroup
  mark_body<false>(R + lo, hi - lo, k, sZ, bits, nullptr, threadIdx.x, 256u);
}

// Workgroup (range, chunk): the marks of one range of the tail among one chunk
// of the removals, ranges of a chunk side by side.
__global__ __launch_bounds__(1024) void rz_mark_ranges(const int32_t* __restrict__ R, uint32_t k, uint32_t sZ,
                                                       uint32_t* __restrict__ bits, uint32_t ranges, uint32_t span,
                                                       uint32_t chunk) {
  extern __shared__ uint32_t s_orph[];
  const uint32_t lo = blockIdx.x % ranges * span, a = blockIdx.x / ranges * chunk;
  mark_range<1024, false, 16>(R, a, min(a + chunk, k), sZ, lo, min(span, k - lo), false, s_orph, bits);
}

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_move(T* __restrict__ A, const int32_t* __restrict__ R,
                                               int32_t* __restrict__ Rd, uint32_t k, uint32_t sZ, uint32_t L,
                                               uint32_t* __restrict__ bits, uint64_t* __restrict__ counts) {
  __shared__ MoveShared<WG, IPT> sh;
  move_slice<T, WG, IPT, false>(A, R, Rd, k, sZ, L, blockIdx.x, bits, counts, sh);
}

template <typename T>
__global__ __launch_bounds__(256) void rz_pair(T* __restrict__ A, const int32_t* __restrict__ Rd, uint32_t k, uint32_t sZ,
                                                uint32_t L, uint32_t ns, const uint64_t* __restrict__ counts,
                                                uint32_t* __restrict__ ctrl, int stats) {
  __shared__ PairShared<256, kMaxSlices> sh;
  pair_body<T, 256, kMaxSlices, false>(A, Rd, k, sZ, L, ns, counts, ctrl, stats, blockIdx.x, gridDim.x, sh);
}

// ---------------------------------------------------------------------------
// fused move + pair (variant 4): mark, then one kernel that moves and pairs
// (body: move_pair_core, rz_fused_dev.hpp).  The status words live in two
// halves of kMaxSlices used on alternate calls (parity of the call epoch,
// which the last workgroup to leave bumps for the next call); a call zeroes
// the half it does not use, so the next call starts from zeros.  The epoch is
// also the exchange words' tag.
// ---------------------------------------------------------------------------
// COH: the bitmap was marked in the same launch (rz_mark_move_pair): after the
// first step's loads of R and the red zone, wait until the mark workgroups
// have raised the ready word (this call's epoch + 1), then read bitmap words
// with coherent loads.
template <typename T, int WG, int IPT, bool COH>
__device__ __forceinline__ void move_pair_body(T* __restrict__ A, const int32_t* __restrict__ R, uint32_t k,
                                               uint32_t sZ, uint32_t L, uint32_t ns, uint32_t* __restrict__ bits,
                                               uint64_t* __restrict__ mstatus, uint64_t* __restrict__ slots,
                                               uint32_t slot_cap, uint32_t* __restrict__ ctrl, int stats,
                                               int early, uint32_t slice, uint32_t backoff,
                                               uint32_t* __restrict__ err_out, uint64_t* __restrict__ stamps,
                                               const T* __restrict__ add = nullptr, uint32_t split = 0xffffffffu) {
  const int tid = threadIdx.x;
  // RZ_PROFILE: thread 0 stamps the wall clock at each stage boundary
  uint64_t* const my_stamps = stamps ? stamps + (size_t)blockIdx.x * kStampsPerGroup : nullptr;
  if (my_stamps && tid == 0) my_stamps[kStampStart] = wall_clock64();
  const uint32_t epoch = ld_relaxed(&ctrl[kCtrlMoveEpoch]);
  uint64_t* __restrict__ st = mstatus + (size_t)(epoch & 1u) * kMaxSlices;
  {
    uint64_t* other = mstatus + (size_t)((epoch & 1u) ^ 1u) * kMaxSlices;
    for (uint32_t w = slice * WG + tid; w < (uint32_t)kMaxSlices; w += ns * WG) other[w] = 0ull;
  }
  move_pair_core<T, WG, IPT, COH, COH>(A, R, k, sZ, L, ns, bits, st, slots, slot_cap, ctrl, stats, early, slice,
                                       backoff, epoch, my_stamps, add, split);
  // the last workgroup to leave (all of them have read the epoch by then)
  // starts the next call's epoch.  With err_out, it also hands the call's
  // error bits to the caller's word: every bit a workgroup sets is set by its
  // thread 0, whose returning atomics have completed before its exit count.
  if (tid == 0) {
    if (err_out) wait_all_memory();
    if (add_relaxed(&ctrl[kCtrlMoveExit], 1u) == ns - 1u) {
      st_relaxed(&ctrl[kCtrlMoveExit], 0u);
      st_relaxed(&ctrl[kCtrlMoveEpoch], epoch + 1u);
      if (err_out) {
        const uint32_t e = ld_relaxed(&ctrl[kCtrlError]);
        if (e) or_relaxed(err_out, e);
      }
    }
    if (my_stamps) my_stamps[kStampExit] = wall_clock64();
  }
}

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_move_pair(T* __restrict__ A, const int32_t* __restrict__ R, uint32_t k,
                                                    uint32_t sZ, uint32_t L, uint32_t ns,
                                                    uint32_t* __restrict__ bits, uint64_t* __restrict__ mstatus,
                                                    uint64_t* __restrict__ slots, uint32_t slot_cap,
                                                    uint32_t* __restrict__ ctrl, int stats, int early,
                                                    uint32_t* __restrict__ err_out, uint64_t* __restrict__ stamps,
                                                    const T* __restrict__ add, uint32_t split) {
  move_pair_body<T, WG, IPT, false>(A, R, k, sZ, L, ns, bits, mstatus, slots, slot_cap, ctrl, stats, early,
                                    blockIdx.x, 0u, err_out, stamps, add, split);
}

// Variant 6: the mark step in the same launch.  Workgroups [0, nm) each mark
// a tile of `tile` removals (of dense lists a range of the tail among a chunk of
// them, see range_marks) and count themselves done, and the last of them
// raises a ready word per XCD; the move-and-pair slices come after them in
// dispatch order (so every mark workgroup is running or done when a slice
// waits), prefetch their first step and wait for their XCD's ready word.
constexpr int kFusedMarkTileLog = 12;  // default tile: 4096 removals
constexpr uint32_t kMarkWaitBackoff = 16;  // longest pause between polls of the ready word: 16 x 64 cycles

// One mark workgroup of the one-launch form (id < nm): mark its tile of the
// removals, then count itself done.
template <int WG>
__device__ __forceinline__ void mark_group_body(const int32_t* __restrict__ R, uint32_t k, uint32_t sZ,
                                                uint32_t* __restrict__ bits, uint32_t* __restrict__ ctrl, int stats,
                                                uint32_t nm, uint32_t tile, int sorted,
                                                uint64_t* __restrict__ stamps, uint32_t ranges = 0,
                                                uint32_t span = 0) {
  uint64_t* const my_stamps = stamps ? stamps + (size_t)blockIdx.x * kStampsPerGroup : nullptr;
  if (my_stamps && threadIdx.x == 0) my_stamps[kStampStart] = wall_clock64();
  const uint32_t lo = blockIdx.x * tile, hi = min(lo + tile, k);
  if (ranges) {
    // this workgroup's range of the tail and chunk (of `tile` removals), as in rz_mark_ranges
    extern __shared__ uint32_t s_orph[];  // span / 32 words or more
    const uint32_t z0 = blockIdx.x % ranges * span, a = blockIdx.x / ranges * tile;
    const uint32_t b = min(a + tile, k), len = min(span, k - z0);
    if (stats)
      mark_range<WG, true, 16>(R, a, b, sZ, z0, len, false, s_orph, bits, (uint64_t*)&ctrl[kCtrlStatTail]);
    else
      mark_range<WG, false, 16>(R, a, b, sZ, z0, len, false, s_orph, bits);
  } else if (!sorted || (uint32_t)R[hi - 1] >= sZ) {  // a sorted chunk below the red zone has no marks
    // a whole tile's loads in flight at once (16 per thread for 4,096 removals and 256 threads)
    if (stats)
      mark_body<true, 16>(R + lo, hi - lo, k, sZ, bits, (uint64_t*)&ctrl[kCtrlStatTail], threadIdx.x, WG);
    else
      mark_body<false, 16>(R + lo, hi - lo, k, sZ, bits, nullptr, threadIdx.x, WG);
  }
  // Done counts in two levels: the mark workgroups with ids equal mod 8
  // share a group counter, the last of each group adds one to the global
  // count, and the last group resets it and raises the 8 ready words (one
  // per XCD, so that the waiting slices poll 8 lines).  One counter for all
  // of them serialises: same-address atomics take about 11 ns each.
  wait_all_memory();
  __syncthreads();
  if (my_stamps && threadIdx.x == 0) my_stamps[kStampMarked] = wall_clock64();
  if (threadIdx.x == 0) {
    const uint32_t x = blockIdx.x & 7u;
    const uint32_t gsize = (nm - x + 7u) / 8u;  // mark workgroups with id = x mod 8
    if (add_relaxed(&ctrl[kCtrlMarkGroup + 32 * x], 1u) == gsize - 1u) {
      st_relaxed(&ctrl[kCtrlMarkGroup + 32 * x], 0u);
      const uint32_t groups = nm < 8u ? nm : 8u;
      if (add_relaxed(&ctrl[kCtrlMarkDone], 1u) == groups - 1u) {
        st_relaxed(&ctrl[kCtrlMarkDone], 0u);
        const uint32_t ready = ld_relaxed(&ctrl[kCtrlMoveEpoch]) + 1u;  // no slice can have finished yet
        for (int r = 0; r < 8; ++r) st_relaxed(&ctrl[kCtrlMarkReady + 32 * r], ready);
        if (my_stamps) my_stamps[kStampRaised] = wall_clock64();
      }
    }
  }
}

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_mark_move_pair(T* __restrict__ A, const int32_t* __restrict__ R, uint32_t k,
                                                         uint32_t sZ, uint32_t L, uint32_t ns,
                                                         uint32_t* __restrict__ bits,
                                                         uint64_t* __restrict__ mstatus,
                                                         uint64_t* __restrict__ slots, uint32_t slot_cap,
                                                         uint32_t* __restrict__ ctrl, int stats, uint32_t nm,
                                                         uint32_t tile, uint32_t backoff, int sorted, int early,
                                                         uint32_t* __restrict__ err_out,
                                                         uint64_t* __restrict__ stamps, const T* __restrict__ add,
                                                         uint32_t split, uint32_t ranges) {
  if (blockIdx.x < nm) {
    mark_group_body<WG>(R, k, sZ, bits, ctrl, stats, nm, tile, sorted, stamps, ranges, 32u * L);
    return;
  }
  move_pair_body<T, WG, IPT, true>(A, R, k, sZ, L, ns, bits, mstatus, slots, slot_cap, ctrl, stats, early,
                                   blockIdx.x - nm, backoff, err_out, stamps, add, split);
}

// The one-launch form with n and k read from device memory (rz_remove_sized;
// the reference's TestGPUWide dereferences sizeA and sizeR in the kernel,
// redzone.hxx:457-465).  The grid is sized on the host for k_cap removals:
// nm_cap mark workgroups, then ns_cap = min(cap, ceil(k_cap / step)) slices.
// Each workgroup derives this call's shape from the device k with the host's
// slice rule (L = whole steps so that at most `cap` slices cover k), so
// L(k) <= L(k_cap) fits the launch's LDS and ns(k) <= ns_cap; the workgroups
// beyond nm(k) marks and ns(k) slices leave at once and take part in no count.
// Sizes outside 0 <= k <= n <= n_cap, k <= k_cap move nothing and set
// kErrSizes.
template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_mark_move_pair_sized(T* __restrict__ A, const int32_t* __restrict__ R,
                                                               const int32_t* __restrict__ d_n,
                                                               const int32_t* __restrict__ d_k, uint32_t n_cap,
                                                               uint32_t k_cap, uint32_t cap, uint32_t nm_cap,
                                                               uint32_t* __restrict__ bits,
                                                               uint64_t* __restrict__ mstatus,
                                                               uint64_t* __restrict__ slots,
                                                               uint32_t* __restrict__ ctrl, int stats, uint32_t tile,
                                                               uint32_t backoff, int sorted, int early) {
  const int64_t n = d_n[0], k = d_k[0];
  if (k < 0 || k > n || n > (int64_t)n_cap || k > (int64_t)k_cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) or_relaxed(&ctrl[kCtrlError], kErrSizes);
    return;
  }
  if (k == 0 || k == n) return;  // nothing moves
  const uint32_t uk = (uint32_t)k, sZ = (uint32_t)(n - k);
  constexpr uint64_t step = (uint64_t)WG * IPT;
  const uint64_t span = step * cap;
  const uint32_t L = (uint32_t)(((uk + span - 1) / span) * step);
  const uint32_t ns = (uk + L - 1) / L;
  const uint32_t nm = (uint32_t)(((uint64_t)uk + tile - 1) / tile);
  if (blockIdx.x < nm_cap) {
    if (blockIdx.x < nm) mark_group_body<WG>(R, uk, sZ, bits, ctrl, stats, nm, tile, sorted, nullptr);
    return;
  }
  const uint32_t slice = blockIdx.x - nm_cap;
  if (slice >= ns) return;
  move_pair_body<T, WG, IPT, true>(A, R, uk, sZ, L, ns, bits, mstatus, slots, uk / 2 + 1, ctrl, stats, early, slice,
                                   backoff, nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// direct form (variant 7): one launch whose workgroups never wait for each
// other.  Every workgroup reads all of R and builds two k-bit maps in LDS:
// pair i's source is dead (an LDS atomicOr per red-zone removal), pair i's
// destination is a hole (a ballot).  These give every pair's class and, with
// a prefix sum over the words, every orphan's global rank, so the workgroup
// moves its own slice of pairs and, for the t-th dest orphan, selects the
// t-th source orphan's bit itself.  No scratch, no look-back, no exchange and
// no epoch.  It reads R once per workgroup: (k / slice) * 4k bytes from the
// caches, which is what bounds its k.
// Below that it is bound by latency: R, the maps, one prefix sum, the moves,
// where the one-launch fused form pays eight device-scope round trips (marks,
// two done counters, ready word, bitmap, look-back, exchange, exit count).
// Back-to-back calls from Python on MI355X, this form (512 x 1) against the
// tuned fused shape, 4- and 16-byte items alike, us: k = 2^14 at k/n = 1% 7.2
// (the caller's own rate) against 8.5, at 50% 7.3 against 12.5; k = 2^14.5
// 8.2 against 8.5 and 7.5 against 13.1; k = 2^15.5 (1024 x 1) 11.2 against
// 8.8 and 10.1 against 13.5.  So the tuned table has it up to 2^15 removals.  From
// a fourth round of 8,192 removals on (k above 24,576) it is 0.4 to 0.8 us slower
// than a fused shape for random lists of 10 k items and more (k = 32,767 of 2^22:
// 9.3 against 8.4), and 4 us faster for tail-heavy ones (8.7 against 12.8), which
// the sizes do not tell apart.
// ---------------------------------------------------------------------------
// position of the r-th set bit of m (r below its count)
__device__ __forceinline__ uint32_t select_bit(uint64_t m, uint32_t r) {
  uint32_t pos = 0;
#pragma unroll
  for (int sh = 32; sh >= 1; sh >>= 1) {
    const uint32_t c = (uint32_t)__popcll(m & ((1ull << sh) - 1));
    if (r >= c) {
      r -= c;
      pos += sh;
      m >>= sh;
    }
  }
  return pos;
}

// PROF: thread 0 stamps the wall clock (a kernel of its own: a test for the
// stamps' address costs every other call 0.05 to 0.1 us).
template <typename T, int WG, int IPT, bool PROF>
__global__ __launch_bounds__(WG) void rz_direct(T* __restrict__ A, const int32_t* __restrict__ R, uint32_t k,
                                                 uint32_t sZ, const T* __restrict__ add, uint32_t split,
                                                 uint32_t* __restrict__ ctrl, int stats,
                                                 uint64_t* __restrict__ stamps) {
  extern __shared__ uint64_t s_direct[];
  __shared__ uint64_t s_tmp[WG / kWave + 1];
  const uint32_t W = (k + 63u) >> 6;
  uint64_t* const hole = s_direct;       // bit i: R[i] is a hole in the head
  uint64_t* const dead = hole + W;       // bit i: red-zone item i was removed
  uint64_t* const pre = dead + W;        // orphans before a word: dest | source << 32
  const uint32_t tid = threadIdx.x;
  auto stamp = [&](StampIndex at) {
    if (PROF && tid == 0) stamps[(size_t)blockIdx.x * kStampsPerGroup + at] = wall_clock64();
  };
  stamp(kStampStart);
  const RedZone<T> Z{A + sZ, add, split};
  const uint32_t base = blockIdx.x * (WG * IPT);
  // this slice's pairs, loaded ahead of the maps
  uint32_t d[IPT];
  T z[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t p = base + j * WG + tid;
    d[j] = sZ;  // no destination
    z[j] = T();
    if (p < k) {
      d[j] = (uint32_t)R[p];
      z[j] = Z[p];
    }
  }
  for (uint32_t w = tid; w < W; w += WG) dead[w] = 0ull;
  __syncthreads();
  // The maps, U words of 64 removals per wave and round: lane u collects word
  // u's ballot, so a round stores its hole words at once.  A wave64
  // instruction takes four cycles of its SIMD and every workgroup does this
  // for all of R, so the instructions per word bound the form from 2^14
  // removals up (k = 2^16 at k/n = 1%: 512 threads 13.6 us a call, 18.1 with a
  // bounds check and a one-lane store per word).
  constexpr uint32_t U = 16;
  auto round = [&](uint32_t c0, auto whole) {
    uint32_t r[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t i = c0 + u * WG + tid;
      r[u] = decltype(whole)::value || i < k ? (uint32_t)R[i] : 0xffffffffu;  // in neither zone
    }
    uint64_t words = 0;
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint64_t m = ballot(r[u] < sZ);
      if ((uint32_t)lane_id() == u) words = m;
      const uint32_t q = r[u] - sZ;  // wraps to >= 2^31 > k below the red zone
      if (q < k) atomicOr((uint32_t*)dead + (q >> 5), 1u << (q & 31));
    }
    const uint32_t w = (c0 + (tid & ~63u)) / 64u + (uint32_t)lane_id() * (WG / 64);
    if ((uint32_t)lane_id() < U && w < W) hole[w] = words;
  };
  uint32_t c0 = 0;
  for (; c0 + WG * U <= k; c0 += WG * U) round(c0, std::true_type{});
  if (c0 < k) round(c0, std::false_type{});
  __syncthreads();
  auto sources = [&](uint32_t w) {  // source orphans of word w (bits past k are none)
    const uint64_t valid = w == W - 1 && (k & 63u) ? (1ull << (k & 63u)) - 1 : ~0ull;
    return ~(hole[w] | dead[w]) & valid;
  };
  auto dests = [&](uint32_t w) { return hole[w] & dead[w]; };
  const uint32_t per = (W + WG - 1) / WG, w0 = tid * per, w1 = min(w0 + per, W);
  uint64_t sum = 0, tails = 0;
  for (uint32_t w = w0; w < w1; ++w) {
    sum += (uint64_t)__popcll(dests(w)) | (uint64_t)__popcll(sources(w)) << 32;
    tails += (uint64_t)__popcll(dead[w]);
  }
  uint64_t total;
  uint64_t ex = block_excl_scan<WG>(sum, s_tmp, &total);
  for (uint32_t w = w0; w < w1; ++w) {
    pre[w] = ex;
    ex += (uint64_t)__popcll(dests(w)) | (uint64_t)__popcll(sources(w)) << 32;
  }
  const uint32_t tot_d = (uint32_t)total, tot_s = (uint32_t)(total >> 32);
  if (blockIdx.x == 0) {
    if (tid == 0 && tot_d != tot_s) or_relaxed(&ctrl[kCtrlError], kErrOrphanMismatch);
    if (stats) {
      tails = wave_sum(tails);
      if (lane_id() == 0 && tails) add_relaxed((uint64_t*)&ctrl[kCtrlStatTail], tails);
      if (tid == 0) st_relaxed((uint64_t*)&ctrl[kCtrlStatOrphans], (uint64_t)min(tot_d, tot_s));
    }
  }
  __syncthreads();
  stamp(kStampLookback);
  // the dest orphans' sources first: a load after the moves would wait for them to drain
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t p = base + j * WG + tid, w = p >> 6;
    if (p >= k || d[j] >= sZ || !((dead[w] >> (p & 63u)) & 1ull)) {
      if (p >= k) d[j] = sZ;
      continue;
    }
    const uint32_t t = (uint32_t)pre[w] + (uint32_t)__popcll(dests(w) & ((1ull << (p & 63u)) - 1));
    if (t >= tot_s) {  // only with an invalid removal list
      d[j] = sZ;
      continue;
    }
    const uint32_t ws = (uint32_t)upper_row((int)W, t, [&](int q) { return (uint32_t)(pre[q] >> 32); });
    z[j] = Z[ws * 64u + select_bit(sources(ws), t - (uint32_t)(pre[ws] >> 32))];
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (d[j] < sZ) A[d[j]] = z[j];
  stamp(kStampMoves);
  if (PROF) wait_all_memory();
  stamp(kStampExit);
}

// ---------------------------------------------------------------------------
// cooperative single launch: the three steps separated by in-kernel grid
// barriers built from relaxed atomics (no agent-scope fences; everything a
// later step reads across workgroups was written coherently)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void grid_barrier(uint32_t* __restrict__ ctrl, uint64_t target) {
  wait_all_memory();  // this thread's coherent stores have been acknowledged
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t* cnt = (uint64_t*)&ctrl[kCtrlBarCount];
    add_relaxed(cnt, 1ull);
    uint32_t spins = 0;
    const uint32_t cap = spin_cap(ctrl, 1u << 22);
    while (ld_relaxed(cnt) < target) {
      __builtin_amdgcn_s_sleep(2);
      if (++spins > cap) {
        or_relaxed(&ctrl[kCtrlError], kErrBarrierTimeout);
        break;
      }
    }
  }
  __syncthreads();
}

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_coop(T* __restrict__ A, const int32_t* __restrict__ R,
                                               int32_t* __restrict__ Rd, uint32_t k, uint32_t sZ, uint32_t L,
                                               uint32_t ns, uint32_t* __restrict__ bits,
                                               uint64_t* __restrict__ counts, uint32_t* __restrict__ ctrl,
                                               int stats) {
  __shared__ MoveShared<WG, IPT> msh;
  __shared__ PairShared<WG, kMaxSlices> psh;
  const uint64_t base = ld_relaxed((const uint64_t*)&ctrl[kCtrlBarEpoch]);
  const uint32_t G = gridDim.x;
  if (stats)
    mark_body<true>(R, k, k, sZ, bits, (uint64_t*)&ctrl[kCtrlStatTail], blockIdx.x * WG + threadIdx.x, G * WG);
  else
    mark_body<false>(R, k, k, sZ, bits, nullptr, blockIdx.x * WG + threadIdx.x, G * WG);
  grid_barrier(ctrl, base + G);
  // every workgroup has read `base` before arriving: publish the next launch's base
  if (blockIdx.x == 0 && threadIdx.x == 0) st_relaxed((uint64_t*)&ctrl[kCtrlBarEpoch], base + 2ull * G);
  for (uint32_t s = blockIdx.x; s < ns; s += G) move_slice<T, WG, IPT, true>(A, R, Rd, k, sZ, L, s, bits, counts, msh);
  grid_barrier(ctrl, base + 2ull * G);
  pair_body<T, WG, kMaxSlices, true>(A, Rd, k, sZ, L, ns, counts, ctrl, stats, blockIdx.x, G, psh);
}

// ---------------------------------------------------------------------------
// ordered single launch: workgroups take their role from their id,
// [0, nm) mark tiles of LM removals, [nm, nm+ns) move slices, the rest pair
// shares.  Workgroups are dispatched in id order and each waits only on lower
// ids, so the launch needs neither a cooperative launch nor co-residency.
// Every workgroup does one item and exits, so the random stores of one slice
// never hold up the loads of the next (a persistent workgroup's vmcnt would).
// The last workgroup to leave resets the three counters.
// ---------------------------------------------------------------------------
enum OrderedWord : int { kOrdMark = 0, kOrdMove = 32, kOrdExit = 64 };
constexpr uint32_t kOrdMarkTile = 4096;
constexpr int kOrdCtlOffset = 128;  // words into the context's queue block

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_ordered(T* __restrict__ A, const int32_t* __restrict__ R,
                                                  int32_t* __restrict__ Rd, uint32_t k, uint32_t sZ, uint32_t L,
                                                  uint32_t ns, uint32_t nm, uint32_t* __restrict__ bits,
                                                  uint64_t* __restrict__ counts, uint32_t* __restrict__ ctrl,
                                                  uint32_t* __restrict__ q, int stats) {
  __shared__ MoveShared<WG, IPT> msh;
  __shared__ uint32_t s_last;
  extern __shared__ uint64_t dyn[];  // pairing prefix: ns + 1 entries, then WG/64 + 1 scan cells
  const uint32_t b = blockIdx.x, tid = threadIdx.x;
  if (b < nm) {
    const uint32_t lo = b * kOrdMarkTile, hi = min(lo + kOrdMarkTile, k);
    if (stats)
      mark_body<true>(R + lo, hi - lo, k, sZ, bits, (uint64_t*)&ctrl[kCtrlStatTail], tid, WG);
    else
      mark_body<false>(R + lo, hi - lo, k, sZ, bits, nullptr, tid, WG);
    signal_done(&q[kOrdMark]);
  } else if (b < nm + ns) {
    wait_count(&q[kOrdMark], nm, ctrl);
    move_slice<T, WG, IPT, true>(A, R, Rd, k, sZ, L, b - nm, bits, counts, msh, &q[kOrdMove]);
  } else {
    wait_count(&q[kOrdMove], ns, ctrl);
    pair_body_lds<T, WG, true>(A, Rd, k, sZ, L, ns, counts, ctrl, stats, b - nm - ns, gridDim.x - nm - ns, dyn,
                               dyn + ns + 1);
  }
  if (tid == 0) {
    wait_all_memory();
    s_last = add_relaxed(&q[kOrdExit], 1u) == gridDim.x - 1;
  }
  __syncthreads();
  if (s_last && tid == 0) {
    st_relaxed(&q[kOrdMark], 0u);
    st_relaxed(&q[kOrdMove], 0u);
    st_relaxed(&q[kOrdExit], 0u);
  }
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
template <typename T, int WG, int IPT>
static rz_status ordered_launch(rz_ctx* ctx, T* A, int32_t* R, int32_t* Rd, uint32_t k, uint32_t sZ, uint32_t L,
                                uint32_t ns, uint32_t* bits, uint64_t* counts, uint32_t* ctrl, int stats,
                                hipStream_t s) {
  const uint32_t nm = (k + kOrdMarkTile - 1) / kOrdMarkTile;
  uint32_t np = ns / 8;
  if (np < 1) np = 1;
  if (np > (uint32_t)ctx->cu_count) np = (uint32_t)ctx->cu_count;
  const size_t lds = ((size_t)ns + 1 + WG / kWave + 1) * sizeof(uint64_t);
  rz_status st;
  if ((st = ensure(ctx, ctx->queue, 4096, s)) != RZ_OK) return st;
  uint32_t* q = (uint32_t*)ctx->queue.ptr + kOrdCtlOffset;
  hipLaunchKernelGGL((rz_ordered<T, WG, IPT>), dim3(nm + ns + np), dim3(WG), lds, s, A, R, Rd, k, sZ, L, ns, nm,
                     bits, counts, ctrl, q, stats);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

template <typename T>
static rz_status dispatch_ordered(int wg, int ipt, rz_ctx* ctx, T* A, int32_t* R, int32_t* Rd, uint32_t k,
                                  uint32_t sZ, uint32_t L, uint32_t ns, uint32_t* bits, uint64_t* counts,
                                  uint32_t* ctrl, int stats, hipStream_t s) {
#define RZ_ORD_CASE(W, I) \
  if (wg == W && ipt == I) return ordered_launch<T, W, I>(ctx, A, R, Rd, k, sZ, L, ns, bits, counts, ctrl, stats, s);
  RZ_ORD_CASE(256, 2) RZ_ORD_CASE(256, 4) RZ_ORD_CASE(256, 8) RZ_ORD_CASE(256, 16)
  RZ_ORD_CASE(512, 2) RZ_ORD_CASE(512, 4) RZ_ORD_CASE(512, 8) RZ_ORD_CASE(512, 16)
#undef RZ_ORD_CASE
  return RZ_EINVAL;
}
template <typename T, int WG, int IPT>
static void launch_move(dim3 grid, hipStream_t s, T* A, const int32_t* R, int32_t* Rd, uint32_t k, uint32_t sZ,
                        uint32_t L, uint32_t* bits, uint64_t* counts) {
  hipLaunchKernelGGL((rz_move<T, WG, IPT>), grid, dim3(WG), 0, s, A, R, Rd, k, sZ, L, bits, counts);
}

template <typename T>
static bool dispatch_move(int wg, int ipt, dim3 grid, hipStream_t s, T* A, const int32_t* R, int32_t* Rd,
                          uint32_t k, uint32_t sZ, uint32_t L, uint32_t* bits, uint64_t* counts) {
#define RZ_MOVE_CASE(W, I) \
  if (wg == W && ipt == I) { launch_move<T, W, I>(grid, s, A, R, Rd, k, sZ, L, bits, counts); return true; }
  RZ_MOVE_CASE(256, 2) RZ_MOVE_CASE(256, 4) RZ_MOVE_CASE(256, 8) RZ_MOVE_CASE(256, 16)
  RZ_MOVE_CASE(512, 2) RZ_MOVE_CASE(512, 4) RZ_MOVE_CASE(512, 8) RZ_MOVE_CASE(512, 16)
#undef RZ_MOVE_CASE
  return false;
}

template <typename T>
static bool dispatch_move_pair(int wg, int ipt, hipStream_t s, T* A, const int32_t* R, uint32_t k, uint32_t sZ,
                               uint32_t L, uint32_t ns, uint32_t* bits, uint64_t* mstatus, uint64_t* slots,
                               uint32_t slot_cap, uint32_t* ctrl, int stats, int early, uint32_t* err_out = nullptr,
                               uint64_t* stamps = nullptr, const T* add = nullptr, uint32_t split = 0xffffffffu) {
  const size_t lds = (size_t)L * 4;
#define RZ_MP_CASE(W, I)                                                                                     \
  if (wg == W && ipt == I) {                                                                                 \
    hipLaunchKernelGGL((rz_move_pair<T, W, I>), dim3(ns), dim3(W), lds, s, A, R, k, sZ, L, ns, bits, mstatus, \
                       slots, slot_cap, ctrl, stats, early, err_out, stamps, add, split);                    \
    return true;                                                                                             \
  }
  RZ_MP_CASE(256, 2) RZ_MP_CASE(256, 4) RZ_MP_CASE(256, 8) RZ_MP_CASE(256, 16)
  RZ_MP_CASE(512, 2) RZ_MP_CASE(512, 4) RZ_MP_CASE(512, 8) RZ_MP_CASE(512, 16)
#undef RZ_MP_CASE
  return false;
}

template <typename T>
static bool dispatch_direct(int wg, int ipt, hipStream_t s, T* A, const int32_t* R, uint32_t k, uint32_t sZ,
                            const T* add, uint32_t split, uint32_t* ctrl, int stats, uint64_t* stamps) {
  const size_t lds = (size_t)((k + 63) / 64) * 24;
  const uint32_t grid = (k + wg * ipt - 1) / (wg * ipt);
#define RZ_DIRECT_CASE(W, I)                                                                                     \
  if (wg == W && ipt == I) {                                                                                     \
    auto* kern = stamps ? rz_direct<T, W, I, true> : rz_direct<T, W, I, false>;                                  \
    hipLaunchKernelGGL(kern, dim3(grid), dim3(W), lds, s, A, R, k, sZ, add, split, ctrl, stats, stamps);         \
    return true;                                                                                                 \
  }
  RZ_DIRECT_CASE(256, 1) RZ_DIRECT_CASE(256, 2) RZ_DIRECT_CASE(256, 4)
  RZ_DIRECT_CASE(512, 1) RZ_DIRECT_CASE(512, 2) RZ_DIRECT_CASE(512, 4)
  RZ_DIRECT_CASE(1024, 1) RZ_DIRECT_CASE(1024, 2)
#undef RZ_DIRECT_CASE
  return false;
}

// The one-launch fused shape of lists the direct form would run (tuned for k
// up to 2^14; it covers any k a fused form can).
constexpr rz_tile_config kSmallFused = {256, 4, 512, 6, 12, 1};

static int clamp_tile_log(int tile_log) {
  return tile_log == 0 ? kFusedMarkTileLog : (tile_log < 8 ? 8 : (tile_log > 16 ? 16 : tile_log));
}

// Whether the tail marks of an unsorted list are gathered by ranges in LDS: a
// mark by itself is a memory request, of which 26 G/s is the most, and a call
// makes k * k / n of them; by ranges every removal is read once per range, from
// the caches.  Whole calls on MI355X, 4-byte items, marks one by one -> by ranges,
// us, at n = 1.3 k / 2.2 k / 4 k / 5 k / 8 k:
//   k = 2^15.6     15.0 -> 10.4 / 13.7 -> 11.1 / 11.6 -> 10.5 / 11.0 -> 10.5 / 10.5 -> 10.6
//   k = 2^17.5     17.3 -> 12.1 / 15.5 -> 13.1 / 13.8 -> 13.0 / 13.5 -> 13.2 / 12.2 -> 12.4
//   k = 2^19.0     34.0 -> 17.3 / 26.9 -> 19.1 / 21.8 -> 19.6 / 20.3 -> 19.8 / 18.0 -> 19.3
//   k = 2^20.95    80.8 -> 36.5 / 64.0 -> 42.1 / 52.4 -> 45.8 / 49.2 -> 45.8 / 44.1 -> 46.8
//   k = 2^22.6    232.9 -> 98.9 / 199 -> 145 / 171 -> 166 / 177 -> 184 / 186 -> 212
//   k = 2^23.3    388 -> 214 / 324 -> 283 / 276 -> 315 / 273 -> 332 / 302 -> 393
// and much the same for 8- and 16-byte items.  The two meet at n = 4.3 k for
// 2^19.5 and 2^20.5 and later for the others; the direct form has k below 2^15.
// From 2^23 on the line lies elsewhere (between n = 2.2 k and 4 k at 2^23.3) and the
// marks stay single: the table's shapes of 2^24 and up group them in buckets.
static bool range_marks(int64_t n, int64_t k) { return k >= 1 << 15 && k < 1 << 23 && 4 * n <= 17 * k; }

// The mark workgroups of a call: tiles of removals, or (ranges > 0) ranges of
// `span` tail positions times chunks of `tile` removals.
struct MarkPlan {
  uint32_t nm, tile, ranges;
};
static MarkPlan range_plan(int64_t k, uint32_t span) {
  MarkPlan p;
  // A chunk's words are merged once per workgroup, so small calls take fewer:
  // 128 / 256 / 512 workgroups, n = 2.2 k, us: k = 2^17.5 13.1 / 13.8 / -,
  // 2^18.5 17.0 / 17.1 / -, 2^20 - / 27.9 / 28.5, 2^20.95 - / 48.7 / 42.1.
  const uint32_t groups = (uint32_t)std::min<int64_t>(512, std::max<int64_t>(128, k / 4096));
  p.ranges = (uint32_t)((k + span - 1) / span);
  const uint32_t chunks = groups > p.ranges ? groups / p.ranges : 1u;
  p.tile = (uint32_t)((k + chunks - 1) / chunks);
  p.nm = p.ranges * (uint32_t)((k + p.tile - 1) / p.tile);
  return p;
}
// One-launch form: the mark workgroups' LDS is the slices', so a range is 32 L
// positions, and shapes of short slices (more than 16 ranges) keep the tiles.
static MarkPlan mark_plan(int64_t n, int64_t k, uint32_t L, int tile_log, bool sorted) {
  if (!sorted && range_marks(n, k) && k <= 16ll * 32 * L) return range_plan(k, 32u * L);
  MarkPlan p;
  p.tile = 1u << clamp_tile_log(tile_log);
  p.nm = (uint32_t)((k + p.tile - 1) / p.tile);
  p.ranges = 0;
  return p;
}

// The marks as a kernel of their own; `grid` for one mark at a time.
static void launch_marks(const int32_t* R, int64_t n, int64_t k, uint32_t* bits, bool sorted, dim3 grid,
                         hipStream_t s) {
  const uint32_t sZ = (uint32_t)(n - k);
  if (sorted) {
    hipLaunchKernelGGL(rz_mark_tail_sorted, dim3((uint32_t)((k + kSortedChunk - 1) / kSortedChunk)), dim3(256), 0, s,
                       R, (uint32_t)k, sZ, bits);
  } else if (range_marks(n, k)) {
    // ranges of 8, 16 and 32 KB: about 16 of them
    const uint32_t span = k <= 1 << 20 ? 1u << 16 : k <= 1 << 21 ? 1u << 17 : 1u << 18;
    const MarkPlan p = range_plan(k, span);
    hipLaunchKernelGGL(rz_mark_ranges, dim3(p.nm), dim3(1024), span / 8, s, R, (uint32_t)k, sZ, bits, p.ranges, span,
                       p.tile);
  } else {
    hipLaunchKernelGGL(rz_mark_tail<false>, grid, dim3(256), 0, s, R, (uint32_t)k, sZ, bits, (uint64_t*)nullptr);
  }
}

// Variant 6: nm mark workgroups, then the ns move-and-pair slices, one grid.
template <typename T>
static bool dispatch_mark_move_pair(int wg, int ipt, hipStream_t s, T* A, const int32_t* R, uint32_t k, uint32_t sZ,
                                    uint32_t L, uint32_t ns, uint32_t* bits, uint64_t* mstatus, uint64_t* slots,
                                    uint32_t slot_cap, uint32_t* ctrl, int stats, int tile_log, int sorted,
                                    int early, uint32_t* err_out = nullptr, uint64_t* stamps = nullptr,
                                    const T* add = nullptr, uint32_t split = 0xffffffffu) {
  const uint32_t bo = kMarkWaitBackoff;
  const size_t lds = (size_t)L * 4;
  const MarkPlan mp = mark_plan((int64_t)sZ + k, k, L, tile_log, sorted != 0);
#define RZ_MMP_CASE(W, I)                                                                                      \
  if (wg == W && ipt == I) {                                                                                   \
    hipLaunchKernelGGL((rz_mark_move_pair<T, W, I>), dim3(mp.nm + ns), dim3(W), lds, s, A, R, k, sZ, L, ns,    \
                       bits, mstatus, slots, slot_cap, ctrl, stats, mp.nm, mp.tile, bo, sorted, early, err_out, \
                       stamps, add, split, mp.ranges);                                                         \
    return true;                                                                                               \
  }
  RZ_MMP_CASE(256, 2) RZ_MMP_CASE(256, 4) RZ_MMP_CASE(256, 8) RZ_MMP_CASE(256, 16)
  RZ_MMP_CASE(512, 2) RZ_MMP_CASE(512, 4) RZ_MMP_CASE(512, 8) RZ_MMP_CASE(512, 16)
#undef RZ_MMP_CASE
  return false;
}

// The fused form keeps a slice's orphan list in LDS (4 bytes per pair); a
// slice too long for the device's per-workgroup LDS runs the three-kernel form.
static bool fused_fits(const rz_ctx* ctx, const rz_tile_config& cfg, uint32_t L) {
  const size_t fixed = 4096;  // static LDS of the kernel, rounded up
  return (size_t)L * 4 + fixed <= (size_t)ctx->lds_per_block && cfg.wg_size * cfg.items <= (int)L;
}

void slice_shape(int64_t k, const rz_tile_config& cfg, int max_slices_cap, uint32_t* L, uint32_t* ns) {
  const int64_t step = (int64_t)cfg.wg_size * cfg.items;
  int64_t cap = cfg.max_slices < 1 ? 1 : cfg.max_slices;
  if (cap > max_slices_cap) cap = max_slices_cap;
  const int64_t steps = (k + step * cap - 1) / (step * cap);
  *L = (uint32_t)(steps * step);
  *ns = (uint32_t)((k + *L - 1) / *L);
}

template <typename T, int WG, int IPT>
static rz_status coop_launch(rz_ctx* ctx, T* A, int32_t* R, int32_t* Rd, uint32_t k, uint32_t sZ, uint32_t L,
                             uint32_t ns, uint32_t* bits, uint64_t* counts, uint32_t* ctrl, int stats,
                             hipStream_t s) {
  int per_cu = 0;
  RZ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, rz_coop<T, WG, IPT>, WG, 0));
  if (per_cu < 1) return RZ_ECOOP;
  const uint32_t resident = (uint32_t)per_cu * (uint32_t)ctx->cu_count;
  const uint32_t G = ns < resident ? ns : resident;
  void* args[] = {&A, &R, &Rd, &k, &sZ, &L, &ns, &bits, &counts, &ctrl, &stats};
  const hipError_t e = hipLaunchCooperativeKernel((const void*)rz_coop<T, WG, IPT>, dim3(G), dim3(WG), args, 0, s);
  if (e == hipErrorCooperativeLaunchTooLarge) return RZ_ECOOP;
  if (e != hipSuccess) return RZ_EHIP;
  return RZ_OK;
}

template <typename T>
static rz_status dispatch_coop(int wg, int ipt, rz_ctx* ctx, T* A, int32_t* R, int32_t* Rd, uint32_t k,
                               uint32_t sZ, uint32_t L, uint32_t ns, uint32_t* bits, uint64_t* counts,
                               uint32_t* ctrl, int stats, hipStream_t s) {
#define RZ_COOP_CASE(W, I) \
  if (wg == W && ipt == I) return coop_launch<T, W, I>(ctx, A, R, Rd, k, sZ, L, ns, bits, counts, ctrl, stats, s);
  RZ_COOP_CASE(256, 2) RZ_COOP_CASE(256, 4) RZ_COOP_CASE(256, 8) RZ_COOP_CASE(256, 16)
  RZ_COOP_CASE(512, 2) RZ_COOP_CASE(512, 4) RZ_COOP_CASE(512, 8) RZ_COOP_CASE(512, 16)
#undef RZ_COOP_CASE
  return RZ_EINVAL;
}

// RZ_PROFILE: a zeroed row of stamps for each of `groups` workgroups, the first `marks` of them mark workgroups.
static rz_status stamp_rows(rz_ctx* ctx, uint32_t groups, uint32_t marks, hipStream_t s, uint64_t** out) {
  rz_status st;
  if ((st = ensure(ctx, ctx->stamps, (size_t)groups * kStampsPerGroup * 8, s)) != RZ_OK) return st;
  *out = (uint64_t*)ctx->stamps.ptr;
  if ((st = fill_u32((uint32_t*)*out, 0u, (size_t)groups * kStampsPerGroup * 2, s)) != RZ_OK) return st;
  ctx->stamp_groups = groups;
  ctx->stamp_marks = marks;
  return RZ_OK;
}

template <typename T>
static rz_status plain_impl(rz_ctx* ctx, T* A, int64_t n, int32_t* R, int64_t k, uint32_t flags,
                            const rz_tile_config& cfg, bool coop, hipStream_t s, uint32_t* ext_bits, const T* add,
                            uint32_t split) {
  const uint32_t sZ = (uint32_t)(n - k);
  uint32_t L, ns;
  slice_shape(k, cfg, kMaxSlices, &L, &ns);
  rz_status st;
  ctx->stamp_groups = 0;  // stage stamps only from a fused call with RZ_PROFILE
  if (cfg.variant == 7 && !coop) {
    uint32_t* ctrl = (uint32_t*)ctx->ctrl.ptr;
    const int stats = (flags & RZ_STATS) ? 1 : 0;
    if (stats && (st = fill_u32(ctrl + kCtrlStatTail, 0u, 2, s)) != RZ_OK) return st;
    uint64_t* stamps = nullptr;
    if ((flags & RZ_PROFILE) &&
        (st = stamp_rows(ctx, (uint32_t)((k + cfg.wg_size * cfg.items - 1) / (cfg.wg_size * cfg.items)), 0u, s,
                         &stamps)) != RZ_OK)
      return st;
    if ((st = prof_mark(ctx, flags, 0, s)) != RZ_OK) return st;
    if ((st = prof_mark(ctx, flags, 1, s)) != RZ_OK) return st;
    if (!dispatch_direct<T>(cfg.wg_size, cfg.items, s, A, R, (uint32_t)k, sZ, add, split, ctrl, stats, stamps))
      return RZ_EINVAL;
    RZ_HIP(hipGetLastError());
    if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
    return prof_mark(ctx, flags, 3, s);
  }
  if (!ext_bits && (st = ensure(ctx, ctx->tail_bits, (size_t)((k + 63) / 64) * 8, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->counts, (size_t)ns * 8, s)) != RZ_OK) return st;
  int32_t* Rd = R;
  if (flags & RZ_PRESERVE_REMOVALS) {
    if ((st = ensure(ctx, ctx->orphans, (size_t)k * 4, s)) != RZ_OK) return st;
    Rd = (int32_t*)ctx->orphans.ptr;
  }
  uint32_t* bits = ext_bits ? ext_bits : (uint32_t*)ctx->tail_bits.ptr;
  uint64_t* counts = (uint64_t*)ctx->counts.ptr;
  uint32_t* ctrl = (uint32_t*)ctx->ctrl.ptr;
  const int stats = (flags & RZ_STATS) ? 1 : 0;
  if (stats) {  // RZ_STATS reports the counts of this call only (the error word is cleared when it is read)
    if ((st = fill_u32(ctrl + kCtrlStatTail, 0u, 2, s)) != RZ_OK) return st;
    if ((st = fill_u32(ctrl + kCtrlStatOrphans, 0u, 2, s)) != RZ_OK) return st;
  }
  if ((st = prof_mark(ctx, flags, 0, s)) != RZ_OK) return st;
  if (coop || cfg.variant == 3) {
    if ((st = prof_mark(ctx, flags, 1, s)) != RZ_OK) return st;
    if (coop)
      st = dispatch_coop<T>(cfg.wg_size, cfg.items, ctx, A, R, Rd, (uint32_t)k, sZ, L, ns, bits, counts, ctrl, stats,
                            s);
    else
      st = dispatch_ordered<T>(cfg.wg_size, cfg.items, ctx, A, R, Rd, (uint32_t)k, sZ, L, ns, bits, counts, ctrl,
                               stats, s);
    if (st != RZ_OK) return st;
    if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
    return prof_mark(ctx, flags, 3, s);
  }
  const bool fused = (cfg.variant == 4 || cfg.variant == 6) && fused_fits(ctx, cfg, L);
  const bool one_launch = fused && cfg.variant == 6;  // marks inside the fused kernel
  if (fused) {
    if ((st = ensure(ctx, ctx->mstatus, 2 * (size_t)kMaxSlices * 8, s)) != RZ_OK) return st;
    if ((st = ensure(ctx, ctx->slots, ((size_t)k / 2 + 1) * 8, s)) != RZ_OK) return st;
  }
  const bool premarked = (flags & kFlagPremarked) != 0;
  const bool dense_marks = !premarked && dense_bucket_marks(cfg, k, flags);
  const int64_t g1w = (k + 256 * 4 - 1) / (256 * 4);
  const dim3 g1((uint32_t)(g1w < (int64_t)ctx->cu_count * 8 ? g1w : ctx->cu_count * 8));
  if (premarked || dense_marks || one_launch) {
    // the caller's producer set the tail marks, or the launch below sets them itself
  } else if (stats)
    hipLaunchKernelGGL(rz_mark_tail<true>, g1, dim3(256), 0, s, R, (uint32_t)k, sZ, bits,
                       (uint64_t*)(ctrl + kCtrlStatTail));
  else
    launch_marks(R, n, k, bits, (flags & RZ_SORTED) != 0, g1, s);
  RZ_HIP(hipGetLastError());
  if ((st = prof_mark(ctx, flags, 1, s)) != RZ_OK) return st;
  if (cfg.variant == 5) {
    if ((st = dense_moves<T>(ctx, A, n, R, k, cfg, bits, ctrl, stats, dense_marks, s)) != RZ_OK) {
      // the marks are in but no move step will clear them: leave the bitmap zero
      if (!premarked) (void)fill_u32(bits, 0u, (size_t)((k + 31) / 32), s);
      return st;
    }
    if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
    return prof_mark(ctx, flags, 3, s);
  }
  uint64_t* stamps = nullptr;
  if (fused && (flags & RZ_PROFILE)) {
    const uint32_t marks =
        one_launch ? mark_plan(n, k, L, cfg.slice_steps, (flags & RZ_SORTED) != 0).nm : 0u;
    if ((st = stamp_rows(ctx, ns + marks, marks, s, &stamps)) != RZ_OK) return st;
  }
  if (one_launch) {
    if (!dispatch_mark_move_pair<T>(cfg.wg_size, cfg.items, s, A, R, (uint32_t)k, sZ, L, ns, bits,
                                    (uint64_t*)ctx->mstatus.ptr, (uint64_t*)ctx->slots.ptr, (uint32_t)(k / 2 + 1),
                                    ctrl, stats, cfg.slice_steps, (flags & RZ_SORTED) ? 1 : 0,
                                    (flags & RZ_ANY_PAIRING) ? 1 : 0, nullptr, stamps, add, split))
      return RZ_EINVAL;
    RZ_HIP(hipGetLastError());
    if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
    return prof_mark(ctx, flags, 3, s);
  }
  if (fused) {
    if (!dispatch_move_pair<T>(cfg.wg_size, cfg.items, s, A, R, (uint32_t)k, sZ, L, ns, bits,
                               (uint64_t*)ctx->mstatus.ptr, (uint64_t*)ctx->slots.ptr, (uint32_t)(k / 2 + 1), ctrl,
                               stats, (flags & RZ_ANY_PAIRING) ? 1 : 0, nullptr, stamps, add, split))
      return RZ_EINVAL;
    RZ_HIP(hipGetLastError());
    if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
    return prof_mark(ctx, flags, 3, s);
  }
  if (!dispatch_move<T>(cfg.wg_size, cfg.items, dim3(ns), s, A, R, Rd, (uint32_t)k, sZ, L, bits, counts))
    return RZ_EINVAL;
  RZ_HIP(hipGetLastError());
  if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
  const dim3 g3((uint32_t)ctx->cu_count);
  hipLaunchKernelGGL(rz_pair<T>, g3, dim3(256), 0, s, A, Rd, (uint32_t)k, sZ, L, ns, counts, ctrl, stats);
  RZ_HIP(hipGetLastError());
  return prof_mark(ctx, flags, 3, s);
}

// ---------------------------------------------------------------------------
// the fused forms on scratch the caller provides (rz_remove_noalloc)
// ---------------------------------------------------------------------------
// Clears what a fused call needs at zero: the tail bitmap words of this k, the
// error word, the exit counter and the mark-done counters.  A kernel, not a memset, so that the
// whole call can be captured in a graph.
__global__ __launch_bounds__(256) void rz_static_prologue(uint32_t* __restrict__ bits, uint32_t nwords,
                                                          uint32_t* __restrict__ ctrl) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  for (uint32_t w = i; w < nwords; w += gridDim.x * 256u) bits[w] = 0u;
  if (i == 0) {
    ctrl[kCtrlError] = 0u;
    ctrl[kCtrlMoveExit] = 0u;
    ctrl[kCtrlMarkDone] = 0u;
  }
  if (i < 8) ctrl[kCtrlMarkGroup + 32 * i] = 0u;
}

template <typename T>
static rz_status fused_static_impl(T* A, int64_t n, const int32_t* R, int64_t k, uint32_t flags,
                                   const rz_tile_config& cfg, const FusedScratch& fs, hipStream_t s) {
  const uint32_t sZ = (uint32_t)(n - k);
  uint32_t L, ns;
  slice_shape(k, cfg, kMaxSlices, &L, &ns);
  if ((size_t)L * 4 + 4096 > 65536 || cfg.wg_size * cfg.items > (int)L) return RZ_EINVAL;
  const uint32_t nwords = (uint32_t)((k + 31) / 32);
  const uint32_t g0 = (nwords + 255) / 256;
  hipLaunchKernelGGL(rz_static_prologue, dim3(g0 < 1024 ? (g0 ? g0 : 1) : 1024), dim3(256), 0, s, fs.bits, nwords,
                     fs.ctrl);
  RZ_HIP(hipGetLastError());
  const int early = (flags & RZ_ANY_PAIRING) ? 1 : 0;
  const uint32_t slot_cap = (uint32_t)(k / 2 + 1);
  if (cfg.variant == 6) {
    if (!dispatch_mark_move_pair<T>(cfg.wg_size, cfg.items, s, A, R, (uint32_t)k, sZ, L, ns, fs.bits, fs.mstatus,
                                    fs.slots, slot_cap, fs.ctrl, 0, cfg.slice_steps, (flags & RZ_SORTED) ? 1 : 0,
                                    early, fs.err_out))
      return RZ_EINVAL;
  } else {
    const int64_t g1w = (k + 256 * 4 - 1) / (256 * 4);
    launch_marks(R, n, k, fs.bits, (flags & RZ_SORTED) != 0, dim3((uint32_t)(g1w < 2048 ? g1w : 2048)), s);
    RZ_HIP(hipGetLastError());
    if (!dispatch_move_pair<T>(cfg.wg_size, cfg.items, s, A, R, (uint32_t)k, sZ, L, ns, fs.bits, fs.mstatus,
                               fs.slots, slot_cap, fs.ctrl, 0, early, fs.err_out))
      return RZ_EINVAL;
  }
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

rz_status launch_fused_static(void* data, int64_t n, uint32_t esz, const int32_t* R, int64_t k, uint32_t flags,
                              const rz_tile_config& cfg, const FusedScratch& fs, hipStream_t s) {
  if (cfg.variant != 4 && cfg.variant != 6) return RZ_EINVAL;
  switch (esz) {
    case 4: return fused_static_impl<uint32_t>((uint32_t*)data, n, R, k, flags, cfg, fs, s);
    case 8: return fused_static_impl<uint64_t>((uint64_t*)data, n, R, k, flags, cfg, fs, s);
    case 16: return fused_static_impl<uint4>((uint4*)data, n, R, k, flags, cfg, fs, s);
    default: return RZ_EINVAL;
  }
}

// Whether a launch shape can run, checked before any kernel of a call is
// launched: a call that marked the tail and then refused its move step would
// leave the bitmap set for the next call.
static bool plain_shape_ok(const rz_ctx* ctx, const rz_tile_config& cfg, uint32_t esz, int64_t n, int64_t k,
                           uint32_t flags) {
  const bool wg_ok = cfg.wg_size == 256 || cfg.wg_size == 512;
  switch (cfg.variant) {
    case 0: case 1: case 3: case 4: case 6:
      return wg_ok && (cfg.items == 2 || cfg.items == 4 || cfg.items == 8 || cfg.items == 16);
    case 2: return wg_ok && (cfg.items == 4 || cfg.items == 8);
    case 5: return dense_shape_ok(ctx, cfg, esz, n, k, flags);
    case 7:
      return k <= kDirectMaxK &&
             (cfg.items == 1 || cfg.items == 2 ? wg_ok || cfg.wg_size == 1024 : wg_ok && cfg.items == 4);
    default: return false;
  }
}

// The launch shape a call runs for a given one: the forms that take no marks
// from outside or have no cooperative launch run another.
static rz_tile_config effective_shape(const rz_tile_config& in, uint32_t flags) {
  rz_tile_config cfg = in;
  const bool premarked = (flags & kFlagPremarked) != 0;
  // the direct form marks in LDS and has neither a premarked nor a cooperative shape
  if (cfg.variant == 7 && (premarked || (flags & RZ_COOPERATIVE))) cfg = kSmallFused;
  // the single-launch forms include their own mark step: with the marks set
  // by the caller, run their shape as the two-kernel fused form
  if (premarked && ((cfg.variant >= 1 && cfg.variant <= 3) || cfg.variant == 6)) cfg.variant = 4;
  return cfg;
}

bool reads_added_in_place(const rz_ctx* ctx, const rz_tile_config& in, int64_t k, uint32_t flags) {
  const rz_tile_config cfg = effective_shape(in, flags);
  if (flags & RZ_COOPERATIVE) return false;
  if (cfg.variant == 7) return true;
  if ((cfg.variant != 4 && cfg.variant != 6) || cfg.wg_size < 1 || cfg.items < 1) return false;
  uint32_t L, ns;
  slice_shape(k, cfg, kMaxSlices, &L, &ns);
  return fused_fits(ctx, cfg, L);
}

rz_status launch_plain(rz_ctx* ctx, void* data, int64_t n, uint32_t esz, int32_t* R, int64_t k, uint32_t flags,
                       const rz_tile_config& cfg_in, hipStream_t s, uint32_t* ext_bits, const void* add,
                       uint32_t split) {
  const rz_tile_config cfg = effective_shape(cfg_in, flags);
  const bool premarked = (flags & kFlagPremarked) != 0;
  if (cfg_in.variant == 7 && !plain_shape_ok(ctx, cfg_in, esz, n, k, flags)) return RZ_EINVAL;
  if (!plain_shape_ok(ctx, cfg, esz, n, k, flags)) return RZ_EINVAL;
  if (cfg.variant == 2) return launch_queue_single(ctx, data, n, esz, R, k, flags, cfg, s);
  const bool coop = !premarked && (cfg.variant == 1 || (flags & RZ_COOPERATIVE));
  switch (esz) {
    case 4:
      return plain_impl<uint32_t>(ctx, (uint32_t*)data, n, R, k, flags, cfg, coop, s, ext_bits, (const uint32_t*)add,
                                  split);
    case 8:
      return plain_impl<uint64_t>(ctx, (uint64_t*)data, n, R, k, flags, cfg, coop, s, ext_bits, (const uint64_t*)add,
                                  split);
    case 16:
      return plain_impl<uint4>(ctx, (uint4*)data, n, R, k, flags, cfg, coop, s, ext_bits, (const uint4*)add, split);
    default: return RZ_EINVAL;
  }
}

// ---------------------------------------------------------------------------
// sizes in device memory (rz_remove_sized)
// ---------------------------------------------------------------------------
// The one-launch shape for up to k_cap removals: the context's tuned shape for
// k_cap when it is a fused form whose slices fit LDS at k_cap, else 256 x 8 with
// up to kMaxSlices slices.  false when no fused shape fits k_cap.
bool sized_shape(const rz_ctx* ctx, uint32_t esz, int64_t k_cap, rz_tile_config* out) {
  rz_tile_config c = ctx->table[esz_index(esz)][log2_floor(k_cap)];
  if (c.variant == 7) c = kSmallFused;  // the direct form takes its sizes from the host
  uint32_t L, ns;
  const bool tuned = (c.variant == 4 || c.variant == 6) && (c.wg_size == 256 || c.wg_size == 512) &&
                     (c.items == 2 || c.items == 4 || c.items == 8 || c.items == 16);
  if (tuned) {
    if (c.variant == 4) c.slice_steps = 0;  // the default mark tile
    c.variant = 6;
    slice_shape(k_cap, c, kMaxSlices, &L, &ns);
    if (fused_fits(ctx, c, L)) {
      *out = c;
      return true;
    }
  }
  c = rz_tile_config{256, 8, kMaxSlices, 6, 0, 0};
  slice_shape(k_cap, c, kMaxSlices, &L, &ns);
  if (!fused_fits(ctx, c, L)) return false;
  *out = c;
  return true;
}

template <typename T>
static rz_status sized_impl(rz_ctx* ctx, T* A, int64_t n_cap, const int32_t* R, int64_t k_cap, const int32_t* d_n,
                            const int32_t* d_k, uint32_t flags, const rz_tile_config& cfg, hipStream_t s) {
  uint32_t L_cap, ns_unused;
  slice_shape(k_cap, cfg, kMaxSlices, &L_cap, &ns_unused);
  const int64_t step = (int64_t)cfg.wg_size * cfg.items;
  const uint32_t cap = (uint32_t)(cfg.max_slices < 1 ? 1 : (cfg.max_slices > kMaxSlices ? kMaxSlices : cfg.max_slices));
  const int64_t ns_k = (k_cap + step - 1) / step;
  const uint32_t ns_cap = (uint32_t)(ns_k < (int64_t)cap ? ns_k : (int64_t)cap);
  const uint32_t tile = 1u << clamp_tile_log(cfg.slice_steps);
  const uint32_t nm_cap = (uint32_t)((k_cap + tile - 1) / tile);
  rz_status st;
  ctx->stamp_groups = 0;
  if ((st = ensure(ctx, ctx->tail_bits, (size_t)((k_cap + 63) / 64) * 8, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->mstatus, 2 * (size_t)kMaxSlices * 8, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->slots, ((size_t)k_cap / 2 + 1) * 8, s)) != RZ_OK) return st;
  uint32_t* ctrl = (uint32_t*)ctx->ctrl.ptr;
  const int stats = (flags & RZ_STATS) ? 1 : 0;
  if (stats) {
    if ((st = fill_u32(ctrl + kCtrlStatTail, 0u, 2, s)) != RZ_OK) return st;
    if ((st = fill_u32(ctrl + kCtrlStatOrphans, 0u, 2, s)) != RZ_OK) return st;
  }
  if ((st = prof_mark(ctx, flags, 0, s)) != RZ_OK) return st;
  if ((st = prof_mark(ctx, flags, 1, s)) != RZ_OK) return st;
  uint32_t* bits = (uint32_t*)ctx->tail_bits.ptr;
  uint64_t* mstatus = (uint64_t*)ctx->mstatus.ptr;
  uint64_t* slots = (uint64_t*)ctx->slots.ptr;
  const uint32_t bo = kMarkWaitBackoff, nc = (uint32_t)n_cap, kc = (uint32_t)k_cap;
  const int sorted = (flags & RZ_SORTED) ? 1 : 0, early = (flags & RZ_ANY_PAIRING) ? 1 : 0;
  const size_t lds = (size_t)L_cap * 4;
  bool launched = false;
#define RZ_SZ_CASE(W, I)                                                                                         \
  if (!launched && cfg.wg_size == W && cfg.items == I) {                                                         \
    hipLaunchKernelGGL((rz_mark_move_pair_sized<T, W, I>), dim3(nm_cap + ns_cap), dim3(W), lds, s, A, R, d_n, d_k, \
                       nc, kc, cap, nm_cap, bits, mstatus, slots, ctrl, stats, tile, bo, sorted, early);          \
    launched = true;                                                                                             \
  }
  RZ_SZ_CASE(256, 2) RZ_SZ_CASE(256, 4) RZ_SZ_CASE(256, 8) RZ_SZ_CASE(256, 16)
  RZ_SZ_CASE(512, 2) RZ_SZ_CASE(512, 4) RZ_SZ_CASE(512, 8) RZ_SZ_CASE(512, 16)
#undef RZ_SZ_CASE
  if (!launched) return RZ_EINVAL;
  RZ_HIP(hipGetLastError());
  if ((st = prof_mark(ctx, flags, 2, s)) != RZ_OK) return st;
  return prof_mark(ctx, flags, 3, s);
}

rz_status launch_sized(rz_ctx* ctx, void* data, int64_t n_cap, uint32_t esz, const int32_t* R, int64_t k_cap,
                       const int32_t* d_n, const int32_t* d_k, uint32_t flags, const rz_tile_config& cfg,
                       hipStream_t s) {
  switch (esz) {
    case 4: return sized_impl<uint32_t>(ctx, (uint32_t*)data, n_cap, R, k_cap, d_n, d_k, flags, cfg, s);
    case 8: return sized_impl<uint64_t>(ctx, (uint64_t*)data, n_cap, R, k_cap, d_n, d_k, flags, cfg, s);
    case 16: return sized_impl<uint4>(ctx, (uint4*)data, n_cap, R, k_cap, d_n, d_k, flags, cfg, s);
    default: return RZ_EINVAL;
  }
}

}  // namespace rz
