// rz_gather.hip -- add+remove, and the in-place gather by a preserve list.
//
// Preserve-list gather (paper p.14, eq. 3): A'[i] = A[P[i]] for i < p, P
// strictly ascending.  Two forms:
//  - one pass, in place, no scratch for the items: tiles of outputs in
//    blockIdx order; a tile writes once every earlier tile whose sources lie
//    in its output range has read them.  At most two tiles do: the sources in
//    T positions are at most T consecutive entries of P.  A tile finds them
//    with a search over the tiles' first entries.
//  - two passes (gather_two_passes): gather into context scratch with no ordering
//    between workgroups, then a device copy back to the front of the list.
#include "rz_ctx.hpp"
#include "rz_device.hpp"
#include "rz_rules.hpp"

namespace rz {

template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_gather_kernel(const T* __restrict__ A, uint32_t n,
                                                       const int32_t* __restrict__ P, uint32_t p,
                                                       T* __restrict__ out) {
  const uint32_t base = blockIdx.x * (uint32_t)(WG * IPT) + threadIdx.x;
  uint32_t src[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = base + j * WG;
    src[j] = i < p ? (uint32_t)P[i] : 0u;
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = base + j * WG;
    if (i < p) out[i] = A[src[j] < n ? src[j] : i];  // an index out of range (invalid list) reads in bounds
  }
}

// One pass, in place: tile t gathers outputs [t T, (t + 1) T) into registers,
// sets its loaded flag, waits for the two earlier tiles that may still have to
// read from its output range, and writes.  P ascends, so P[i] >= i: a tile's sources lie at or after
// its own outputs, and only earlier tiles' sources can sit in its output range.
// With `lo` the last tile whose first source lies before t T, the sources in
// [t T, (t + 1) T) start in tile lo and, being at most T, end in tile lo + 1.
// Tiles are dispatched in id order and wait on earlier ones only.  Flags carry
// the call's tag, the epoch word plus one; the last tile to leave (every tile
// has read the epoch by then) stores the tag as the new epoch, so no flag is
// ever cleared and no separate launch advances the epoch.
//
// Bound: P, the sources' lines and the outputs, streamed; for small p the
// chain load P, load sources, flag, poll, write.  Waiting for every earlier
// tile (a counter per 64 tiles, whole groups polled) took 98 us for 2^24.5 of
// 2.5 p 4-byte items where this takes 89, and 23.3 against 19.4 for 2^22 at 95%.
template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_gather_inplace(T* __restrict__ A, uint32_t n,
                                                        const int32_t* __restrict__ P, uint32_t p,
                                                        uint32_t* __restrict__ loaded, uint32_t* __restrict__ gcnt,
                                                        uint32_t ntiles, uint32_t follow,
                                                        uint32_t* __restrict__ ctrl) {
  constexpr uint32_t TILE = WG * IPT;
  const uint32_t t = blockIdx.x, i0 = t * TILE;
  const uint32_t e0 = ld_relaxed(&ctrl[kCtrlEpoch]);
  const uint32_t epoch = (e0 + 1u) & 0x3fffffffu;  // this call's tag
  uint32_t src[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = i0 + j * WG + threadIdx.x;
    src[j] = i < p ? (uint32_t)P[i] : 0u;
  }
  T v[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = i0 + j * WG + threadIdx.x;
    v[j] = T();
    if (i < p) v[j] = A[src[j] < n ? src[j] : i];  // an index out of range (invalid list) reads in bounds
  }
  uint32_t lo = 0;  // P[u TILE] < i0 for tiles u in [0, lo], or for none and lo is 0
  if (threadIdx.x < kWave && t > 0) {
    // First the 64 tiles around where a list as dense as up to here would have
    // it (one round of loads, behind the items'), then 64-way over the side it lies on.
    const float first = (float)(uint32_t)__builtin_amdgcn_readfirstlane((int)src[0]);  // P[i0]
    const float guess = first > 0.f ? (float)i0 * ((float)i0 / first) * (1.f / TILE) : 0.f;
    const uint32_t g = guess < (float)t ? (uint32_t)guess : t, w0 = g > 32u ? g - 32u : 0u, w = w0 + lane_id();
    uint64_t below = ballot(w < t && (uint32_t)P[min(w, t) * TILE] < i0);
    uint32_t len = 0;  // lo is in [lo, lo + len)
    if (below) {
      const uint32_t last = 63u - (uint32_t)__builtin_clzll(below);
      lo = w0 + last;
      if (last == 63u) len = t - lo;
    } else {
      len = w0;
    }
    while (len > 1) {
      const uint32_t step = (len + kWave - 1) / kWave;
      const uint32_t u = lo + lane_id() * step;
      below = ballot(lane_id() * step < len && (uint32_t)P[min(u, t) * TILE] < i0);
      const uint32_t last = below ? 63u - (uint32_t)__builtin_clzll(below) : 0u;
      lo += last * step;
      len = min(step, len - last * step);
    }
  }
  wait_all_memory();
  __syncthreads();
  if (threadIdx.x == 0) st_relaxed(&loaded[t * kFlagStride], epoch);
  if (threadIdx.x < kWave && t != 0) {
    // lanes 0 and 1: the tiles that may read here; lanes 2 on: the `follow` tiles just before this one
    const uint32_t l = lane_id(), u = l < 2 ? lo + l : t - min(t, l - 1u);
    const bool wait = l < 2 + follow && u < t;
    uint32_t spins = 0, pause = 1;
    while (ballot(wait && ld_relaxed(&loaded[u * kFlagStride]) != epoch)) {
      if (++spins > spin_cap(ctrl, 1u << 22)) {
        if (lane_id() == 0) or_relaxed(&ctrl[kCtrlError], kErrLookbackTimeout);
        break;
      }
      for (uint32_t i = 0; i < pause; ++i) __builtin_amdgcn_s_sleep(1);
      if (pause < 16u) pause <<= 1;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = i0 + j * WG + threadIdx.x;
    if (i < p) A[i] = v[j];
  }
  if (threadIdx.x == 0) {
    // exits counted per 64 tiles, then the groups: same-address atomics take about 11 ns each
    const uint32_t g = t >> 6, members = min(64u, ntiles - (g << 6));
    if (add_relaxed(&gcnt[g], 1u) == members - 1u) {
      st_relaxed(&gcnt[g], 0u);
      if (add_relaxed(&ctrl[kCtrlGatherExit], 1u) == ((ntiles + 63u) >> 6) - 1u) {
        st_relaxed(&ctrl[kCtrlGatherExit], 0u);
        st_relaxed(&ctrl[kCtrlEpoch], e0 + 1u);
      }
    }
  }
}

template <typename T, int WG, int IPT>
static rz_status gather_inplace_launch(rz_ctx* ctx, T* A, uint32_t n, const int32_t* P, uint32_t p, hipStream_t s) {
  const uint32_t tiles = (p + WG * IPT - 1) / (WG * IPT);
  const uint32_t groups = (tiles + 63) / 64;
  rz_status st;
  if ((st = ensure(ctx, ctx->ploaded, (size_t)tiles * kFlagStride * 4, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->pgcnt, (size_t)groups * 4, s)) != RZ_OK) return st;
  uint32_t* ctrl = (uint32_t*)ctx->ctrl.ptr;
  const uint32_t follow = gather_follow(sizeof(T), n, p);
  hipLaunchKernelGGL((rz_gather_inplace<T, WG, IPT>), dim3(tiles), dim3(WG), 0, s, A, n, P, p,
                     (uint32_t*)ctx->ploaded.ptr, (uint32_t*)ctx->pgcnt.ptr, tiles, follow, ctrl);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

template <typename T, int IPT>
static rz_status gather_launch(rz_ctx* ctx, T* A, uint32_t n, const int32_t* P, uint32_t p, hipStream_t s) {
  constexpr int WG = 256;
  rz_status st;
  if ((st = ensure(ctx, ctx->gstatus, (size_t)p * sizeof(T), s)) != RZ_OK) return st;
  T* out = (T*)ctx->gstatus.ptr;
  const uint32_t tiles = (p + WG * IPT - 1) / (WG * IPT);
  hipLaunchKernelGGL((rz_gather_kernel<T, WG, IPT>), dim3(tiles), dim3(WG), 0, s, A, n, P, p, out);
  RZ_HIP(hipGetLastError());
  RZ_HIP(hipMemcpyAsync(A, out, (size_t)p * sizeof(T), hipMemcpyDeviceToDevice, s));
  return RZ_OK;
}

template <typename T, int IPT>
static rz_status gather_form(rz_ctx* ctx, void* A, int64_t n, const int32_t* P, int64_t p, hipStream_t s) {
  if (gather_two_passes(sizeof(T), n, p)) return gather_launch<T, IPT>(ctx, (T*)A, (uint32_t)n, P, (uint32_t)p, s);
  // Big tiles: every workgroup pays for its dispatch, flags and exit (2^21 of
  // 5 M 8-byte items: 245 tiles of 1,024 x 8 14.6 us, 489 of 512 x 8 18.6).
  // With a quarter of the CUs or fewer at work, half tiles win (2^19 of 2.5 p
  // items: 8.4 against 9.2 us, 4-byte 7.8 against 8.4).
  if (p <= (int64_t)1024 * IPT * (ctx->cu_count / 4))
    return gather_inplace_launch<T, 1024, IPT / 2>(ctx, (T*)A, (uint32_t)n, P, (uint32_t)p, s);
  return gather_inplace_launch<T, 1024, IPT>(ctx, (T*)A, (uint32_t)n, P, (uint32_t)p, s);
}

}  // namespace rz

using namespace rz;

extern "C" {

rz_status rz_gather_preserve(rz_ctx* ctx, void* d_data, int64_t n, uint32_t elem_bytes, const int32_t* d_keep,
                             int64_t p, uint32_t flags, void* stream) {
  if (!ctx || n < 0 || p < 0 || p > n || n >= (1ll << 31) || esz_index(elem_bytes) < 0) return RZ_EINVAL;
  if (p == 0) return RZ_OK;
  if (!d_data || !d_keep) return RZ_EINVAL;
  if (((uintptr_t)d_data % (elem_bytes > 8 ? 16 : elem_bytes)) != 0 || ((uintptr_t)d_keep % 4) != 0) return RZ_EINVAL;
  std::lock_guard<std::mutex> lock(ctx->mu);
  int prev = -1;
  (void)hipGetDevice(&prev);
  if (prev != ctx->device) (void)hipSetDevice(ctx->device);
  hipStream_t s = (hipStream_t)stream;
  rz_status st = RZ_OK;
  if (flags & RZ_VALIDATE) st = launch_validate(ctx, d_keep, n, p, RZ_SORTED, s);
  if (st == RZ_OK) {
    switch (elem_bytes) {
      case 4: st = gather_form<uint32_t, 8>(ctx, d_data, n, d_keep, p, s); break;
      case 8: st = gather_form<uint64_t, 8>(ctx, d_data, n, d_keep, p, s); break;
      default: st = gather_form<uint4, 4>(ctx, d_data, n, d_keep, p, s); break;
    }
  }
  if (st == RZ_OK) st = finish_call(ctx, flags, s);
  if (prev >= 0 && prev != ctx->device) (void)hipSetDevice(prev);
  return st;
}

rz_status rz_add_remove(rz_ctx* ctx, void* d_data, int64_t n, int64_t capacity, uint32_t elem_bytes,
                        const void* d_add, int64_t g, int32_t* d_removals, int64_t k, uint32_t flags, void* stream) {
  if (!ctx || n < 0 || g < 0 || capacity < n + g || esz_index(elem_bytes) < 0) return RZ_EINVAL;
  if (g > 0 && (!d_add || !d_data)) return RZ_EINVAL;
  const int64_t m = n + g;
  if (m >= (1ll << 31) || k < 0 || k > m) return RZ_EINVAL;
  if (g > 0) {
    const char* add = (const char*)d_add;
    char* list = (char*)d_data;
    char* dst = list + (size_t)n * elem_bytes;
    const size_t bytes = (size_t)g * elem_bytes, head = (size_t)(m - k) * elem_bytes;
    if (add < dst + bytes && dst < add + bytes) return RZ_EINVAL;  // the added items may not overlap their slot
    std::lock_guard<std::mutex> lock(ctx->mu);
    DeviceGuard guard(ctx->device);
    hipStream_t s = (hipStream_t)stream;
    // The added items that fall into the red zone go from d_add straight to
    // their holes: the red zone is scratch afterwards, so writing them there
    // first is a copy (and a launch) for nothing.  Not if a hole could be
    // written over an added item not yet read, or if the items are not
    // aligned as the kernels load them.
    const uintptr_t align = elem_bytes > 8 ? 16 : elem_bytes;
    const rz_tile_config cfg = k > 0 && k < m ? ctx->table[esz_index(elem_bytes)][log2_floor(k)] : rz_tile_config{};
    const bool direct = k > 0 && k < m && d_removals && (uintptr_t)d_data % align == 0 &&
                        (uintptr_t)d_removals % 4 == 0 && (uintptr_t)d_add % align == 0 &&
                        !(add < list + head && list < add + bytes) && reads_added_in_place(ctx, cfg, k, flags);
    const int64_t copied = !direct ? g : g > k ? g - k : 0;  // added items that stay where they are appended
    if (copied > 0)
      RZ_HIP(hipMemcpyAsync(dst, add, (size_t)copied * elem_bytes, hipMemcpyDeviceToDevice, s));
    if (direct) {
      const size_t done = (size_t)copied * elem_bytes;
      rz_status st = flags & RZ_VALIDATE ? launch_validate(ctx, d_removals, m, k, flags, s) : RZ_OK;
      if (st == RZ_OK)
        st = launch_plain(ctx, d_data, m, elem_bytes, d_removals, k, flags, cfg, s, nullptr, add + done,
                          (uint32_t)(g < k ? k - g : 0));
      if (st == RZ_OK) return finish_call(ctx, flags, s);
      // refused: nothing is removed, and the items are appended all the same
      if (done < bytes) (void)hipMemcpyAsync(dst + done, add + done, bytes - done, hipMemcpyDeviceToDevice, s);
      return st;
    }
  }
  return rz_remove(ctx, d_data, m, elem_bytes, d_removals, k, flags, stream);
}

}  // extern "C"
