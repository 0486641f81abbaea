// rz_dense.hip -- region-bucketed Redzone for dense removal lists (variant 5).
//
// A scattered 4-byte write costs one read-modify-write of a DRAM burst, so the
// move step of the plain forms runs at about 25 G holes/s whatever the
// density, and so does the atomic tail marking.  When removals are dense
// (k/n of several percent and up) most bursts hold several targets, and
// writing them while the burst's line sits in one L2 turns many
// read-modify-writes into one.  This form regroups both the tail marks and the
// head writes by address before issuing them, in streaming passes:
//
//   tail marks (cfg.chunk == 2; otherwise the atomic rz_mark_tail)
//     bucket_marks (rz_partition.hip) over the window [sZ, n): the red-zone
//               removals appended to per-bin entry lists, then each bin's
//               bits set in an LDS bitmap and stored (two kernels)
//   head writes
//     split     one pass over the pairs: a tile classifies its pairs with the
//               wave's ballots, learns the earlier tiles' orphan counts by
//               decoupled look-back, and writes three streams without
//               staging: the moves as (position, value) entries, appended in
//               any order to a region per XCD; the t-th dest orphan's
//               position to dpos[t]; the t-th source orphan's value to
//               src[t].  Orphan ranks follow i, so the pairing is the
//               canonical one (redzone.hxx:834-934).
//     bin       the moves, then the orphan pairs (dpos[t], src[t]), in chunks
//               grouped in LDS by fine bin; a chunk's runs go to
//               fixed-capacity bins through one atomic cursor add per (chunk,
//               bin).  Distinct removals write each position at most once, so
//               a bin never holds more entries than it has positions.
//     write     one workgroup per 128 KiB window of the head: it reads its
//               bin's entries, keeps those of its window in LDS by position,
//               and writes them in address order, so a wave's store is a few
//               whole lines where one entry per lane is 64 requests.  A bin's
//               windows run on one XCD (workgroups go to the 8 XCDs round
//               robin), whose L2 serves the entries to all of them.  Items
//               that no removal names are neither read nor written.  In
//               lists above half a GiB where windows would read more than they
//               save (dense_scatter), a bin's entries are stored one by one.
//
// Every array is refilled by each call; the look-back words and the cursors
// are cleared by its first kernel.  The tail bitmap is zero on entry, set by
// the tail marks (or rz_mark_tail) and cleared by the split as it reads it.
// With an invalid list every index is checked against its buffer, and the
// orphan-count mismatch (or a bin overflow) is flagged.
//
// Bound: the streams above, 4.2 GB for 2^27 of 2^28 4-byte items at random
// (R twice, the red zone, the entries four times, the head's lines once: 840 us
// at the copy rate).  That call takes 1,460 us of kernels: marks 260 + 60,
// split 385, bin 320, write 430.  A count pass with two scans, coarse runs, two
// refine passes and a scatter of one request per hole took 1,950.
#include <algorithm>
#include <atomic>

#include "rz_fused_dev.hpp"
#include "rz_rules.hpp"

namespace rz {

constexpr int kFineMax = 4096;          // destination bins
constexpr int64_t kTailMax = 1ll << 29;  // the bucketed tail marks' largest k
constexpr uint32_t kWindowBytes = 1u << 17;  // head window of a write workgroup, staged in LDS
constexpr uint32_t kRegions = 8;             // move regions, one per XCD
constexpr uint32_t kCurStride = 32;          // words between their cursors (a line each)

// Exclusive scan of a[0, N) in LDS, in place (N <= kFineMax); returns the total.
template <int WG>
__device__ uint32_t lds_excl_scan(uint32_t* a, uint32_t N, uint32_t* tmp) {
  constexpr uint32_t MAXPER = kFineMax / WG;
  const uint32_t per = (N + WG - 1) / WG;
  const uint32_t t = threadIdx.x;
  uint32_t loc[MAXPER], sum = 0;
#pragma unroll
  for (uint32_t q = 0; q < MAXPER; ++q) {
    const uint32_t idx = t * per + q;
    loc[q] = (q < per && idx < N) ? a[idx] : 0u;
    sum += loc[q];
  }
  uint32_t total;
  uint32_t ex = block_excl_scan<WG>(sum, tmp, &total);
#pragma unroll
  for (uint32_t q = 0; q < MAXPER; ++q) {
    const uint32_t idx = t * per + q;
    if (q < per && idx < N) {
      a[idx] = ex;
      ex += loc[q];
    }
  }
  __syncthreads();
  return total;
}

// An array of (position, value) entries: interleaved for 4-byte items (a run
// of a bin is then one run of lines), positions and values apart otherwise.
template <typename T>
struct Entries {
  char* base;
  size_t cap;
  static size_t bytes(size_t cap) {
    return sizeof(T) == 4 ? cap * 8 : ((cap * 4 + 255) & ~(size_t)255) + cap * sizeof(T);
  }
  __device__ __forceinline__ const uint32_t* pos() const { return (const uint32_t*)base; }
  __device__ __forceinline__ T* val() const { return (T*)(base + ((cap * 4 + 255) & ~(size_t)255)); }
  __device__ __forceinline__ void put(size_t i, uint32_t p, const T& v) const {
    if constexpr (sizeof(T) == 4) {
      ((uint2*)base)[i] = make_uint2(p, v);
    } else {
      ((uint32_t*)base)[i] = p;
      val()[i] = v;
    }
  }
  __device__ __forceinline__ void get(size_t i, uint32_t& p, T& v) const {
    if constexpr (sizeof(T) == 4) {
      const uint2 e = ((const uint2*)base)[i];
      p = e.x;
      v = e.y;
    } else {
      p = pos()[i];
      v = val()[i];
    }
  }
};

// ---- init: the call's look-back words and cursors ---------------------------
__global__ __launch_bounds__(256) void rz_dense_init(uint64_t* __restrict__ st, uint32_t nt,
                                                     uint32_t* __restrict__ mcur, uint32_t* __restrict__ fcur,
                                                     uint32_t NBf) {
  const uint32_t i0 = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
  for (uint32_t i = i0; i < nt; i += stride) st[i] = 0ull;
  for (uint32_t i = i0; i < kRegions * kCurStride; i += stride) mcur[i] = 0u;
  for (uint32_t i = i0; i < NBf; i += stride) fcur[i] = 0u;
}

// ---- split: moves, dest orphan positions and source orphan values -----------
// Tile t takes pairs [t S, (t + 1) S), S = WG * IPT; each wave a contiguous
// 64 IPT of them, so a rank is the wave's base plus scalar counts plus a lane
// rank.  Status words as in rz_fused_dev.hpp; tiles are dispatched in id order
// and wait on earlier ones only.
template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG, 8) void rz_dense_split(const T* __restrict__ A, const int32_t* __restrict__ R,
                                                      uint32_t k, uint32_t sZ, uint32_t* __restrict__ bits,
                                                      uint64_t* __restrict__ st, uint32_t* __restrict__ mcur,
                                                      Entries<T> moves, uint32_t region, uint32_t* __restrict__ dpos,
                                                      T* __restrict__ src, uint32_t src_cap,
                                                      uint32_t* __restrict__ npairs, uint32_t* __restrict__ ctrl,
                                                      int stats) {
  constexpr int NW = WG / kWave;
  static_assert(2 * IPT <= kWave, "a lane per bitmap word of the wave");
  __shared__ uint64_t s_orph[NW];  // per wave: dest << 31 | source orphans, then their exclusive prefix
  __shared__ uint32_t s_move[NW];
  __shared__ uint64_t s_excl;
  __shared__ uint32_t s_mbase;
  const uint32_t tid = threadIdx.x, lane = lane_id(), t = blockIdx.x;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / kWave));  // scalar addresses and masks
  const uint32_t base = t * (WG * IPT) + wave * (kWave * IPT);
  // the wave's bitmap words, left zero for the next call
  uint32_t dw = 0u;
  {
    const uint32_t w = (base >> 5) + lane;
    if (lane < 2 * IPT && w < (k + 31u) >> 5) {
      dw = bits[w];
      bits[w] = 0u;
    }
  }
  uint32_t d[IPT];
  T z[IPT];
  {
    const int32_t* Rw = R + base;
    const T* Zw = A + (size_t)sZ + base;
    if (base + kWave * IPT <= k) {
#pragma unroll
      for (int j = 0; j < IPT; ++j) d[j] = (uint32_t)Rw[j * kWave + lane];
#pragma unroll
      for (int j = 0; j < IPT; ++j) z[j] = Zw[j * kWave + lane];
    } else {
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const bool in = base + j * kWave + lane < k;
        d[j] = in ? (uint32_t)Rw[j * kWave + lane] : 0xffffffffu;
        z[j] = T();
        if (in) z[j] = Zw[j * kWave + lane];
      }
    }
  }
  uint64_t hole[IPT], dead[IPT];
  uint32_t nm = 0, nd = 0, ns = 0;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t p0 = base + j * kWave;
    hole[j] = ballot(d[j] < sZ);
    // pairs past k count as dead sources without a destination
    const uint64_t past = p0 >= k ? ~0ull : (k - p0 >= 64u ? 0ull : ~0ull << (k - p0));
    dead[j] = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dw, 2 * j) |
              (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dw, 2 * j + 1) << 32 | past;
    nm += (uint32_t)__popcll(hole[j] & ~dead[j]);
    nd += (uint32_t)__popcll(hole[j] & dead[j]);
    ns += (uint32_t)__popcll(~hole[j] & ~dead[j]);
  }
  if (lane == 0) {
    s_orph[wave] = (uint64_t)nd << 31 | ns;
    s_move[wave] = nm;
  }
  __syncthreads();
  if (wave == 0) {
    const uint64_t o = lane < NW ? s_orph[lane] : 0ull;
    const uint32_t m = lane < NW ? s_move[lane] : 0u;
    const uint64_t oi = wave_incl_scan(o);
    const uint32_t mi = wave_incl_scan(m);
    const uint64_t agg = __shfl(oi, NW - 1, kWave);
    // the counts go out before anything else is waited for
    if (lane == 0) st_relaxed(&st[t], (t == 0 ? kStIncl : kStAgg) | agg);
    if (lane == NW - 1)
      s_mbase = (t % kRegions) * region + add_relaxed(&mcur[(t % kRegions) * kCurStride], mi);
    if (lane < NW) {
      s_orph[lane] = oi - o;
      s_move[lane] = mi - m;
    }
    uint64_t excl = 0;
    if (t > 0) {
      const uint32_t cap = spin_cap(ctrl, 1u << 22);
      const bool stall = stalled(ctrl);
      uint32_t spins = 0, pause = 1;
      // the nearest predecessor's word alone first (one load per poll), then
      // windows of 64 back to an inclusive prefix
      while (stall || ld_relaxed(&st[t - 1]) >> 62 == 0) {
        if (++spins > cap) break;
        for (uint32_t i = 0; i < pause; ++i) __builtin_amdgcn_s_sleep(1);
        if (pause < 16u) pause <<= 1;
      }
      int64_t jb = (int64_t)t - 1;
      spins = 0;
      pause = 1;
      while (true) {
        const int64_t q = jb - lane;
        const uint64_t w = q >= 0 ? ld_relaxed(&st[q]) : kStIncl;
        const uint32_t flag = (uint32_t)(w >> 62);
        const uint64_t incl_m = ballot(flag == 2u);
        const uint64_t none_m = ballot(flag == 0u);
        const uint64_t upto = incl_m ? ((incl_m & (~incl_m + 1)) << 1) - 1 : ~0ull;
        if (stall || (none_m & upto)) {
          // a give-up leaves excl short: every index below is checked
          if (++spins > cap) {
            if (lane == 0) or_relaxed(&ctrl[kCtrlError], kErrLookbackTimeout);
            break;
          }
          for (uint32_t i = 0; i < pause; ++i) __builtin_amdgcn_s_sleep(1);
          if (pause < 16u) pause <<= 1;
          continue;
        }
        excl += wave_sum(((upto >> lane) & 1ull) ? (w & kStCount) : 0ull);
        if (incl_m) break;
        jb -= kWave;
      }
      if (lane == 0) st_relaxed(&st[t], kStIncl | (excl + agg));
    }
    if (lane == 0) {
      s_excl = excl;
      if (t == gridDim.x - 1) {
        const uint64_t tot = excl + agg;
        const uint32_t td = (uint32_t)(tot >> 31), ts = (uint32_t)tot & 0x7fffffffu;
        *npairs = min(min(td, ts), src_cap);
        if (td != ts) or_relaxed(&ctrl[kCtrlError], kErrOrphanMismatch);
        if (stats) st_relaxed((uint64_t*)&ctrl[kCtrlStatOrphans], (uint64_t)min(td, ts));
      }
    }
  }
  __syncthreads();
  const uint64_t before = s_excl + s_orph[wave];
  uint32_t xm = s_mbase + s_move[wave], xd = (uint32_t)(before >> 31), xs = (uint32_t)before & 0x7fffffffu;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint64_t mv = hole[j] & ~dead[j], ds = hole[j] & dead[j], so = ~hole[j] & ~dead[j];
    if ((mv >> lane) & 1ull) moves.put(xm + lane_rank(mv), d[j], z[j]);
    if ((ds >> lane) & 1ull) {
      const uint32_t r = xd + lane_rank(ds);
      if (r < src_cap) dpos[r] = d[j];
    }
    if ((so >> lane) & 1ull) {
      const uint32_t r = xs + lane_rank(so);
      if (r < src_cap) src[r] = z[j];
    }
    xm += (uint32_t)__popcll(mv);
    xd += (uint32_t)__popcll(ds);
    xs += (uint32_t)__popcll(so);
  }
}

// ---- bin: entries -> fixed-capacity destination bins -------------------------
// Persistent: workgroup w takes chunks of S = WG * IPT moves of region w mod 8,
// then chunks of orphan pairs; the next chunk's loads are issued ahead of the
// stores.  Bin f holds the entries of positions [f << bsf, (f + 1) << bsf).
template <typename T, int WG, int IPT>
__global__ __launch_bounds__(WG) void rz_dense_bin(Entries<T> moves, uint32_t region, const uint32_t* __restrict__ mcur,
                                                    const uint32_t* __restrict__ dpos, const T* __restrict__ src,
                                                    const uint32_t* __restrict__ npairs, Entries<T> fine,
                                                    uint32_t* __restrict__ fcur, uint32_t NBf, uint32_t bsf,
                                                    uint32_t* __restrict__ ctrl) {
  constexpr uint32_t S = WG * IPT;
  constexpr uint32_t BPT = kFineMax / WG;  // bins per thread
  static_assert(S <= 1u << 16, "ranks of 16 bits");
  extern __shared__ __align__(16) unsigned char dyn[];
  T* const sv = (T*)dyn;
  uint32_t* const sd = (uint32_t*)(sv + S);
  __shared__ uint32_t s_bin[kFineMax + 1];
  __shared__ uint32_t tmp[WG / kWave + 1];
  const uint32_t tid = threadIdx.x;
  const uint32_t x = blockIdx.x % kRegions;
  const uint32_t nmove = min(mcur[x * kCurStride], region), npair = *npairs;
  uint32_t left = 0;  // entries of the next chunk
  uint32_t dn[IPT];  // the next chunk's entries
  T vn[IPT];
  // chunk c of this workgroup's sequence; false past its end
  uint32_t c = blockIdx.x / kRegions;
  bool pairs = false;
  auto load = [&]() -> bool {
    if (!pairs && (uint64_t)c * S >= nmove) {
      pairs = true;
      c = blockIdx.x;
    }
    const uint32_t n = pairs ? npair : nmove;
    if ((uint64_t)c * S >= n) return false;
    const uint32_t c0 = c * S, t = fresh_tid();
    // an entry past the end reads the last one again and then has no position
    if (pairs) {
#pragma unroll
      for (int q = 0; q < IPT; ++q) {
        dn[q] = dpos[min(c0 + q * WG + t, n - 1)];
        vn[q] = src[min(c0 + q * WG + t, n - 1)];
        if (q % 4 == 3) sched_fence();
      }
    } else {
#pragma unroll
      for (int q = 0; q < IPT; ++q) {
        moves.get((size_t)x * region + min(c0 + q * WG + t, n - 1), dn[q], vn[q]);
        if (q % 4 == 3) sched_fence();
      }
    }
    left = n - c0;
    c += pairs ? gridDim.x : gridDim.x / kRegions;
    return true;
  };
  auto wait_loads = [&]() {
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      arrived(dn[q]);
      arrived(vn[q]);
    }
  };
  bool over = false;
  bool more = load();
  if (more) wait_loads();
  while (more) {
    uint32_t d[IPT], rk[IPT];
    T v[IPT];
    const uint32_t t0 = fresh_tid();
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      d[q] = q * WG + t0 < left ? dn[q] : 0xffffffffu;
      v[q] = vn[q];
    }
    for (uint32_t q = tid; q <= NBf; q += WG) s_bin[q] = 0u;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < IPT; h += 4) {
      uint32_t f[4], r[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) f[q] = min(d[h + q] >> bsf, NBf);  // bin NBf: no entry
      lds_bin_ranks<4>(s_bin, f, r);
#pragma unroll
      for (int q = 0; q < 4; ++q) rk[h + q] = r[q];
    }
    __syncthreads();
    uint32_t cnt[BPT], gb[BPT];
#pragma unroll
    for (uint32_t b = 0; b < BPT; ++b) {
      const uint32_t q = b * WG + tid;
      cnt[b] = q < NBf ? s_bin[q] : 0u;
    }
    __syncthreads();
    const uint32_t tot = lds_excl_scan<WG>(s_bin, NBf, tmp);
    // room in each bin; the atomics stay in flight while the entries are staged
#pragma unroll
    for (uint32_t b = 0; b < BPT; ++b) gb[b] = cnt[b] ? add_relaxed(&fcur[b * WG + tid], cnt[b]) : 0u;
    // bin after bin, the slots without an entry last (S in all, so every slot is staged)
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const uint32_t f = min(d[q] >> bsf, NBf);
      const uint32_t e = (f == NBf ? tot : s_bin[f]) + rk[q];
      sd[e] = d[q];
      sv[e] = v[q];
      if (q % 4 == 3) sched_fence();
    }
    __syncthreads();
#pragma unroll
    for (uint32_t b = 0; b < BPT; ++b) {
      const uint32_t q = b * WG + tid;
      if (q < NBf) s_bin[q] = gb[b] - s_bin[q];  // a staged entry's place in its bin, less its place in the stage
    }
    more = load();
    __syncthreads();
    const uint32_t cap = 1u << bsf, t1 = fresh_tid();
    // no branch and S stores whatever the chunk holds, so that the wait for
    // the next chunk's loads behind them is one for the loads alone; past the
    // chunk's entries the last of them again
    const uint32_t last = max(tot, 1u) - 1u;
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const uint32_t e = min(q * WG + t1, last);
      const uint32_t p = sd[e], fe = min(p >> bsf, NBf - 1u);  // a chunk without entries only after a wait gave up
      const uint32_t r = s_bin[fe] + e;
      over |= tot && r >= cap;
      fine.put(((size_t)fe << bsf) + min(r, cap - 1u), p, sv[e]);
      if (q % 4 == 3) sched_fence();
    }
    if (more) wait_loads();
    __syncthreads();
  }
  if (over) or_relaxed(&ctrl[kCtrlError], kErrOrphanMismatch);
}

// ---- write -------------------------------------------------------------------
// Workgroup w: window g of bin f, laid out so that a bin's G windows are
// neighbours on one XCD.
template <typename T>
__global__ __launch_bounds__(1024) void rz_dense_write(T* __restrict__ A, Entries<T> fine,
                                                       const uint32_t* __restrict__ fcur, uint32_t NBf, uint32_t bsf,
                                                       uint32_t G, uint32_t wlog, uint32_t sZ) {
  extern __shared__ __align__(16) unsigned char dyn[];
  const uint32_t W = 1u << wlog;
  T* const win = (T*)dyn;
  uint32_t* const have = (uint32_t*)(win + W);  // one bit per position of the window
  const uint32_t tid = threadIdx.x;
  const uint32_t x = blockIdx.x & 7u, rest = blockIdx.x >> 3;
  const uint32_t g = rest % G, f = (rest / G) * 8u + x;
  if (f >= NBf) return;
  const uint32_t p0 = (f << bsf) + (g << wlog);
  if (p0 >= sZ) return;  // f << bsf stays below 2^32: the bins cover [0, sZ) rounded up to 8 bins
  for (uint32_t i = tid; i < W / 32; i += 1024u) have[i] = 0u;
  __syncthreads();
  const uint32_t cnt = min(fcur[f], 1u << bsf);
  const size_t s = (size_t)f << bsf;
  // U entries per thread and round; the next round's loads are in flight while this one's go to LDS
  constexpr uint32_t U = sizeof(T) == 4 ? 8 : 4;
  uint32_t p[U], pn[U];
  T v[U], vn[U];
  auto load = [&](uint32_t q0) {
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      pn[u] = 0xffffffffu;  // outside every window
      vn[u] = T();
      if (q0 + u * 1024u < cnt) {
        if constexpr (sizeof(T) == 4) fine.get(s + q0 + u * 1024u, pn[u], vn[u]);
        else pn[u] = fine.pos()[s + q0 + u * 1024u];
      }
    }
    if constexpr (sizeof(T) != 4) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u)
        if (pn[u] - p0 < W) vn[u] = fine.val()[s + q0 + u * 1024u];
    }
  };
  load(tid);
  for (uint32_t q0 = tid; q0 - tid < cnt; q0 += 1024u * U) {
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      p[u] = pn[u];
      v[u] = vn[u];
    }
    load(q0 + 1024u * U);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t o = p[u] - p0;
      if (o < W) {
        win[o] = v[u];
        atomicOr(&have[o >> 5], 1u << (o & 31u));
      }
    }
  }
  __syncthreads();
  for (uint32_t o = tid; o < W; o += 1024u)
    if (((have[o >> 5] >> (o & 31u)) & 1u) && p0 + o < sZ) A[p0 + o] = win[o];
}

// Large or sparse lists (dense_scatter): a bin's entries split among G
// workgroups on one XCD, one store per entry.  Bins in order, so an XCD writes
// into one or two of them at a time and the stores combine in its L2.
// Bound: those stores, 25 to 40 G/s.
template <typename T>
__global__ __launch_bounds__(1024) void rz_dense_scatter(T* __restrict__ A, Entries<T> fine,
                                                         const uint32_t* __restrict__ fcur, uint32_t NBf, uint32_t bsf,
                                                         uint32_t G, uint32_t sZ) {
  const uint32_t x = blockIdx.x & 7u, rest = blockIdx.x >> 3;
  const uint32_t g = rest % G, f = (rest / G) * 8u + x;
  if (f >= NBf) return;
  const uint32_t cnt = min(fcur[f], 1u << bsf), per = (cnt + G - 1) / G;
  const uint32_t lo = min(g * per, cnt), hi = min(lo + per, cnt);
  const size_t s = (size_t)f << bsf;
  for (uint32_t q = lo + threadIdx.x; q < hi; q += 1024u) {
    uint32_t p;
    T v;
    fine.get(s + q, p, v);
    if (p < sZ) A[p] = v;
  }
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
struct DenseShape {
  uint32_t NBf, bsf;   // destination bins (multiple of 8)
  bool scatter;        // single stores, else windows
  uint32_t G, wlog;    // write workgroups per bin, log2 of a window's positions
  bool bucket_marks;   // tail marks grouped (else atomic, made by the caller)
};

static uint32_t bin_log(int64_t span, int64_t target) {
  uint32_t lg = 10;
  while (((span + ((int64_t)1 << lg) - 1) >> lg) > target) ++lg;
  return lg;
}

// Dynamic-LDS limits are set with hipFuncSetAttribute once per device (the
// current one, which every entry point selects): bit d of the mask.
static bool attr_needed(const std::atomic<uint64_t>& mask, int dev) {
  return dev < 0 || dev >= 64 || !(mask.load(std::memory_order_relaxed) & (1ull << dev));
}
static void attr_done(std::atomic<uint64_t>& mask, int dev) {
  if (dev >= 0 && dev < 64) mask.fetch_or(1ull << dev, std::memory_order_relaxed);
}

// small buffer (words): move cursors, orphan pairs, bin cursors
constexpr size_t kSmallPairs = kRegions * kCurStride, kSmallFine = kSmallPairs + kCurStride;
constexpr size_t kSmallBytes = (kSmallFine + kFineMax) * 4;

// pairs of a tile, and entries of a bin chunk (4-byte items take twice as many: the longer runs)
template <typename T, int WG, int IPT>
struct DenseTiles {
  static constexpr int SPLIT_IPT = sizeof(T) == 4 ? 2 * IPT : IPT;
  static constexpr uint32_t S = WG * SPLIT_IPT;
  static constexpr int BIN_IPT = sizeof(T) == 4 ? 2 * IPT : IPT;
  static constexpr size_t LDS = (size_t)WG * BIN_IPT * (sizeof(T) + 4);
};
static uint32_t region_entries(int64_t k, uint32_t S) {
  const int64_t nt = (k + S - 1) / S;
  return (uint32_t)((nt + kRegions - 1) / kRegions) * S;
}

template <typename T, int WG, int IPT>
static rz_status dense_launch(rz_ctx* ctx, T* A, const int32_t* R, uint32_t k, uint32_t sZ, const DenseShape& d,
                              uint32_t* bits, uint32_t* ctrl, int stats, uint32_t src_cap, hipStream_t s) {
  using D = DenseTiles<T, WG, IPT>;
  const uint32_t nt = (k + D::S - 1) / D::S, region = region_entries(k, D::S);
  const size_t fcap = (size_t)d.NBf << d.bsf, mcap = (size_t)kRegions * region;
  const size_t src_off = ((size_t)src_cap * sizeof(T) + 255) & ~(size_t)255;
  rz_status st;
  if ((st = ensure(ctx, ctx->dense_cnt, (size_t)nt * 8, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->dense_small, kSmallBytes, s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->dense_ent, Entries<T>::bytes(mcap), s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->dense_fine, Entries<T>::bytes(fcap), s)) != RZ_OK) return st;
  if ((st = ensure(ctx, ctx->dense_src, src_off + (size_t)src_cap * 4, s)) != RZ_OK) return st;
  const size_t lds_win = ((size_t)sizeof(T) << d.wlog) + ((size_t)4 << d.wlog) / 32;
  static std::atomic<uint64_t> attr_mask{0};
  if (attr_needed(attr_mask, ctx->device)) {
    RZ_HIP(hipFuncSetAttribute((const void*)rz_dense_bin<T, WG, D::BIN_IPT>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)D::LDS));
    RZ_HIP(hipFuncSetAttribute((const void*)rz_dense_write<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(kWindowBytes + kWindowBytes / sizeof(T) / 8)));
    attr_done(attr_mask, ctx->device);
  }
  uint64_t* status = (uint64_t*)ctx->dense_cnt.ptr;
  uint32_t* mcur = (uint32_t*)ctx->dense_small.ptr;
  uint32_t *npairs = mcur + kSmallPairs, *fcur = mcur + kSmallFine;
  const Entries<T> moves{(char*)ctx->dense_ent.ptr, mcap}, fine{(char*)ctx->dense_fine.ptr, fcap};
  T* src = (T*)ctx->dense_src.ptr;
  uint32_t* dpos = (uint32_t*)((char*)ctx->dense_src.ptr + src_off);
  if (d.bucket_marks) {
    // tail marks grouped by tail region (the tail bitmap is zero here: every
    // launch form leaves it clear)
    st = bucket_marks(ctx, R, k, sZ, k, bits, nullptr, stats ? (uint64_t*)(ctrl + kCtrlStatTail) : (uint64_t*)nullptr,
                      s);
    if (st != RZ_OK) return st;
  }
  const uint32_t gi = (nt + 255) / 256;
  hipLaunchKernelGGL(rz_dense_init, dim3(gi < 1024 ? gi : 1024), dim3(256), 0, s, status, nt, mcur, fcur, d.NBf);
  hipLaunchKernelGGL((rz_dense_split<T, WG, D::SPLIT_IPT>), dim3(nt), dim3(WG), 0, s, A, R, k, sZ, bits, status, mcur, moves,
                     region, dpos, src, src_cap, npairs, ctrl, stats);
  // one chunk's LDS leaves one or two workgroups per CU
  const size_t per_cu = (size_t)ctx->lds_max / (D::LDS + (size_t)kFineMax * 4 + 1024);
  uint32_t gb = (uint32_t)ctx->cu_count * (uint32_t)(per_cu < 1 ? 1 : per_cu > 4 ? 4 : per_cu);
  gb = (gb + kRegions - 1) / kRegions * kRegions;
  hipLaunchKernelGGL((rz_dense_bin<T, WG, D::BIN_IPT>), dim3(gb), dim3(WG), D::LDS, s, moves, region, mcur, dpos, src,
                     npairs, fine, fcur, d.NBf, d.bsf, ctrl);
  if (d.scatter)
    hipLaunchKernelGGL(rz_dense_scatter<T>, dim3(d.NBf * d.G), dim3(1024), 0, s, A, fine, fcur, d.NBf, d.bsf, d.G, sZ);
  else
    hipLaunchKernelGGL(rz_dense_write<T>, dim3(d.NBf * d.G), dim3(1024), lds_win, s, A, fine, fcur, d.NBf, d.bsf, d.G,
                       d.wlog, sZ);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

bool dense_bucket_marks(const rz_tile_config& cfg, int64_t k, uint32_t flags) {
  return cfg.variant == 5 && cfg.chunk == 2 && k <= kTailMax && !(flags & RZ_SORTED);
}

// Fewest windows of a bin (log2).  Larger bins give the bin kernel longer runs,
// more windows make the write kernel read a bin's entries more often, of which
// 8- and 16-byte items take only the positions again.  bin + write, us, for
// 1 / 2 / 4 / 8 / 16 windows: 2^28 4-byte items, half removed 813 / 750 / 746 /
// 834 / 1105, a tenth 627 / 625 / 602 / 633 / 727; 2^27 8-byte items, 30%
// - / 744 / 689 / 762 / 956; 2^26 16-byte items, 30% - / 570 / 528 / 501 / 582.
static uint32_t min_windows_log(uint32_t esz) { return esz == 16 ? 3 : 2; }

// The dense form's bins for (cfg, n, k); RZ_EINVAL when the shape cannot be
// launched (some kernel's LDS above the device's, or a workgroup shape with none).  No
// side effect, so a caller can check before it launches anything.
static rz_status dense_shape(const rz_ctx* ctx, const rz_tile_config& cfg, uint32_t esz, int64_t n, int64_t k,
                             bool bucket_marks, DenseShape* out) {
  DenseShape& d = *out;
  const int64_t sZ = n - k;
  int lg = cfg.slice_steps > 0 ? cfg.slice_steps : 10;
  if (lg > 12) lg = 12;
  if (lg < 3) lg = 3;
  d.wlog = (uint32_t)log2_floor(kWindowBytes / esz);
  d.scatter = dense_scatter(esz, n, k);
  if (d.scatter)
    d.bsf = std::max(bin_log(sZ, (int64_t)1 << std::min<int>(lg, dense_scatter_bins_log(esz, n, k))),
                     (uint32_t)log2_floor((1 << 20) / esz));
  else
    d.bsf = std::max(bin_log(sZ, (int64_t)1 << lg), std::min(bin_log(sZ, 8), d.wlog + min_windows_log(esz)));
  d.NBf = (uint32_t)((sZ + ((int64_t)1 << d.bsf) - 1) >> d.bsf);
  d.NBf = (d.NBf + 7u) & ~7u;
  d.bucket_marks = bucket_marks;
  if (d.wlog > d.bsf) d.wlog = d.bsf;
  d.G = d.scatter ? (uint32_t)std::max(1, ctx->cu_count / 8) : 1u << (d.bsf - d.wlog);
  if (d.NBf > (uint32_t)kFineMax) return RZ_EINVAL;
  if (dense_lds_bytes(esz, cfg.wg_size, cfg.items, d.scatter, d.wlog) > ctx->lds_max) return RZ_EINVAL;
  const bool kernel = (cfg.wg_size == 256 || cfg.wg_size == 512 || cfg.wg_size == 1024) &&
                      (cfg.items == 4 || cfg.items == 8);
  return kernel ? RZ_OK : RZ_EINVAL;
}

bool dense_shape_ok(const rz_ctx* ctx, const rz_tile_config& cfg, uint32_t esz, int64_t n, int64_t k, uint32_t flags) {
  DenseShape d;
  return dense_shape(ctx, cfg, esz, n, k, dense_bucket_marks(cfg, k, flags), &d) == RZ_OK;
}

template <typename T>
rz_status dense_moves(rz_ctx* ctx, T* A, int64_t n, const int32_t* R, int64_t k, const rz_tile_config& cfg,
                      uint32_t* bits, uint32_t* ctrl, int stats, bool bucket_marks, hipStream_t s) {
  const int64_t sZ = n - k;
  DenseShape d;
  rz_status st = dense_shape(ctx, cfg, (uint32_t)sizeof(T), n, k, bucket_marks, &d);
  if (st != RZ_OK) return st;
  const uint32_t src_cap = (uint32_t)(k / 2 + 1);
#define RZ_DENSE_CASE(W, I) \
  if (cfg.wg_size == W && cfg.items == I) return dense_launch<T, W, I>(ctx, A, R, (uint32_t)k, (uint32_t)sZ, d, bits, ctrl, stats, src_cap, s);
  RZ_DENSE_CASE(256, 4) RZ_DENSE_CASE(256, 8) RZ_DENSE_CASE(512, 4) RZ_DENSE_CASE(512, 8)
  RZ_DENSE_CASE(1024, 4) RZ_DENSE_CASE(1024, 8)
#undef RZ_DENSE_CASE
  return RZ_EINVAL;
}

template rz_status dense_moves<uint32_t>(rz_ctx*, uint32_t*, int64_t, const int32_t*, int64_t,
                                         const rz_tile_config&, uint32_t*, uint32_t*, int, bool, hipStream_t);
template rz_status dense_moves<uint64_t>(rz_ctx*, uint64_t*, int64_t, const int32_t*, int64_t,
                                         const rz_tile_config&, uint32_t*, uint32_t*, int, bool, hipStream_t);
template rz_status dense_moves<uint4>(rz_ctx*, uint4*, int64_t, const int32_t*, int64_t, const rz_tile_config&,
                                      uint32_t*, uint32_t*, int, bool, hipStream_t);

}  // namespace rz
