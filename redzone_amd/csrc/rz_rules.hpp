// rz_rules.hpp -- which form a call takes, as plain functions of its sizes (no
// HIP: a host program can include this file alone).
#pragma once

#include <cstdint>

namespace rz {

// ---------------------------------------------------------------------------
// the partition's marks
// ---------------------------------------------------------------------------
constexpr int64_t kPartMaxWindow = (int64_t)1 << 29;  // bucketed marks: entry lists of 2 GiB

enum class PartMarks { kAtomic, kRanges, kBuckets };

// Marks of lists of at least kPartBucketMinN items and kPartBucketMinK removals
// are grouped by bitmap region first: one random device atomic per removal
// runs at about 40 G/s, where the two bucketing kernels stream.  Whole calls
// on 4-byte items, random atomics -> bucketed: n=2^22, k=n/2 105 -> 43 us
// (clustered 160 -> 47 us); n=6,000,000, k=0.8n 202 -> 55 us; n=2^21,
// k=n/4 40 -> 36 us.  At n=2^20, k=2^18 the atomics still win (30 vs 41 us).
constexpr int64_t kPartBucketMinK = 1 << 19, kPartBucketMinN = 1 << 20;

// Below that, and where the two kernels of the bucketed marks are mostly their
// launches, workgroup (range, chunk) marks one range of the list among one chunk
// of the removals in LDS and merges the words (mark_range).  Whole calls on 4-byte
// items, us, random atomics or bucketed (b) -> by ranges, k/n = 0.1 / 0.4 / 0.8:
//   n = 74,000       8.9 ->  9.8 / 11.0 ->  9.7 / 13.7   ->  9.3
//   n = 296,000     10.2 -> 10.4 / 15.4 -> 10.1 / 22.5   -> 10.3
//   n = 592,000     11.6 -> 10.8 / 19.5 -> 11.3 / 30.6   -> 12.2
//   n = 1,185,000   14.7 -> 12.9 / 28.6 -> 15.0 / 20.3 b -> 16.3
//   n = 2,370,000   22.3 -> 18.4 / 23.4 b -> 21.6 / 26.1 b -> 23.3
//   n = 4,740,000   36.1 -> 27.7 / 31.0 b -> 34.5 / 33.4 b -> 40
//   n = 9,480,000 and k/n = 0.02: 35.5 -> 35.1
// and the same differences for 16-byte items.
constexpr int64_t kPartRangeMaxN = 3 << 20;  // where the bucketed marks are the other choice

// Every range reads all of the removals once, so ranges are for lists of few of
// them: with fewer than kPartBucketMinK removals n <= 12 k keeps them to 24 of 2^18
// positions, and above the bucketed marks' window (where a list would have
// thousands) the atomics mark whatever k is.
inline PartMarks part_marks(int64_t n, int64_t k) {
  if (n > kPartMaxWindow) return PartMarks::kAtomic;
  const bool bucketed = k >= kPartBucketMinK && n >= kPartBucketMinN;
  if (bucketed && n > kPartRangeMaxN) return PartMarks::kBuckets;
  if (k >= 1 << 15 ? n <= 12 * k : k >= 1 << 14 && n <= 4 * k) return PartMarks::kRanges;
  return bucketed ? PartMarks::kBuckets : PartMarks::kAtomic;
}

// Positions per range: 3 to 5 ranges while a range fits 32 KB of LDS bitmap.
inline uint32_t part_range_span(int64_t n) {
  uint32_t span = 1u << 15;
  while (span < 1u << 18 && 5ll * span < n) span <<= 1;
  return span;
}

// ---------------------------------------------------------------------------
// small removals: the direct form
// ---------------------------------------------------------------------------
constexpr int64_t kDirectMaxK = 1 << 17;  // 24 bytes of LDS per 64 removals: 48 KiB

// Whether every k of the table's bucket of k, [2^b, 2^(b+1)), fits the form.
inline bool direct_covers_bucket(int64_t k) {
  int64_t top = 1;
  while (top <= k) top *= 2;
  return top - 1 <= kDirectMaxK;
}

// ---------------------------------------------------------------------------
// the dense form's last step
// ---------------------------------------------------------------------------
// Whether a bin's entries are written one store per entry instead of through
// LDS windows.  A window is 128 KiB of the list and reads all entries of its bin
// to keep its own, and there are at most 4,096 bins: in larger lists a bin has
// more windows, and with few entries per line of the list the windows save no
// requests either.  Whole calls, windows / single stores, us:
//   4 B, 2^28 items (1 GiB): k/n = 0.01 222 / 122, 0.125 858 / 833, 0.25 1,128 / 1,123, 0.4 1,396 / 1,412
//   4 B, 2^31 items: k/n = 0.01 1,807 / 1,245, 0.06 5,787 / 4,952, 0.25 11,810 / 11,426, 0.4 25,736 / 27,050
//   8 B, 2^27 items (1 GiB): k/n = 0.01 161 / 81, 0.125 704 / 667, 0.25 949 / 909, 0.4 1,130 / 1,061
//   8 B, 2^29 items: k/n = 0.01 660 / 361, 0.06 1,852 / 1,678, 0.25 4,198 / 4,172, 0.4 5,032 / 4,773
//   16 B, 2^26 items (1 GiB): k/n = 0.25 733 / 735, 0.4 881 / 889
//   16 B, 2^27 items: k/n = 0.01 233 / 101, 0.125 998 / 938, 0.25 1,502 / 1,480, 0.4 1,767 / 1,817
//   16 B, 2^29 items: k/n = 0.01 1,049 / 386, 0.06 2,700 / 2,060, 0.25 6,985 / 5,938, 0.4 8,350 / 7,185
// Up to half a GiB (1 GiB of 16-byte items) the windows are as fast or faster.
inline bool dense_scatter(uint32_t esz, int64_t n, int64_t k) {
  const int64_t head = (n - k) * esz;
  return head > (esz == 16 ? (int64_t)1 << 30 : (int64_t)1 << 29) &&
         (esz == 8 || 3 * k < n || (esz == 16 && head > (int64_t)1 << 32));
}
// Then a bin is 1 MiB of the list or more, and the most bins (log2) are fewer for
// larger items, whose shorter chunks leave the bin kernel shorter runs (s / 8 / 9 /
// 11 for 512 / 2,048 bins: 16 B, 2^28 items, k/n = 0.125 1,944 / 1,983; 8 B, 2^28
// items, k/n = 0.06 811 / 862, 0.25 2,050 / 1,887).
inline uint32_t dense_scatter_bins_log(uint32_t esz, int64_t n, int64_t k) {
  return esz == 4 ? 12 : esz == 8 && 16 * k >= n ? 11 : 9;
}

// LDS of the dense form's largest kernel: the split's and the bin kernel's stage with
// their static part, or a window of 2^wlog positions and a bit for each.
inline int64_t dense_lds_bytes(uint32_t esz, int wg, int items, bool scatter, uint32_t wlog) {
  const int64_t stage = (int64_t)wg * items * (esz + 6) + 48 * 1024;
  const int64_t window = scatter ? 0 : ((int64_t)esz << wlog) + ((int64_t)4 << wlog) / 32;
  return stage > window ? stage : window;
}

// ---------------------------------------------------------------------------
// the gather of preserved items
// ---------------------------------------------------------------------------
// Two passes (through scratch) instead of one in place, for p below 2^22.
// Fewer than an eighth of the items kept: every item comes from a page of its own,
// and many small workgroups with nothing to wait for hide that better (p = 2^19 of
// 50 p 4-byte items: 11.2 us two passes, 12.8-14 one; 500 p: 14.3 and 21).  From an
// eighth up one launch in place is the faster one: 2^17 of 2.5 p 9.4 -> 7.0 us,
// 2^22 of 8-byte items 25.5 -> 22.7 at 95% kept.
// 4-byte lists have a band (6 p + n from 25 to 40 M) where the one pass is a single
// round of one or two tiles per CU whose waits nothing hides, two passes / one, us,
// n = 1.3 p / 2.5 p / 4 p / 6 p:
//   p = 2,300,000  12.7 / 11.4  13.4 / 12.2  14.5 / 14.3  15.8 / 15.9
//   p = 3,000,000  14.9 / 13.8  14.8 / 15.9  16.2 / 18.3  18.6 / 19.3
//   p = 3,600,000  15.7 / 16.5  16.5 / 18.7  18.6 / 19.0  22.1 / 21.9
//   p = 4,194,299  16.8 / 19.2  18.3 / 20.6  21.3 / 21.6  25.6 / 25.0
//   p = 5,000,000  21.8 / 19.1  23.6 / 21.0  26.6 / 23.9  31.8 / 28.7
inline bool gather_two_passes(uint32_t esz, int64_t n, int64_t p) {
  if (p >= (int64_t)1 << 22) return false;
  return p * 8 < n || (esz == 4 && 6 * p + n >= 25000000 && 6 * p + n <= 40000000);
}

// Earlier tiles that a tile of the one pass waits for beside the two it has to.
// Where sources and outputs are far apart, tiles that follow each other read and
// write them in longer stretches (fewer than half of 2^24.5 items kept: 16-byte 258
// us with 32, 270 without; 8-byte 146 and 149).  Dense lists lose by it (8-byte, 95%
// kept 104 against 97), and 4-byte ones unless fewer than a quarter of many are kept:
// with 16 / without, 2^26 of 4 p 293 / 311, of 8 p 476 / 502, 2^25 of 6 p 200 / 208,
// 2^24 of 4 p 78 / 77.
inline uint32_t gather_follow(uint32_t esz, int64_t n, int64_t p) {
  if (esz == 4) return p >= 3 << 23 && p * 4 <= n ? 16 : 0;
  return p >= 1 << 22 && p * 2 < n ? 32 : 0;
}

}  // namespace rz
