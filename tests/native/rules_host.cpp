// The rules of rz_rules.hpp at the sizes on stdin, one question a line:
//   part <n> <k>               ->  atomic | buckets | ranges <number of ranges>
//   dense <elem_bytes> <n> <k> ->  windows | stores <log2 of the most bins>
//   gather <elem_bytes> <n> <p> ->  two | one <tiles followed>
//   lds <elem_bytes> <wg> <items> <stores> <log2 of a window's positions>  ->  bytes

#include <cstdio>
#include <cstring>

#include "../../redzone_amd/csrc/rz_rules.hpp"

int main() {
  char what[32];
  while (scanf("%31s", what) == 1) {
    if (!strcmp(what, "part")) {
      long long n, k;
      if (scanf("%lld %lld", &n, &k) != 2) return 1;
      switch (rz::part_marks(n, k)) {
        case rz::PartMarks::kAtomic: printf("atomic\n"); break;
        case rz::PartMarks::kBuckets: printf("buckets\n"); break;
        case rz::PartMarks::kRanges: {
          const long long span = rz::part_range_span(n);
          printf("ranges %lld\n", (n + span - 1) / span);
        }
      }
    } else if (!strcmp(what, "dense")) {
      long long e, n, k;
      if (scanf("%lld %lld %lld", &e, &n, &k) != 3) return 1;
      if (rz::dense_scatter((uint32_t)e, n, k)) printf("stores %u\n", rz::dense_scatter_bins_log((uint32_t)e, n, k));
      else printf("windows\n");
    } else if (!strcmp(what, "gather")) {
      long long e, n, p;
      if (scanf("%lld %lld %lld", &e, &n, &p) != 3) return 1;
      if (rz::gather_two_passes((uint32_t)e, n, p)) printf("two\n");
      else printf("one %u\n", rz::gather_follow((uint32_t)e, n, p));
    } else if (!strcmp(what, "lds")) {
      int e, wg, items, stores, wlog;
      if (scanf("%d %d %d %d %d", &e, &wg, &items, &stores, &wlog) != 5) return 1;
      printf("%lld\n", (long long)rz::dense_lds_bytes((uint32_t)e, wg, items, stores != 0, (uint32_t)wlog));
    } else {
      return 1;
    }
  }
  return 0;
}
