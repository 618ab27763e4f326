// Host check of xcd_order and xcd_runs (csrc/segment.h): over plan sizes, pieces per chunk and run
// lengths the order is a permutation of the workgroups, leaves those past `end` alone, and gives XCD
// w % 8 whole runs, in order; and emrs_tuning.xcd_remap selects the hardware's order (0), runs (1) or
// one contiguous eighth per XCD (2).
#include <cstdint>
#include <cstdio>
#include <vector>
#include "segment.h"

using namespace emrs_internal;

static uint64_t cases = 0;

// `run`: pieces of one XCD that lie together.
static int check(uint64_t n, uint64_t end, uint32_t lg, uint64_t run) {
  std::vector<uint8_t> seen(n, 0);
  for (uint64_t w = 0; w < n; ++w, ++cases) {
    const uint64_t p = xcd_order(w, end, lg);
    if (p >= n || seen[p]++) return 1;
    if (w >= end && p != w) return 2;
    if (w < end && p / run % 8 != w % 8) return 3;
    if (w < end && w >= 8 && p % run && p != xcd_order(w - 8, end, lg) + 1) return 4;
  }
  return 0;
}

int main() {
  for (uint32_t lg : {0u, 1u, 3u, 8u, 10u, 12u})
    for (uint64_t n : {1ull, 7ull, 8ull, 9ull, 8191ull, 8192ull, 8193ull, 32768ull, 100003ull})
      if (const int rc = check(n, n >> (lg + 3) << (lg + 3), lg, 1ull << lg)) return rc;
  const uint64_t small = kXcdLongRunMinChunks - 1, large = kXcdLongRunMinChunks;
  for (uint32_t per : {1u, 2u, 4u})
    for (uint64_t chunks : {1ull, 2ull, 9ull, 2048ull, 3000ull, 100003ull, (unsigned long long)small, (unsigned long long)large}) {
      const uint64_t n = chunks * per;
      if (xcd_runs(0, chunks, per).end != 0) return 5;
      const XcdRuns eighths = xcd_runs(2, chunks, per), runs = xcd_runs(1, chunks, per);
      if (eighths.end != n / 8 * 8 || runs.end > n) return 6;
      if (eighths.end)
        if (const int rc = check(n, eighths.end, eighths.log2, eighths.end / 8)) return 10 + rc;
      const uint64_t run = (uint64_t)per << (chunks >= large ? kXcdLongRunLog2 : kXcdRunLog2);
      if (n - runs.end >= 8 * run) return 7;
      if (const int rc = check(n, runs.end, runs.log2, run)) return 20 + rc;
    }
  std::printf("checked %llu\n", (unsigned long long)cases);
  return 0;
}
