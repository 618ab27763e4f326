// Host check of xcd_order (csrc/segment.h): over plan sizes and run lengths it is a permutation of the
// workgroups, leaves those past `end` alone, and gives XCD w % 8 whole runs, in order.
#include <cstdint>
#include <cstdio>
#include <vector>
#include "segment.h"

int main() {
  uint64_t cases = 0;
  for (uint32_t lg : {0u, 1u, 3u, 8u, 10u, 12u})
    for (uint64_t n : {1ull, 7ull, 8ull, 9ull, 8191ull, 8192ull, 8193ull, 32768ull, 100003ull}) {
      const uint64_t end = n >> (lg + 3) << (lg + 3), run = 1ull << lg;
      std::vector<uint8_t> seen(n, 0);
      for (uint64_t w = 0; w < n; ++w, ++cases) {
        const uint64_t p = emrs_internal::xcd_order(w, end, lg);
        if (p >= n || seen[p]++) return 1;
        if (w >= end && p != w) return 2;
        if (w < end && p / run % 8 != w % 8) return 3;
        if (w < end && w >= 8 && p % run && p != emrs_internal::xcd_order(w - 8, end, lg) + 1) return 4;
      }
    }
  std::printf("checked %llu\n", (unsigned long long)cases);
  return 0;
}
