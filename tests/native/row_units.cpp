// Host check of the row units of device segments (csrc/segment.h): over element sizes, row lengths,
// pitches and base addresses, the units of a segment lie inside their rows, and their [first, last)
// elements cover every element of every row exactly once.
#include <cstdio>
#include <cstdint>
#include <vector>
#include "segment.h"

using namespace emrs_internal;

static int check(uint32_t lg, uint32_t len, uint32_t rows, uint32_t ds, uint64_t dst_off, uint64_t base, bool lines) {
  DevSeg s{};
  s.len = len;
  s.rows = rows;
  s.src_stride = rows > 1 ? len + 3 : 0;
  s.dst_stride = rows > 1 ? ds : 0;
  s.aux_stride = rows > 1 ? len + 1 : 0;
  s.src_off = 5;
  s.dst_off = dst_off;
  s.aux_off = 7;
  s.set_kind(kRowUnits, lg, 0, lines);
  uint32_t m = 0, sh1 = 0, sh2 = 0;
  make_magic(s.row_units(), &m, &sh1, &sh2);
  s.set_division(m, sh1, sh2);
  if (s.sh1() != sh1 || s.sh2() != sh2 || s.unit_log2() != kRowUnits || s.elem_log2() != lg) return 1;
  const uint32_t per = 16u >> lg, units = s.units();
  std::vector<uint8_t> seen((size_t)len * rows, 0);
  for (uint32_t u = 0; u < units + 3; ++u) {
    const RowUnit r = row_unit(s, reinterpret_cast<const char *>(base), u, units);
    if (!r.on) continue;
    if (u >= units || r.first >= r.last || r.last > per) return 2;
    const uint32_t row = u / s.row_units();
    const uint64_t col = r.src - (s.src_off + (uint64_t)row * s.src_stride);
    if (col + per > len) return 3;                                                  // inside its row
    if (r.dst != s.dst_off + (uint64_t)row * s.dst_stride + col) return 4;
    if (r.aux != s.aux_off + (uint64_t)row * s.aux_stride + col) return 5;
    if (r.first == 0 && r.last == per && (base + (r.dst << lg)) % 16 != 0) return 6;  // inner units are aligned
    for (uint64_t e = col + r.first; e < col + r.last; ++e)
      if (seen[row * (size_t)len + e]++) return 7;
  }
  for (uint8_t x : seen)
    if (x != 1) return 8;
  return 0;
}

int main() {
  long n = 0;
  for (uint32_t lg = 1; lg <= 3; ++lg) {
    const uint32_t per = 16u >> lg, line = 128u >> lg;
    for (uint32_t len : {per, per + 1, 2 * per - 1, 2 * per, line - 1, line, line + 1, 4 * line - 1, 4 * line, 4 * line + 1,
                         8 * line + 3, 667u, 1021u})
      for (uint32_t rows : {1u, 2u, 3u, 17u, 129u})
        for (uint32_t gap : {0u, 1u, 3u, line / 2, line})
          for (uint64_t off = 0; off < 2 * line; off += (off < per ? 1 : 3))
            for (uint64_t base : {0x10000ull, 0x10010ull, 0x10070ull})
              for (int lines = 0; lines < 2; ++lines, ++n) {
                const int rc = check(lg, len, rows, len + gap, off, base, lines != 0);
                if (rc) {
                  fprintf(stderr, "check %d failed: elem %u len %u rows %u gap %u off %llu base %llx lines %d\n", rc,
                          1u << lg, len, rows, gap, (unsigned long long)off, (unsigned long long)base, lines);
                  return 1;
                }
              }
  }
  printf("ok %ld\n", n);
  return 0;
}
