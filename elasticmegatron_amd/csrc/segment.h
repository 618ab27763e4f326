// Device segments: the descriptors a copy plan is lowered to, and the arithmetic
// that places a lane's unit in them.  Plain C++ as well, so that it can be
// checked on the host.
#ifndef EMRS_SEGMENT_H
#define EMRS_SEGMENT_H

#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define EMRS_HD __host__ __device__
#else
#define EMRS_HD
#endif

namespace emrs_internal {

// A segment's unit: 2^unit_log2 bytes, one per lane, at multiples of its size
// (16 bytes: the vector path; an element: the element path); or kRowUnits:
// 16 bytes anywhere in a row, for rows of at least 16 bytes whose source,
// destination or length is no whole number of 16-byte units.  Row units follow
// the destination: unit k of a row holds the row's bytes
// [16k - p, 16k - p + 16), p being the row's distance from the 128-byte line
// (or, in rows under kLineRowBytes, from the 16-byte boundary) before it, so
// whole lines are written by one workgroup each and inner stores are aligned;
// the loads are not, and read a line twice where a workgroup ends inside it.
// A unit that reaches over an end of the row is moved inside it: it then writes
// again, with the same values, bytes that the next or previous unit writes.
// Every row has units for the largest possible p; those past its end idle.
// The element path that these segments took before moves 64 elements per
// workgroup and is bound by launching them.  Measured, before and now (12 GiB
// copied, one process): fp32 one element off 2.36 and 6.49 TB/s; bf16 one
// element off 1.22 and 6.23; rows of 667 fp32 gathered 2.41 and 6.20,
// scattered 2.39 and 5.77, gathered with their bf16 image 2.88 and 5.63.  A
// 24-layer model of hidden size 1000, TP1 DP8 -> TP4 DP2 (9.2 GB): 1805 us
// and 1494 us.
constexpr uint32_t kRowUnits = 5;
constexpr uint64_t kLineRowBytes = 512;

// Segment as the kernel sees it.  Offsets and strides are in units of
// (1 << unit_log2) bytes: 16 for the vector path, the element size otherwise
// (row units too, whose len also counts elements).
// A cast segment (fp32 only) also writes bf16 copies to aux, whose offset and
// stride are in units of half that size (8 bytes, or one bf16).  A duplicating
// segment writes its values to aux as well, in the segment's own units.
struct DevSeg {
  uint64_t src_off;
  uint64_t dst_off;
  uint64_t chunk_begin;  // index of this segment's first chunk
  uint64_t aux_off;
  uint32_t len;          // units per row
  uint32_t rows;
  uint32_t src_stride;
  uint32_t dst_stride;
  uint32_t aux_stride;
  uint32_t magic;        // row = (t + ((u - t) >> sh1)) >> sh2, t = umulhi(magic, u)
  // Whole 32-bit words only, so that a workgroup reads its descriptor with
  // scalar loads alone (the compiler reads 8- and 16-bit fields with vector
  // loads, which put a vector-memory round trip ahead of the workgroup's data).
  uint32_t bufs;         // bits 0-15: source buffer; bits 16-31: destination buffer
  uint32_t meta;         // bits 0-15: second destination (aux) buffer; 16-23: shifts; 24-31: kind

  // shifts: bits 0-4 sh2, bit 5 sh1, bit 6 row units on lines (else on 16-byte
  // boundaries), bit 7 row units (again: one bit to test).  kind: bits 0-2 unit_log2 (or kRowUnits), bits 3-4
  // elem_log2, bits 5-7 ops.  ops bit 0: also write bf16 to aux; bit 1: write
  // zeros, read nothing; bit 2: also write the values unchanged to aux.
  // elem_log2: element size of the input segment (read by the compare kernel
  // and for duplicates).
  EMRS_HD uint32_t src_buf() const { return bufs & 0xffffu; }
  EMRS_HD uint32_t dst_buf() const { return bufs >> 16; }
  EMRS_HD uint32_t aux_buf() const { return meta & 0xffffu; }
  EMRS_HD uint32_t sh1() const { return (meta >> 21) & 1u; }
  EMRS_HD uint32_t sh2() const { return (meta >> 16) & 31u; }
  EMRS_HD uint32_t unit_log2() const { return (meta >> 24) & 7u; }
  EMRS_HD uint32_t elem_log2() const { return (meta >> 27) & 3u; }
  EMRS_HD uint32_t ops() const { return meta >> 29; }
  EMRS_HD bool by_rows() const { return (meta >> 23) & 1u; }
  // A copy of 16-byte units with one destination: most of every plan.
  EMRS_HD bool plain() const { return (meta & 0xe7000000u) == 4u << 24; }
  void set_bufs(uint32_t src, uint32_t dst, uint32_t aux) {
    bufs = (src & 0xffffu) | (dst << 16);
    meta = (meta & 0xffff0000u) | (aux & 0xffffu);
  }
  // Bytes a row unit's phase is counted from, less one.
  EMRS_HD uint32_t phase_mask() const { return (meta >> 22) & 1u ? 127u : 15u; }
  // Units in a row, and in the segment.
  EMRS_HD uint32_t row_units() const {
    if (!by_rows()) return len;
    const uint32_t lg = elem_log2();
    return (len + (phase_mask() >> lg) + (15u >> lg)) >> (4 - lg);
  }
  EMRS_HD uint32_t units() const { return row_units() * rows; }
  // log2 of the bytes that offsets and strides count.
  EMRS_HD uint32_t off_log2() const { return by_rows() ? elem_log2() : unit_log2(); }
  void set_kind(uint32_t unit_log2_, uint32_t elem_log2_, uint32_t ops_, bool on_lines) {
    meta = (meta & 0x003fffffu) | ((on_lines ? 1u : 0u) << 22) | ((unit_log2_ == kRowUnits ? 1u : 0u) << 23) |
           ((unit_log2_ | (elem_log2_ << 3) | (ops_ << 5)) << 24);
  }
  void set_division(uint32_t magic_, uint32_t sh1_, uint32_t sh2_) {
    magic = magic_;
    meta = (meta & ~(63u << 16)) | ((sh2_ | (sh1_ << 5)) << 16);
  }
};
static_assert(sizeof(DevSeg) == 64, "DevSeg layout");

// Division by an invariant divisor (Granlund & Montgomery 1994, fig. 4.1).
inline void make_magic(uint32_t d, uint32_t *m, uint32_t *sh1, uint32_t *sh2) {
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  uint64_t num = (uint64_t)(((unsigned __int128)1 << 32) * (((unsigned __int128)1 << l) - d) / d) + 1;
  *m = (uint32_t)num;
  *sh1 = l < 1 ? l : 1;
  *sh2 = l > 1 ? l - 1 : 0;
}

EMRS_HD inline uint32_t umulhi32(uint32_t a, uint32_t b) {
  return (uint32_t)(((uint64_t)a * b) >> 32);
}

EMRS_HD inline uint32_t magic_div(uint32_t n, uint32_t m, uint32_t sh1,
                                                       uint32_t sh2) {
  uint32_t t = umulhi32(m, n);
  return (t + ((n - t) >> sh1)) >> sh2;
}

// Where row unit `u` of segment `s` lies: element offsets from the bases, and
// the elements [first, last) of the unit that no other unit holds as well.
// on = false: an idle unit.
struct RowUnit {
  uint64_t src, dst, aux;
  uint32_t first, last;
  bool on;
};
EMRS_HD inline RowUnit row_unit(const DevSeg &s, const char *dbase, uint32_t u, uint32_t u_end) {
  const uint32_t lg = s.elem_log2(), per = 16u >> lg, upr = s.row_units();
  uint32_t row = 0;
  if (s.rows > 1) row = magic_div(u, s.magic, s.sh1(), s.sh2());
  RowUnit r;
  r.dst = s.dst_off + (uint64_t)row * s.dst_stride;
  const uint32_t p = ((uint32_t)(uintptr_t)dbase + ((uint32_t)r.dst << lg)) & s.phase_mask();
  const int32_t at = (int32_t)((u - row * upr) * per) - (int32_t)(p >> lg), len = (int32_t)s.len;
  const int32_t end = len - (int32_t)per;  // last place of a unit
  const int32_t col = at < 0 ? 0 : (at < end ? at : end);
  r.on = u < u_end && at > -(int32_t)per && at < len;
  r.first = (uint32_t)((at < 0 ? 0 : at) - col);
  r.last = (uint32_t)((at + (int32_t)per < len ? at + (int32_t)per : len) - col);
  r.src = s.src_off + (uint64_t)row * s.src_stride + col;
  r.dst += col;
  r.aux = s.aux_off + (uint64_t)row * s.aux_stride + col;
  return r;
}

constexpr uint32_t kXcdEighths = 63;  // in place of a run's log2, see xcd_order

// Piece of workgroup `w`.  The hardware deals workgroups out to the 8 XCDs
// round-robin (workgroup w runs on XCD w % 8); the first `end` of them are
// renumbered.  By runs (whole blocks of 8 << lg): each XCD works through a run of
// 1 << lg consecutive pieces of every block, in order.  By eighths (lg kXcdEighths,
// end a multiple of 8): each XCD works through one eighth of all of them.  The
// pieces resident on one XCD then lie together, so that its L2 holds whole what two
// neighbours share, and its translation caches fewer pages.
EMRS_HD inline uint64_t xcd_order(uint64_t w, uint64_t end, uint32_t lg) {
  if (w >= end) return w;
  if (__builtin_expect(lg == kXcdEighths, 0)) return (w & 7) * (end >> 3) + (w >> 3);
  const uint32_t mask = (8u << lg) - 1, i = (uint32_t)w & mask;  // the low lg + 3 bits rotate
  return (w & ~(uint64_t)mask) | ((i & 7) << lg) | (i >> 3);
}

// Chunks in a run of one XCD (see xcd_order): 2^8 (1 MB of 16-byte units), and
// 2^10 in plans of at least 2^19 chunks.  Before, such plans gave each XCD an
// eighth of all their chunks, and smaller ones kept the hardware's order, which
// splits neighbouring kilobytes over XCDs: lines and pages at their ends are
// then fetched by two of them, the more the less aligned the rows are.  us (hardware
// order, eighths, runs of 2^8, of 2^10), one process, same allocations: 0.1 GB
// 30.7, 27.0, 29.1, 28.1; 0.55 GB of short rows 107.7, 99.9, 99.4, 99.2; 0.93 GB
// 164.6, 155.8, 155.4, 155.8; 1.02 GB of long runs 163.0, 170.1, 164.6, 167.9;
// 2.66 GB of short rows 481, 436, 431, 436; 3.4 GB Group ZeRO 637, 605, 595, 597;
// (eighths, 2^8, 2^10) 9.2 GB of short rows 1480, 1475, 1472; 28 GB 4303, 4339,
// 4290; 42 GB 6334, 6374, 6313; 70 GB 10660, 10703, 10678.  Runs of 2^4 on plans
// of every size: 9 GB in short rows 9% slower, 28 GB 11%, 45 GB 6%, 70 GB 4%.
// Time in runs over time in the hardware's order, 109 plans of 0.04 to 6 GB under
// 2^19 chunks: 0.85 to 1.00, on average 0.95, where an eighth or more of the bytes
// lies off 128-byte lines on either side (30 plans); 0.96 to 1.03, on average 1.00,
// where less does (Group ZeRO to two instances at either end).  Neither the rows'
// length nor a second destination tells which of those gain, so they take runs too.
// A comparison's first pass gained on all of the 42 plans it was timed on: 0.92 to 0.99.
constexpr uint32_t kXcdRunLog2 = 8;
constexpr uint32_t kXcdLongRunLog2 = 10;
constexpr uint64_t kXcdLongRunMinChunks = 1ull << 19;

// How the pieces of a plan are dealt out to the XCDs: the arguments of xcd_order.
struct XcdRuns {
  uint64_t end;   // pieces dealt out, the rest in the hardware's order
  uint32_t log2;  // log2 of the pieces per run, or kXcdEighths
};
// For a plan of n_chunks chunks, cut into `per_chunk` (a power of two) pieces each; `remap`: emrs_tuning.xcd_remap.
inline XcdRuns xcd_runs(uint32_t remap, uint64_t n_chunks, uint32_t per_chunk) {
  if (!remap) return XcdRuns{0, 0};
  const uint64_t pieces = n_chunks * per_chunk;
  if (remap == 2) return XcdRuns{pieces / 8 * 8, kXcdEighths};
  uint32_t lg = n_chunks >= kXcdLongRunMinChunks ? kXcdLongRunLog2 : kXcdRunLog2;
  for (; per_chunk > 1; per_chunk >>= 1) ++lg;
  return XcdRuns{pieces >> (lg + 3) << (lg + 3), lg};
}

}  // namespace emrs_internal

#endif  // EMRS_SEGMENT_H
