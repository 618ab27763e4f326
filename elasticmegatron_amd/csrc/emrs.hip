// Copy-plan executor for the reshard repack on MI355X (gfx950, CDNA4).
//
// One launch moves every segment of a plan.  The path is pure data movement
// (no arithmetic), so the kernel is shaped for HBM streaming: the plan is cut
// into chunks of 256 units (4 KB of 16-byte units), and every chunk into four
// pieces, each a workgroup of its own: one wave of 64 lanes with one unit each
// that reads its segment's number from the plan's chunk table and the segment's
// descriptor, loads, stores and exits.  The hardware dispatches workgroups in
// order, so the in-flight ones always cover a few narrow windows of the plan (a
// run of chunks for each XCD) that sweep through memory; a persistent grid,
// whose workgroups drift apart, writes up to 20% slower on most physical
// placements of the same buffers.  The persistent grid remains as a tuning
// option.  Element sizes are irrelevant to the vector path:
// offsets are converted to 16-byte units when the plan is created, so bf16
// parameters and fp32 optimizer state share one launch.
//
// The reference performs the same movement as per-parameter slicing plus
// point-to-point messages (elastic_megatron/transfer/transfer.py:36-101,
// :143-269; elastic_megatron/transfer/communicator.py:61-96).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "emrs.h"
#include "internal.h"
#include "segment.h"

namespace {
thread_local std::string g_last_error;
}  // namespace

// Device scratch of emrs_plan_compare_static, the entry point that allocates
// nothing: its accumulators, group ids, segment table and pointer table.  Each
// device holds its own copy for the life of the process; host code reaches it
// only through the address hipGetSymbolAddress returns on that device.
static __device__ __align__(256) unsigned char scratch[EMRS_STATIC_SCRATCH_BYTES];

namespace emrs_internal {
int fail(int code, const std::string &msg) {
  g_last_error = msg;
  return code;
}
void clear_error() { g_last_error.clear(); }
}  // namespace emrs_internal

namespace {

using namespace emrs_internal;

int hip_fail(hipError_t e, const char *what) {
  return fail(EMRS_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// A call that has to allocate device memory or upload a table cannot be
// recorded into a HIP graph: the captured copy would read host memory that is
// gone when the graph replays, and the allocation would not be replayed at
// all.  Such calls are refused while `st` is capturing; the caller runs the
// same call once outside the capture first, after which calls with the same
// base pointers need neither.
int refuse_capture(hipStream_t st, const char *what) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(st, &cs);
  if (e != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
  if (cs != hipStreamCaptureStatusNone)
    return fail(EMRS_ERR_CAPTURE, std::string(what) +
                                      " would allocate or upload while the stream is capturing a graph; "
                                      "run the call once before the capture, with the same base pointers");
  return EMRS_OK;
}

#ifndef EMRS_COPY_THREADS
#define EMRS_COPY_THREADS 256  // lanes per workgroup
#endif
#ifndef EMRS_COPY_UNROLL
#define EMRS_COPY_UNROLL 8  // chunks of one segment per step of the persistent and compare kernels
#endif
constexpr int kThreads = EMRS_COPY_THREADS;
constexpr int kUnroll = EMRS_COPY_UNROLL;
constexpr uint32_t kChunkUnits = kThreads;  // units per work chunk: one per lane
constexpr uint32_t kStepUnits = kThreads * kUnroll;  // units per step of a persistent workgroup
constexpr uint64_t kMaxGridY = 65535;                     // rows of a one-workgroup-per-chunk grid
// Row units per lane and step in copy_plan_persistent_kernel and differ_plan_kernel.  A kernel's
// registers are those of its largest path, whatever a plan holds: with kUnroll row units in flight they
// took 312-316 vector registers and 80 bytes of scratch, and 91, so that one and five waves fitted on a
// SIMD; with two, 83 (five waves) and 50 (eight).  Persistent grid, us with kUnroll and with two: 1.0 GB
// 293 and 206, 28 GB 6299 and 5451, 9.2 GB in short rows 3675 and 2050.
constexpr int kRowStep = 2;
constexpr uint64_t kMaxUnitsPerSeg = 1ull << 30;       // keeps unit math in 32 bits
// Units per lane of a comparison's first pass.  Same allocations, calls of 4 / 2
// / 1 units: 9.2 GB in short rows 1375 / 1338 / 1335 us, 28 GB 4004 / 3975 /
// 4047, 42 GB 5585 / 5588 / 5655, 44 GB 6414 / 6412 / 6484: two read as much as
// they wait for and leave no lane of a short segment idle.
constexpr int kDifferUnits = 2;
constexpr int kDifferBlocksPerCu = 4;                  // workgroups per CU of a comparison's first pass
// Row pitches of multi-row segments stay below this many bytes, so that a piece
// of at most 256 rows spans less than 2^31 bytes from its first row: the
// buffer-instruction path addresses it with 32-bit offsets.  Segments with
// longer pitches are emitted one row at a time.
constexpr uint64_t kMaxPitchBytes = 1ull << 23;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Buffers passed by value in kernel arguments; plans with more buffers on
// either side pass a device-memory table of pointers instead.  (Kernel
// arguments are limited to a few KB: this table must stay small.)
constexpr uint32_t kArgBuffers = 128;

struct Bases {
  char *p[kArgBuffers];
};
static_assert(sizeof(Bases) <= 1024, "Bases travels in kernel arguments");

// The same for plans of at most 8 buffers a side (every plan over arenas, and
// the resolved segment table of a plan over more than kArgBuffers).
constexpr uint32_t kFewBuffers = 8;
struct FewBases {
  char *p[kFewBuffers];
};

// Where a chunk's segment search starts and ends: chunk c lies in one of the
// segments first[c >> shift] .. first[(c >> shift) + 1], so the search spans
// a few dozen segments of the plan instead of all of them.  Travels in
// kernel arguments beside the two Bases.
constexpr uint32_t kHintBuckets = 256;
struct SegHint {
  uint32_t first[kHintBuckets + 1];
  uint32_t shift;
};
static_assert(2 * sizeof(Bases) + sizeof(SegHint) + 64 <= 4096, "kernel arguments stay under 4 KB");

struct Tuning {
  std::atomic<uint32_t> blocks_per_cu{0};  // persistent grid: 0 = as many as can be resident
  std::atomic<uint32_t> nontemporal{1};
  std::atomic<uint32_t> xcd_remap{1};      // 0: hardware's order; 1: runs of pieces per XCD; 2: eighths
  std::atomic<uint32_t> run{4};            // persistent grid: round-robin runs of 4 x kUnroll chunks
  std::atomic<uint32_t> persistent{0};     // 0: one workgroup per piece of a chunk
  std::atomic<uint32_t> lanes{64};         // lanes per workgroup of one piece: 64, 128 or 256
  std::atomic<uint32_t> units{1};          // 16-byte units per lane: lanes * units is 64, 128 or 256
  std::atomic<uint32_t> buffer_ops{0};     // 1: 16-byte units through buffer instructions
  std::atomic<uint32_t> chunk_index{1};    // 1: each chunk's segment from the plan's chunk table
  std::atomic<uint32_t> warm_tables{1};    // 1: read the chunk and segment tables just before the copy
};
Tuning g_tuning;

// ---------------------------------------------------------------------------
// Copy kernel
// ---------------------------------------------------------------------------

template <typename T, bool kNT>
__device__ __forceinline__ T ld(const T *p) {
  if constexpr (kNT) return __builtin_nontemporal_load(p);
  else return *p;
}

template <typename T, bool kNT>
__device__ __forceinline__ void st(T *p, T v) {
  if constexpr (kNT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// fp32 -> bf16 rounded to nearest even; NaN becomes the quiet NaN 0x7FC0
// (the rounding torch applies in float -> bfloat16 conversions).
__device__ __forceinline__ uint32_t bf16_rne(uint32_t u) {
  return (u & 0x7fffffffu) > 0x7f800000u ? 0x7fc0u : (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

template <typename T>
struct CastOf;  // bf16 image of one unit
template <>
struct CastOf<u32x4> {
  typedef unsigned int type __attribute__((ext_vector_type(2)));
  __device__ static type cast(u32x4 v) {
    type r;
    r.x = bf16_rne(v.x) | (bf16_rne(v.y) << 16);
    r.y = bf16_rne(v.z) | (bf16_rne(v.w) << 16);
    return r;
  }
};
template <>
struct CastOf<uint32_t> {
  typedef uint16_t type;
  __device__ static type cast(uint32_t v) { return (uint16_t)bf16_rne(v); }
};

// Copy units [u0, u_end) of segment s, 0 < u_end - u0 <= kStepUnits; with
// kCast also store each unit's bf16 image to aux.  In a partial chunk, lanes
// past the end load the last unit again (in bounds) so that every load is
// unconditional; only their stores are masked off.
template <typename T, bool kNT, bool kCast, bool kZero = false, bool kDup = false>
__device__ __forceinline__ void copy_chunk(const DevSeg &s, const char *sbase, char *dbase, char *abase,
                                           uint32_t u0, uint32_t u_end) {
  typedef typename std::conditional<kCast, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename C::type A;
  const T *src = reinterpret_cast<const T *>(sbase);
  T *dst = reinterpret_cast<T *>(dbase);
  A *aux = reinterpret_cast<A *>(abase);
  T *dup = reinterpret_cast<T *>(abase);  // kDup: the second destination, same unit type
  const uint32_t tid = threadIdx.x;
  const uint32_t n = u_end - u0;
  T v[kUnroll];
  if (s.rows == 1) {
    const T *sp = src + s.src_off + u0;
    T *dp = dst + s.dst_off + u0;
    A *ap = aux + s.aux_off + u0;
    T *pp = dup + s.aux_off + u0;
    if constexpr (kZero) {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) v[j] = T{};
    }
    if (n == kStepUnits) {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j)
        if constexpr (!kZero) v[j] = ld<T, kNT>(sp + j * kThreads + tid);
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) {
        st<T, kNT>(dp + j * kThreads + tid, v[j]);
        if constexpr (kCast) st<A, kNT>(ap + j * kThreads + tid, C::cast(v[j]));
        if constexpr (kDup) st<T, kNT>(pp + j * kThreads + tid, v[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j)
        if constexpr (!kZero) v[j] = ld<T, kNT>(sp + min(j * kThreads + tid, n - 1));
#pragma unroll
      for (int j = 0; j < kUnroll; ++j)
        if (j * kThreads + tid < n) {
          st<T, kNT>(dp + j * kThreads + tid, v[j]);
          if constexpr (kCast) st<A, kNT>(ap + j * kThreads + tid, C::cast(v[j]));
          if constexpr (kDup) st<T, kNT>(pp + j * kThreads + tid, v[j]);
        }
    }
    return;
  }
  uint32_t row[kUnroll], col[kUnroll];
#pragma unroll
  for (int j = 0; j < kUnroll; ++j) {
    const uint32_t u = u0 + min(j * kThreads + tid, n - 1);
    row[j] = magic_div(u, s.magic, s.sh1(), s.sh2());
    col[j] = u - row[j] * s.len;
    if constexpr (kZero) v[j] = T{};
    else v[j] = ld<T, kNT>(src + s.src_off + (uint64_t)row[j] * s.src_stride + col[j]);
  }
#pragma unroll
  for (int j = 0; j < kUnroll; ++j)
    if (j * kThreads + tid < n) {
      st<T, kNT>(dst + s.dst_off + (uint64_t)row[j] * s.dst_stride + col[j], v[j]);
      if constexpr (kCast)
        st<A, kNT>(aux + s.aux_off + (uint64_t)row[j] * s.aux_stride + col[j], C::cast(v[j]));
      if constexpr (kDup) st<T, kNT>(dup + s.aux_off + (uint64_t)row[j] * s.aux_stride + col[j], v[j]);
    }
}

// Units at any multiple of 2 bytes (the hardware takes them, and the compiler emits whole loads and stores).
typedef u32x4 __attribute__((aligned(2))) u32x4_any;
typedef CastOf<u32x4>::type __attribute__((aligned(2))) u32x2_any;
// Accesses to them of their own: as a template argument the type would lose its alignment.
template <bool kNT>
__device__ __forceinline__ u32x4 ld16(const char *p) {
  if constexpr (kNT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any *>(p));
  else return *reinterpret_cast<const u32x4_any *>(p);
}
template <bool kNT>
__device__ __forceinline__ CastOf<u32x4>::type ld8(const char *p) {
  if constexpr (kNT) return __builtin_nontemporal_load(reinterpret_cast<const u32x2_any *>(p));
  else return *reinterpret_cast<const u32x2_any *>(p);
}
template <bool kNT>
__device__ __forceinline__ void st16(char *p, u32x4 v) {
  if constexpr (kNT) __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any *>(p));
  else *reinterpret_cast<u32x4_any *>(p) = v;
}
template <bool kNT>
__device__ __forceinline__ void st8(char *p, CastOf<u32x4>::type v) {
  if constexpr (kNT) __builtin_nontemporal_store(v, reinterpret_cast<u32x2_any *>(p));
  else *reinterpret_cast<u32x2_any *>(p) = v;
}

// Row units [u0, u0 + L * U) of segment s (clipped to u_end) by a workgroup of
// L lanes, U units per lane, every load issued before the first store.
template <bool kNT, bool kCast, bool kZero, bool kDup, int L, int U>
__device__ __forceinline__ void copy_rows(const DevSeg &s, const char *sbase, char *dbase, char *abase, uint32_t u0,
                                          uint32_t u_end) {
  const uint32_t lg = s.elem_log2();
  u32x4 v[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    v[j] = u32x4{};
    if constexpr (!kZero) {
      const RowUnit r = row_unit(s, dbase, u0 + j * L + threadIdx.x, u_end);
      if (r.on) v[j] = ld16<kNT>(sbase + (r.src << lg));
    }
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const RowUnit r = row_unit(s, dbase, u0 + j * L + threadIdx.x, u_end);
    if (r.on) {
      st16<kNT>(dbase + (r.dst << lg), v[j]);
      if constexpr (kCast)
        st8<kNT>(abase + (r.aux << 1), CastOf<u32x4>::cast(v[j]));
      if constexpr (kDup) st16<kNT>(abase + (r.aux << lg), v[j]);
    }
  }
}

// copy_rows for what the segment's ops ask for.
template <bool kNT, int L, int U>
__device__ __forceinline__ void dispatch_rows(const DevSeg &s, const char *sb, char *db, char *ab, uint32_t u0,
                                              uint32_t u_end) {
  switch (s.ops()) {
    case 0: copy_rows<kNT, false, false, false, L, U>(s, sb, db, ab, u0, u_end); break;
    case 1: copy_rows<kNT, true, false, false, L, U>(s, sb, db, ab, u0, u_end); break;
    case 2: copy_rows<kNT, false, true, false, L, U>(s, sb, db, ab, u0, u_end); break;
    case 3: copy_rows<kNT, true, true, false, L, U>(s, sb, db, ab, u0, u_end); break;
    case 4: copy_rows<kNT, false, false, true, L, U>(s, sb, db, ab, u0, u_end); break;
    default: copy_rows<kNT, false, true, true, L, U>(s, sb, db, ab, u0, u_end); break;
  }
}

// copy_chunk for the unit width of a segment that carries no bf16 image.
template <bool kNT, bool kCast, bool kZero, bool kDup>
__device__ __forceinline__ void dispatch_units(uint32_t ul, const DevSeg &s, const char *sb, char *db, char *ab,
                                               uint32_t u0, uint32_t u_end) {
  switch (ul) {
    case 4: copy_chunk<u32x4, kNT, kCast, kZero, kDup>(s, sb, db, ab, u0, u_end); break;
    case 3: copy_chunk<uint64_t, kNT, kCast, kZero, kDup>(s, sb, db, ab, u0, u_end); break;
    case 2: copy_chunk<uint32_t, kNT, kCast, kZero, kDup>(s, sb, db, ab, u0, u_end); break;
    case 1: copy_chunk<uint16_t, kNT, kCast, kZero, kDup>(s, sb, db, ab, u0, u_end); break;
    default: copy_chunk<uint8_t, kNT, kCast, kZero, kDup>(s, sb, db, ab, u0, u_end); break;
  }
}

// Base address of buffer i: from the kernel-argument table, or (kTable) from
// a device-memory table of pointers for plans with more buffers than fit in
// kernel arguments.
template <bool kTable, typename B>
__device__ __forceinline__ char *base_of(const B &b, const uint64_t *tab, uint32_t i) {
  if constexpr (kTable) return reinterpret_cast<char *>(tab[i]);
  else return b.p[i];
}

// Copy chunks [c, c_end), starting from the segment that contains chunk c
// (persistent grid).
template <bool kNT, bool kTable>
__device__ __forceinline__ void copy_chunk_run(const DevSeg *__restrict__ segs, uint32_t n_segs, uint64_t n_chunks,
                                               uint64_t c, uint64_t c_end, const Bases &src, const Bases &dst,
                                               const uint64_t *src_tab, const uint64_t *dst_tab) {
  // Last segment whose first chunk is <= c.
  uint32_t lo = 0, hi = n_segs - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (segs[mid].chunk_begin <= c) lo = mid;
    else hi = mid - 1;
  }
  uint32_t si = lo;
  DevSeg s = segs[si];
  uint64_t s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;

  for (uint64_t nq; c < c_end; c += nq) {
    while (c >= s_end) {
      ++si;
      s = segs[si];
      s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;
    }
    // Up to kUnroll chunks of this segment in one step.
    nq = min(min(c_end, s_end) - c, (uint64_t)kUnroll);
    const uint32_t total = s.units();
    const uint32_t u0 = (uint32_t)(c - s.chunk_begin) * kChunkUnits;
    const uint32_t u_end = min(u0 + (uint32_t)nq * kChunkUnits, total);
    const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
    char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
    char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
    const uint32_t ops = s.ops(), ul = s.unit_log2();
    if (s.by_rows()) {
#pragma unroll 1
      for (uint32_t u = u0; u < u_end; u += kThreads * kRowStep)
        dispatch_rows<kNT, kThreads, kRowStep>(s, sb, db, ab, u, u_end);
      continue;
    }
    if (ops & 4) {  // duplicate to aux, with or without zero fill
      if (ops & 2) dispatch_units<kNT, false, true, true>(ul, s, sb, db, ab, u0, u_end);
      else dispatch_units<kNT, false, false, true>(ul, s, sb, db, ab, u0, u_end);
      continue;
    }
    if (ops & 2) {  // zero fill, with or without the bf16 image
      if (ops & 1) {
        if (ul == 4) copy_chunk<u32x4, kNT, true, true>(s, sb, db, ab, u0, u_end);
        else copy_chunk<uint32_t, kNT, true, true>(s, sb, db, ab, u0, u_end);
      } else {
        dispatch_units<kNT, false, true, false>(ul, s, sb, db, ab, u0, u_end);
      }
      continue;
    }
    if (ops & 1) {
      if (ul == 4) copy_chunk<u32x4, kNT, true>(s, sb, db, ab, u0, u_end);
      else copy_chunk<uint32_t, kNT, true>(s, sb, db, ab, u0, u_end);
      continue;
    }
    dispatch_units<kNT, false, false, false>(ul, s, sb, db, ab, u0, u_end);
  }
}

// Persistent grid (a tuning option).  With run == 0 every workgroup takes one
// contiguous run of chunks_per_block chunks (xcd_stride != 0: each XCD's
// workgroups cover one contiguous slice).  With run > 0 the chunks are dealt
// out round-robin in runs of `run` chunks, so the workgroups sweep the plan
// together; with xcd_stride != 0 as well (the grid is then a multiple of 8,
// and workgroup b runs on XCD b % 8), each XCD sweeps its own contiguous
// eighth, so that no page is touched from two XCDs' translation caches.
template <bool kNT, bool kTable>
__global__ __launch_bounds__(kThreads) void copy_plan_persistent_kernel(
    const DevSeg *__restrict__ segs, uint32_t n_segs, uint64_t n_chunks,
    uint64_t chunks_per_block, uint32_t xcd_stride, uint32_t run, Bases src, Bases dst,
    const uint64_t *__restrict__ src_tab, const uint64_t *__restrict__ dst_tab) {
  if (run) {
    uint64_t c1 = n_chunks, c = (uint64_t)blockIdx.x * run, step = (uint64_t)gridDim.x * run;
    if (xcd_stride) {
      const uint64_t x = blockIdx.x & 7;
      const uint64_t c0 = n_chunks * x / 8;
      c1 = n_chunks * (x + 1) / 8;
      c = c0 + (uint64_t)(blockIdx.x >> 3) * run;
      step = (uint64_t)(gridDim.x >> 3) * run;
    }
    for (; c < c1; c += step)
      copy_chunk_run<kNT, kTable>(segs, n_segs, n_chunks, c, min(c + run, c1), src, dst, src_tab, dst_tab);
    return;
  }
  uint64_t b = blockIdx.x;
  if (xcd_stride) b = (b & 7) * xcd_stride + (b >> 3);  // one contiguous slice per XCD
  const uint64_t c = b * chunks_per_block;
  if (c >= n_chunks) return;
  copy_chunk_run<kNT, kTable>(segs, n_segs, n_chunks, c, min(c + chunks_per_block, n_chunks), src, dst, src_tab,
                              dst_tab);
}

// Units [u0, u0 + L * U) of segment s (clipped to its `total` units) by a
// workgroup of L lanes, U units per lane: every load is issued before the
// first store.
template <typename T, bool kNT, bool kCast, bool kZero, bool kDup, int L, int U>
__device__ __forceinline__ void copy_units(const DevSeg &s, const char *sbase, char *dbase, char *abase, uint32_t u0,
                                           uint32_t total) {
  typedef typename std::conditional<kCast, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename C::type A;
  const T *src = reinterpret_cast<const T *>(sbase);
  T *dst = reinterpret_cast<T *>(dbase);
  A *aux = reinterpret_cast<A *>(abase);
  T *dup = reinterpret_cast<T *>(abase);
  T v[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t u = u0 + j * L + threadIdx.x;
    v[j] = T{};
    if constexpr (!kZero) {
      uint64_t so = s.src_off + u;
      if (s.rows > 1) {
        const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2());
        so = s.src_off + (uint64_t)row * s.src_stride + (u - row * s.len);
      }
      if (u < total) v[j] = ld<T, kNT>(src + so);
    }
  }
  // Destination offsets are recomputed rather than kept from the loads: with
  // four units per lane that holds the kernel at 66 VGPRs instead of 74, so
  // seven waves fit on each SIMD instead of six.
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t u = u0 + j * L + threadIdx.x;
    if (u < total) {
      uint64_t dof = s.dst_off + u, ao = s.aux_off + u;
      if (s.rows > 1) {
        const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2()), col = u - row * s.len;
        dof = s.dst_off + (uint64_t)row * s.dst_stride + col;
        ao = s.aux_off + (uint64_t)row * s.aux_stride + col;
      }
      st<T, kNT>(dst + dof, v[j]);
      if constexpr (kCast) st<A, kNT>(aux + ao, C::cast(v[j]));
      if constexpr (kDup) st<T, kNT>(dup + ao, v[j]);
    }
  }
}

// A buffer resource for raw (unstructured) accesses at 32-bit byte offsets from
// `base`, over the whole 4 GiB range (word 3: the gfx9-family raw-buffer
// configuration).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const char *base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), 0, -1, 0x00020000);
}

// Cache policy of buffer instructions: bit 1 is the non-temporal hint on gfx94x/gfx950.
template <bool kNT>
struct BufPolicy {
  static constexpr int value = kNT ? 2 : 0;
};

// One unit of T through a buffer instruction at a 32-bit byte offset.
template <typename T, int kPolicy>
__device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 16) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kPolicy);
  } else if constexpr (sizeof(T) == 8) {
    const auto w = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kPolicy);
    return (uint64_t)w[0] | ((uint64_t)w[1] << 32);
  } else if constexpr (sizeof(T) == 4) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kPolicy);
  } else if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, kPolicy);
  } else {
    return __builtin_amdgcn_raw_buffer_load_b8(r, off, 0, kPolicy);
  }
}

template <typename T, int kPolicy>
__device__ __forceinline__ void buf_store(T v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 16) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, kPolicy);
  } else if constexpr (sizeof(T) == 8) {
    typedef unsigned int v2u __attribute__((__vector_size__(8)));
    uint64_t x;
    memcpy(&x, &v, 8);
    const v2u w = {(unsigned)x, (unsigned)(x >> 32)};
    __builtin_amdgcn_raw_buffer_store_b64(w, r, off, 0, kPolicy);
  } else if constexpr (sizeof(T) == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, off, 0, kPolicy);
  } else if constexpr (sizeof(T) == 2) {
    __builtin_amdgcn_raw_buffer_store_b16(v, r, off, 0, kPolicy);
  } else {
    __builtin_amdgcn_raw_buffer_store_b8(v, r, off, 0, kPolicy);
  }
}

// copy_units with buffer instructions: each stream (source, destination,
// second destination) is one scalar base, the start of the piece's first row,
// plus a 32-bit per-lane byte offset, so a lane needs one VGPR per address
// instead of two.  In a one-row segment the offsets of a lane's units differ
// by constants, which the instructions' immediate offsets hold.  Row pitches
// are below 2^23 bytes (the plan emits longer ones row by row) and a piece
// spans at most 256 rows, so offsets stay below 2^31.  Loads and stores are
// masked exactly as in copy_units.
template <typename T, bool kNT, bool kCast, bool kZero, bool kDup, int L, int U>
__device__ __forceinline__ void copy_units_buf(const DevSeg &s, const char *sbase, char *dbase, char *abase,
                                               uint32_t u0, uint32_t total) {
  typedef typename std::conditional<kCast, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename C::type A;
  constexpr int cp = BufPolicy<kNT>::value;
  constexpr uint32_t B = sizeof(T);                          // bytes per unit
  constexpr uint32_t AB = kCast ? sizeof(A) : sizeof(T);     // second-destination bytes per unit
  const uint32_t tid = threadIdx.x;
  T v[U];
  if (s.rows == 1) {
    const __amdgpu_buffer_rsrc_t rs = raw_rsrc(sbase + (s.src_off + u0) * B);
    const __amdgpu_buffer_rsrc_t rd = raw_rsrc(dbase + (s.dst_off + u0) * B);
    const __amdgpu_buffer_rsrc_t ra = raw_rsrc(abase + (s.aux_off + u0) * AB);
    const uint32_t n = total - u0;  // units left in the segment from u0
#pragma unroll
    for (int j = 0; j < U; ++j) {
      v[j] = T{};
      if constexpr (!kZero)
        if (j * L + tid < n) v[j] = buf_load<T, cp>(rs, (j * L + tid) * B);
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (j * L + tid < n) {
        buf_store<T, cp>(v[j], rd, (j * L + tid) * B);
        if constexpr (kCast) buf_store<A, cp>(C::cast(v[j]), ra, (j * L + tid) * AB);
        if constexpr (kDup) buf_store<T, cp>(v[j], ra, (j * L + tid) * AB);
      }
    return;
  }
  const uint32_t row0 = magic_div(u0, s.magic, s.sh1(), s.sh2());
  const __amdgpu_buffer_rsrc_t rs = raw_rsrc(sbase + (s.src_off + (uint64_t)row0 * s.src_stride) * B);
  const __amdgpu_buffer_rsrc_t rd = raw_rsrc(dbase + (s.dst_off + (uint64_t)row0 * s.dst_stride) * B);
  const __amdgpu_buffer_rsrc_t ra = raw_rsrc(abase + (s.aux_off + (uint64_t)row0 * s.aux_stride) * AB);
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t u = u0 + j * L + tid;
    v[j] = T{};
    if constexpr (!kZero)
      if (u < total) {
        const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2());
        const uint32_t col = u - row * s.len;
        v[j] = buf_load<T, cp>(rs, ((row - row0) * s.src_stride + col) * B);
      }
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t u = u0 + j * L + tid;
    if (u < total) {
      const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2()), dr = row - row0;
      const uint32_t col = u - row * s.len;
      buf_store<T, cp>(v[j], rd, (dr * s.dst_stride + col) * B);
      if constexpr (kCast) buf_store<A, cp>(C::cast(v[j]), ra, (dr * s.aux_stride + col) * AB);
      if constexpr (kDup) buf_store<T, cp>(v[j], ra, (dr * s.aux_stride + col) * AB);
    }
  }
}

// One piece by `UnitsOf<T, kCast, kZero, kDup>` for the segment's unit width and what its ops ask for.
// 16-byte units first, which most segments have: every wave walks these scalar tests, and workgroups
// of several waves that only store are bound by scalar instructions, of which a CU issues one a cycle.
// 26 GiB of zeros by workgroups of 256 and 128 lanes: 6.4 and 6.1 TB/s with the ops tested before the
// unit and the order computed in 64 bits, 7.2 and 7.3 so.
template <template <typename, bool, bool, bool> class UnitsOf, typename... A>
__device__ __forceinline__ void dispatch_piece(const DevSeg &s, A... a) {
  const uint32_t ops = s.ops(), ul = s.unit_log2();
  if (ul == 4) {
    switch (ops) {
      case 0: UnitsOf<u32x4, false, false, false>::run(s, a...); break;
      case 1: UnitsOf<u32x4, true, false, false>::run(s, a...); break;
      case 2: UnitsOf<u32x4, false, true, false>::run(s, a...); break;
      case 3: UnitsOf<u32x4, true, true, false>::run(s, a...); break;
      case 4: UnitsOf<u32x4, false, false, true>::run(s, a...); break;
      default: UnitsOf<u32x4, false, true, true>::run(s, a...); break;
    }
    return;
  }
  if (ops & 1) {  // with the bf16 image: fp32
    if (ops & 2) UnitsOf<uint32_t, true, true, false>::run(s, a...);
    else UnitsOf<uint32_t, true, false, false>::run(s, a...);
    return;
  }
  auto elements = [&](auto zero, auto dup) {
    switch (ul) {
      case 3: UnitsOf<uint64_t, false, decltype(zero)::value, decltype(dup)::value>::run(s, a...); break;
      case 2: UnitsOf<uint32_t, false, decltype(zero)::value, decltype(dup)::value>::run(s, a...); break;
      case 1: UnitsOf<uint16_t, false, decltype(zero)::value, decltype(dup)::value>::run(s, a...); break;
      default: UnitsOf<uint8_t, false, decltype(zero)::value, decltype(dup)::value>::run(s, a...); break;
    }
  };
  if (ops & 4) {
    if (ops & 2) elements(std::true_type(), std::true_type());
    else elements(std::false_type(), std::true_type());
  } else {
    if (ops & 2) elements(std::true_type(), std::false_type());
    else elements(std::false_type(), std::false_type());
  }
}
template <bool kNT, int L, int U>
struct ByAddress {
  template <typename T, bool kCast, bool kZero, bool kDup>
  struct Units {
    __device__ static __forceinline__ void run(const DevSeg &s, const char *sb, char *db, char *ab, uint32_t u0,
                                               uint32_t total) {
      copy_units<T, kNT, kCast, kZero, kDup, L, U>(s, sb, db, ab, u0, total);
    }
  };
};
template <bool kNT, int L, int U>
struct ByBuffer {
  template <typename T, bool kCast, bool kZero, bool kDup>
  struct Units {
    __device__ static __forceinline__ void run(const DevSeg &s, const char *sb, char *db, char *ab, uint32_t u0,
                                               uint32_t total) {
      copy_units_buf<T, kNT, kCast, kZero, kDup, L, U>(s, sb, db, ab, u0, total);
    }
  };
};

// Units [u0, u0 + L * U) of segment s by a workgroup of L lanes.
template <bool kNT, int L, int U>
__device__ __forceinline__ void copy_piece(const DevSeg &s, const char *sb, char *db, char *ab, uint32_t u0,
                                           uint32_t total) {
  if (__builtin_expect(s.plain(), 1)) copy_units<u32x4, kNT, false, false, false, L, U>(s, sb, db, ab, u0, total);
  else if (s.by_rows()) dispatch_rows<kNT, L, U>(s, sb, db, ab, u0, total);
  else dispatch_piece<ByAddress<kNT, L, U>::template Units>(s, sb, db, ab, u0, total);
}

// copy_piece with every unit width but row units through buffer instructions.
template <bool kNT, int L, int U>
__device__ __forceinline__ void copy_piece_buf(const DevSeg &s, const char *sb, char *db, char *ab, uint32_t u0,
                                               uint32_t total) {
  if (s.by_rows()) dispatch_rows<kNT, L, U>(s, sb, db, ab, u0, total);
  else dispatch_piece<ByBuffer<kNT, L, U>::template Units>(s, sb, db, ab, u0, total);
}

// A descriptor in one scalar load of 64 bytes.  `p` is uniform over the wave
// and the table is never written while a kernel reads it.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ DevSeg load_seg(const DevSeg *p) {
  const u32x16 v = *reinterpret_cast<const __attribute__((address_space(4))) u32x16 *>(reinterpret_cast<uintptr_t>(p));
  DevSeg s;
  __builtin_memcpy(&s, &v, sizeof s);
  return s;
}

// Workgroup `w` of the pre-read of a plan's lookup tables (its chunk table,
// then its segment descriptors): the first workgroups of a copy launch read
// both once, with cached loads.  Every copy workgroup starts with a dependent
// load from the chunk table: after unrelated work those loads miss every
// cache, each workgroup waits on HBM before its first data load, and the
// launch ran 4.5% slower than one straight after another copy (whose table
// reads left the table in the memory-side cache).  Read here first, with every
// load in flight at once, the tables are in that cache when the copy's
// workgroups follow, which the hardware dispatches in order; nothing waits for
// them.  The XOR only keeps the loads; nothing is stored.
constexpr uint32_t kWarmUnits = 4;  // 16-byte units per lane
template <int L>
__device__ __forceinline__ void warm_tables(const uint32_t *chunk_seg, const DevSeg *segs, uint64_t n_chunks,
                                            uint32_t n_segs, uint32_t w) {
  // Whole 16-byte units of the chunk table: its last 1-3 words share a line with the ones before.
  const uint64_t na = n_chunks / 4, nb = (uint64_t)n_segs * (sizeof(DevSeg) / sizeof(u32x4));
  const u32x4 *a = reinterpret_cast<const u32x4 *>(chunk_seg), *b = reinterpret_cast<const u32x4 *>(segs);
  uint32_t acc = 0;
#pragma unroll
  for (uint32_t j = 0; j < kWarmUnits; ++j) {
    const uint64_t i = ((uint64_t)w * kWarmUnits + j) * L + threadIdx.x;
    if (i < na + nb) {
      const u32x4 v = i < na ? a[i] : b[i - na];
      acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
  }
  asm volatile("" ::"v"(acc));
}

// One workgroup of L lanes per piece of L * U units of a chunk (the default
// schedule: L = 64, U = 1, four 1 KB pieces per chunk).  A chunk of 256 units
// holds 256 / (L * U) pieces; workgroup w takes piece w % that of chunk
// w / that, and a piece past the end of its segment's last chunk does
// nothing.  Past the 2^32 - 1 lanes of one dimension the grid has rows
// (w = blockIdx.y * gridDim.x + blockIdx.x); workgroups past the last piece
// exit at once.  The segment depends on the chunk alone,
// so finding it runs on the scalar unit, once per wave: one load from the
// plan's chunk table (chunk_seg, by default), or a binary search whose upper
// levels stay in the scalar cache for every workgroup in flight.  With the
// search, small pieces repeat it for little data (256 lanes of one unit ran
// about 20% slower than 64 lanes of four); with the table, 1 KB pieces are
// the fastest shape.
//
// xcd_end != 0: pieces are dealt out to the XCDs in runs; see xcd_order.
template <bool kNT, bool kTable, int L, int U, bool kBuf>
__global__ __launch_bounds__(L) void copy_plan_kernel(const DevSeg *__restrict__ segs, uint64_t n_chunks,
                                                      SegHint hint, Bases src, Bases dst,
                                                      const uint64_t *__restrict__ src_tab,
                                                      const uint64_t *__restrict__ dst_tab, uint64_t xcd_end,
                                                      uint32_t xcd_log2, const uint32_t *__restrict__ chunk_seg,
                                                      uint32_t n_warm, uint32_t n_segs) {
  constexpr uint32_t kPieces = kChunkUnits / (L * U);  // pieces per chunk: 1, 2 or 4
  static_assert(kPieces * L * U == kChunkUnits, "a piece divides a chunk");
  uint64_t w = (uint64_t)blockIdx.y * gridDim.x + blockIdx.x;
  if constexpr (kBuf) {  // without buffer instructions, a launch with the chunk table takes copy_pieces_kernel
    w -= n_warm;
    if ((int32_t)(w >> 32) < 0) {
      warm_tables<L>(chunk_seg, segs, n_chunks, n_segs, blockIdx.x);
      return;
    }
  }
  w = xcd_order(w, xcd_end, xcd_log2);
  const uint64_t c = w / kPieces;
  if (c >= n_chunks) return;
  uint32_t lo;
  if (kBuf && chunk_seg) {  // the segment of every chunk, looked up
    lo = chunk_seg[c];
  } else {  // found by a binary search bounded by the hint
    const uint32_t b = (uint32_t)(c >> hint.shift);
    lo = hint.first[b];
    uint32_t hi = hint.first[b + 1];
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (segs[mid].chunk_begin <= c) lo = mid;
      else hi = mid - 1;
    }
  }
  const DevSeg s = segs[lo];
  const uint32_t total = s.units();
  const uint32_t u0 = (uint32_t)(c - s.chunk_begin) * kChunkUnits + (uint32_t)(w % kPieces) * (L * U);
  if (kPieces > 1 && u0 >= total) return;
  const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
  char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
  char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
  if constexpr (kBuf) copy_piece_buf<kNT, L, U>(s, sb, db, ab, u0, total);
  else copy_piece<kNT, L, U>(s, sb, db, ab, u0, total);
}

// copy_plan_kernel of the default launch: with the chunk table and 64-bit
// global addresses.  A workgroup lives for its chain of dependent scalar loads
// (arguments, chunk-table entry, descriptor, bases) and one round trip to HBM,
// so the chain is kept short: the leading arguments arrive in scalar registers
// (the build preloads 14 words of them), the descriptor is one 64-byte scalar
// load, and plans of at most 8 buffers a side (every arena plan) carry only
// those, 0.2 KB of arguments for the host to write per launch instead of 3 KB.
// Against copy_plan_kernel after a separate launch that read the tables (one
// process, same allocations, back to back / after a 512 MiB fill): 14.5 MB of
// traffic 13.5 / 16.0 us -> 8.7 / 12.0, 113 MB 27.7 / 33.7 -> 24.0 / 29.6,
// 1.0 GB 162 / 168 -> 157 / 162, 70 GB 10587 / 10594 -> 10549 / 10547.
template <bool kNT, bool kTable, int L, int U, typename B>
__global__ __launch_bounds__(L) void copy_pieces_kernel(const uint32_t *__restrict__ chunk_seg,
                                                        const DevSeg *__restrict__ segs, uint64_t n_chunks,
                                                        uint64_t xcd_end, uint32_t gx, uint32_t n_warm,
                                                        uint32_t xcd_log2, const uint64_t *__restrict__ src_tab,
                                                        const uint64_t *__restrict__ dst_tab, B src, B dst,
                                                        uint32_t n_segs) {
  constexpr uint32_t kPieces = kChunkUnits / (L * U);  // pieces per chunk: 1, 2 or 4
  static_assert(kPieces * L * U == kChunkUnits, "a piece divides a chunk");
  uint64_t w = (uint64_t)blockIdx.y * gx + blockIdx.x - n_warm;
  if ((int32_t)(w >> 32) < 0) {  // the sign: among the first n_warm
    warm_tables<L>(chunk_seg, segs, n_chunks, n_segs, blockIdx.x);
    return;
  }
  w = xcd_order(w, xcd_end, xcd_log2);
  const uint64_t c = w / kPieces;
  if (c >= n_chunks) return;
  const DevSeg s = load_seg(segs + chunk_seg[c]);
  const uint32_t total = s.units();
  const uint32_t u0 = (uint32_t)(c - s.chunk_begin) * kChunkUnits + (uint32_t)(w % kPieces) * (L * U);
  const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
  char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
  char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
  if (kPieces > 1 && u0 >= total) return;
  copy_piece<kNT, L, U>(s, sb, db, ab, u0, total);
}

// Writes the chunk table from the device segment table: segment k owns the
// chunks from its chunk_begin to the next segment's.  Built here, on the
// device, a plan's first call costs a few microseconds instead of a host fill
// and an upload of 4 bytes per chunk (79 MB on Llama-2-7B, about 27 ms).
__global__ __launch_bounds__(256) void fill_chunk_table_kernel(const DevSeg *__restrict__ segs, uint32_t nseg,
                                                               uint64_t n_chunks, uint32_t *__restrict__ out) {
  for (uint32_t k = blockIdx.x; k < nseg; k += gridDim.x) {
    const uint64_t c0 = segs[k].chunk_begin;
    const uint64_t c1 = k + 1 < nseg ? segs[k + 1].chunk_begin : n_chunks;
    for (uint64_t c = c0 + threadIdx.x; c < c1; c += 256) out[c] = k;
  }
}

// ---------------------------------------------------------------------------
// Device bookkeeping
// ---------------------------------------------------------------------------

struct DeviceProps {
  int cus = 0;
  int resident_blocks[2] = {0, 0};  // copy_plan_persistent_kernel<false/true> blocks per CU
};

std::mutex g_dev_mu;
std::vector<DeviceProps> g_dev_props;

template <bool kNT>
void persistent_occupancy(int *out) {
  int v = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, copy_plan_persistent_kernel<kNT, false>, kThreads, 0) !=
          hipSuccess ||
      v <= 0) {
    (void)hipGetLastError();
    v = 4;
  }
  *out = v;
}

int current_device(int *dev, int *cus, int *resident_nt, int *resident_t) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0) {
    (void)hipGetLastError();
    return fail(EMRS_ERR_NO_DEVICE, "no HIP device is visible");
  }
  e = hipGetDevice(dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  std::lock_guard<std::mutex> lk(g_dev_mu);
  if ((int)g_dev_props.size() < n) g_dev_props.resize(n);
  if (g_dev_props[*dev].cus == 0) {
    int v = 0;
    e = hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, *dev);
    if (e != hipSuccess) return hip_fail(e, "hipDeviceGetAttribute");
    g_dev_props[*dev].cus = v > 0 ? v : 1;
    persistent_occupancy<false>(&g_dev_props[*dev].resident_blocks[0]);
    persistent_occupancy<true>(&g_dev_props[*dev].resident_blocks[1]);
  }
  *cus = g_dev_props[*dev].cus;
  *resident_t = g_dev_props[*dev].resident_blocks[0];
  *resident_nt = g_dev_props[*dev].resident_blocks[1];
  return EMRS_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// Plan
// ---------------------------------------------------------------------------

struct emrs_plan {
  std::vector<DevSeg> segs;
  std::vector<uint32_t> origin;              // input segment of each device segment
  uint64_t n_chunks = 0;
  SegHint hint{};                            // search bounds of the one-workgroup-per-chunk kernel
  std::vector<uint64_t> src_bytes, dst_bytes;
  std::vector<uint8_t> src_used, dst_used;  // buffers referenced by a non-empty segment
  emrs_plan_stats stats{};
  std::mutex mu;
  std::vector<DevSeg *> dev_tables;  // per device, uploaded on first use
  // Per device, uploaded on first use when emrs_tuning.chunk_index is set:
  // the device segment of every chunk (4 bytes per 4 KB chunk).
  std::vector<uint32_t *> chunk_tables;
  // Plans with more than kArgBuffers buffers on a side: per device, the
  // pointer table of the first execution and the base pointers it holds.
  std::vector<uint64_t *> ptr_tables;
  std::vector<std::vector<uint64_t>> ptr_contents;
  // For those same bases: the segment table with every offset made absolute
  // (units from abs_base, the lowest referenced base), per device.
  std::vector<DevSeg *> abs_tables;
  std::vector<uint64_t> abs_base;
  // Per device: one event recorded after each launch that may still be running (an event is
  // reused once its launch has finished).  Destroying the plan frees its tables in stream order
  // after these launches, and waits for nothing else.
  std::vector<std::vector<hipEvent_t>> launch_events;
  // Per device: the flags of a comparison's first pass, all zero, between two comparisons.
  std::vector<uint32_t *> differ_flags;
  bool captured = false;  // a launch was recorded into a graph: destroy drains the device first
};

namespace {

// The plan's own device tables are stream-ordered allocations: made and
// filled synchronously on first use, and freed by emrs_plan_destroy on a
// library stream once the plan's launches have finished.
hipError_t table_alloc(void **out, size_t bytes, hipStream_t st) {
  *out = nullptr;
  const hipError_t e = hipMallocAsync(out, bytes, st);
  if (e != hipSuccess) *out = nullptr;
  return e;
}

int table_upload(void **out, const void *host, size_t bytes, hipStream_t st, const char *what) {
  hipError_t e = table_alloc(out, bytes, st);
  if (e != hipSuccess) return hip_fail(e, what);
  e = hipMemcpyAsync(*out, host, bytes, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);  // complete before any stream may read it
  if (e != hipSuccess) {
    (void)hipFreeAsync(*out, st);
    (void)hipStreamSynchronize(st);
    *out = nullptr;
    return hip_fail(e, what);
  }
  return EMRS_OK;
}

// Per device, the library's own stream on which destroyed plans free their
// tables (default priority, not blocking the null stream); nullptr if it
// could not be made.
hipStream_t free_stream(int dev) {
  static std::mutex mu;
  static std::vector<hipStream_t> streams;
  std::lock_guard<std::mutex> lk(mu);
  if ((int)streams.size() <= dev) streams.resize(dev + 1, nullptr);
  if (!streams[dev]) {
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess) streams[dev] = s;
    else (void)hipGetLastError();
  }
  return streams[dev];
}

// Record that the plan's tables are in use by the work just enqueued on `st`.
// Under graph capture nothing is recorded: the graph may replay any time, so
// destroy then drains the device instead.
int note_launch(emrs_plan *plan, int dev, hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  hipError_t e = hipStreamIsCapturing(st, &cs);
  if (e != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
  std::lock_guard<std::mutex> lk(plan->mu);
  if (cs != hipStreamCaptureStatusNone) {
    plan->captured = true;
    return EMRS_OK;
  }
  if ((int)plan->launch_events.size() <= dev) plan->launch_events.resize(dev + 1);
  std::vector<hipEvent_t> &evs = plan->launch_events[dev];
  hipEvent_t ev = nullptr;
  bool not_ready = false;
  for (hipEvent_t x : evs) {
    const hipError_t q = hipEventQuery(x);
    if (q == hipSuccess) {  // its launch has finished: reuse it
      ev = x;
      break;
    }
    not_ready = not_ready || q == hipErrorNotReady;
  }
  // A running launch's query answers hipErrorNotReady, which is no failure: do not leave it
  // behind as this thread's last error.
  if (not_ready) (void)hipGetLastError();
  if (!ev) {
    e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e != hipSuccess) return hip_fail(e, "hipEventCreateWithFlags");
    evs.push_back(ev);
  }
  e = hipEventRecord(ev, st);
  if (e != hipSuccess) return hip_fail(e, "hipEventRecord");
  return EMRS_OK;
}

// Second destination of a segment: its bf16 image (cast; offsets in units
// of half the segment's unit) or a duplicate (dup; offsets in the segment's
// own units): buffer, offset and row stride.
struct Aux {
  bool on = false;    // cast or dup
  bool cast = false;  // EMRS_SEG_CAST_BF16
  bool dup = false;   // EMRS_SEG_DUP
  bool zero = false;  // the segment writes zeros (EMRS_SEG_ZERO_FILL)
  uint32_t buf = 0;
  uint64_t off = 0, stride = 0;
};

struct Builder {
  std::vector<DevSeg> out;
  std::vector<uint32_t> origin;  // input segment of each pushed segment
  uint32_t cur_origin = 0;       // input segment being emitted
  uint8_t cur_elem_log2 = 0;     // its element size
  uint64_t chunks = 0;
  uint64_t vec_bytes = 0, scalar_bytes = 0;

  // A copy whose offsets, length and strides count (1 << ul) bytes, optionally
  // with its bf16 image; `by_rows`: in row units.  Splits to the kernel's
  // 32-bit limits.
  void emit(uint32_t sbuf, uint32_t dbuf, uint32_t ul, uint64_t so, uint64_t dof, uint64_t len,
            uint64_t rows, uint64_t ss, uint64_t ds, Aux ax = Aux(), bool by_rows = false) {
    if (len == 0 || rows == 0) return;
    if (rows > 1 && ss == len && ds == len && (!ax.on || ax.stride == len)) {  // contiguous
      len *= rows;
      rows = 1;
    }
    if (rows == 1) {
      for (uint64_t off = 0; off < len; off += kMaxUnitsPerSeg) {
        const uint64_t n = std::min<uint64_t>(kMaxUnitsPerSeg, len - off);
        push(sbuf, dbuf, ul, so + off, dof + off, (uint32_t)n, 1, 0, 0, ax, ax.off + off, 0, by_rows);
      }
      return;
    }
    // Bytes per second-destination unit: half a unit for a bf16 image, a whole one for a duplicate.
    const uint64_t aub = ax.on ? (ax.cast ? (1ull << ul) / 2 : (1ull << ul)) : 0;
    if (len >= kMaxUnitsPerSeg || (ss << ul) >= kMaxPitchBytes || (ds << ul) >= kMaxPitchBytes ||
        ax.stride * aub >= kMaxPitchBytes) {
      for (uint64_t r = 0; r < rows; ++r)
        for (uint64_t off = 0; off < len; off += kMaxUnitsPerSeg) {
          const uint64_t n = std::min<uint64_t>(kMaxUnitsPerSeg, len - off);
          push(sbuf, dbuf, ul, so + r * ss + off, dof + r * ds + off, (uint32_t)n, 1, 0, 0, ax,
               ax.off + r * ax.stride + off, 0, by_rows);
        }
      return;
    }
    const uint64_t rows_per = std::max<uint64_t>(1, kMaxUnitsPerSeg / len);
    for (uint64_t r = 0; r < rows; r += rows_per) {
      const uint64_t n = std::min<uint64_t>(rows_per, rows - r);
      push(sbuf, dbuf, ul, so + r * ss, dof + r * ds, (uint32_t)len, (uint32_t)n, (uint32_t)ss, (uint32_t)ds,
           ax, ax.off + r * ax.stride, (uint32_t)ax.stride, by_rows);
    }
  }

  void push(uint32_t sbuf, uint32_t dbuf, uint32_t ul, uint64_t so, uint64_t dof, uint32_t len, uint32_t rows,
            uint32_t ss, uint32_t ds, const Aux &ax, uint64_t aoff, uint32_t astride, bool by_rows) {
    DevSeg d{};
    d.src_off = so;
    d.dst_off = dof;
    d.chunk_begin = chunks;
    d.len = len;
    d.rows = rows;
    d.src_stride = rows > 1 ? ss : 0;
    d.dst_stride = rows > 1 ? ds : 0;
    const uint32_t ops = (ax.cast ? 1u : 0u) | (ax.zero ? 2u : 0u) | (ax.dup ? 4u : 0u);
    const uint64_t row_bytes = (uint64_t)len << ul;
    // A last piece under 16 bytes of a row cut at kMaxUnitsPerSeg goes element by element.
    const bool row_units = by_rows && row_bytes >= 16;
    d.set_kind(row_units ? kRowUnits : ul, cur_elem_log2, ops, row_units && row_bytes >= kLineRowBytes);
    uint32_t magic = 0, sh1 = 0, sh2 = 0;
    make_magic(d.row_units(), &magic, &sh1, &sh2);
    d.set_division(magic, sh1, sh2);
    d.set_bufs(sbuf, dbuf, ax.on ? ax.buf : dbuf);
    d.aux_off = ax.on ? aoff : 0;
    d.aux_stride = ax.on && rows > 1 ? astride : 0;
    chunks += ((uint64_t)d.units() + kChunkUnits - 1) / kChunkUnits;
    out.push_back(d);
    origin.push_back(cur_origin);
  }
};

// Search bounds per bucket of 2^shift chunks, with at most kHintBuckets
// buckets: first[b] is the segment holding chunk b << shift (the last segment
// past the end).
void make_hint(const std::vector<DevSeg> &segs, uint64_t n_chunks, SegHint *h) {
  const uint32_t last = segs.empty() ? 0 : (uint32_t)segs.size() - 1;
  h->shift = 0;
  while (n_chunks && ((n_chunks - 1) >> h->shift) >= kHintBuckets) ++h->shift;
  for (uint32_t b = 0; b <= kHintBuckets; ++b) {
    const uint64_t c = (uint64_t)b << h->shift;
    if (c >= n_chunks) {
      h->first[b] = last;
      continue;
    }
    // Last segment whose first chunk is <= c.
    auto it = std::upper_bound(segs.begin(), segs.end(), c,
                               [](uint64_t v, const DevSeg &d) { return v < d.chunk_begin; });
    h->first[b] = (uint32_t)(it - segs.begin()) - 1;
  }
}

int log2_of(uint32_t eb) {
  switch (eb) {
    case 1: return 0;
    case 2: return 1;
    case 4: return 2;
    case 8: return 3;
    default: return -1;
  }
}

// Byte extent end of a strided segment (128-bit: cannot overflow).
unsigned __int128 extent_end(uint64_t off, uint64_t len, uint64_t rows, uint64_t stride, uint32_t eb) {
  return ((unsigned __int128)off + (unsigned __int128)(rows - 1) * stride + len) * eb;
}

int check_disjoint(const emrs_segment *segs, uint64_t n_segs) {
  struct Iv {
    uint32_t buf;
    uint64_t b, e;
  };
  uint64_t total_rows = 0;
  for (uint64_t i = 0; i < n_segs; ++i)
    if (segs[i].len) total_rows += segs[i].rows * ((segs[i].flags & (EMRS_SEG_CAST_BF16 | EMRS_SEG_DUP)) ? 2 : 1);
  if (total_rows > (1ull << 27))
    return fail(EMRS_ERR_INVALID_ARGUMENT, "disjointness check: too many rows to check");
  std::vector<Iv> iv;
  iv.reserve(total_rows);
  for (uint64_t i = 0; i < n_segs; ++i) {
    const emrs_segment &s = segs[i];
    if (!s.len) continue;
    for (uint64_t r = 0; r < s.rows; ++r) {
      const uint64_t b = (s.dst_off + r * s.dst_stride) * s.elem_bytes;
      iv.push_back({s.dst_buf, b, b + s.len * s.elem_bytes});
      if (s.flags & (EMRS_SEG_CAST_BF16 | EMRS_SEG_DUP)) {
        const uint64_t w = (s.flags & EMRS_SEG_CAST_BF16) ? 2 : s.elem_bytes;
        const uint64_t a = (s.aux_off + r * s.aux_stride) * w;
        iv.push_back({s.aux_buf, a, a + s.len * w});
      }
    }
  }
  std::sort(iv.begin(), iv.end(), [](const Iv &a, const Iv &b) { return a.buf != b.buf ? a.buf < b.buf : a.b < b.b; });
  for (size_t i = 1; i < iv.size(); ++i) {
    if (iv[i].buf == iv[i - 1].buf && iv[i].b < iv[i - 1].e) {
      char msg[160];
      snprintf(msg, sizeof msg, "destination ranges overlap in buffer %u at byte %llu", iv[i].buf,
               (unsigned long long)iv[i].b);
      return fail(EMRS_ERR_OVERLAP, msg);
    }
  }
  return EMRS_OK;
}

// Base pointers of an execution or comparison, checked (only buffers that
// some segment references) and laid out for the launch.
struct ResolvedBases {
  Bases src{}, dst{};
  bool table = false;         // pointers go through a device table: src then dst
  std::vector<uint64_t> ptrs;
};

// out_of_place: a destination buffer may overlap no other referenced buffer
// (an execution); a comparison only reads, so there any buffers may overlap.
int resolve_bases(const emrs_plan *plan, void *const *src_bases, void *const *dst_bases, ResolvedBases *rb,
                  bool out_of_place = true) {
  const uint32_t ns = plan->stats.n_src_bufs, nd = plan->stats.n_dst_bufs;
  if ((ns && !src_bases) || (nd && !dst_bases))
    return fail(EMRS_ERR_INVALID_ARGUMENT, "base pointer array is NULL");
  // Only buffers that some segment references are checked: an unreferenced
  // buffer may be NULL or alias anything.
  struct Iv {
    uintptr_t b, e;
    bool dst;
  };
  std::vector<Iv> iv;
  iv.reserve(ns + nd);
  for (uint32_t i = 0; i < ns; ++i) {
    if (!plan->src_used[i]) continue;
    const uintptr_t b = reinterpret_cast<uintptr_t>(src_bases[i]);
    if (!b) return fail(EMRS_ERR_INVALID_ARGUMENT, "source base is NULL");
    if (b % 16) return fail(EMRS_ERR_MISALIGNED, "source base is not 16-byte aligned");
    if (plan->src_bytes[i]) iv.push_back({b, b + plan->src_bytes[i], false});
  }
  for (uint32_t i = 0; i < nd; ++i) {
    if (!plan->dst_used[i]) continue;
    const uintptr_t b = reinterpret_cast<uintptr_t>(dst_bases[i]);
    if (!b) return fail(EMRS_ERR_INVALID_ARGUMENT, "destination base is NULL");
    if (b % 16) return fail(EMRS_ERR_MISALIGNED, "destination base is not 16-byte aligned");
    if (plan->dst_bytes[i]) iv.push_back({b, b + plan->dst_bytes[i], true});
  }
  // Out of place: no destination range may overlap another referenced range.
  // Sweep in address order; an earlier range overlaps the current one exactly
  // when its end lies past the current start.
  if (out_of_place) {
    std::sort(iv.begin(), iv.end(), [](const Iv &x, const Iv &y) { return x.b < y.b; });
    uintptr_t end_src = 0, end_dst = 0;
    for (const Iv &x : iv) {
      if (x.b < end_dst)
        return fail(EMRS_ERR_ALIAS, x.dst ? "two destination buffers overlap" : "a source buffer overlaps a destination buffer");
      if (x.dst && x.b < end_src) return fail(EMRS_ERR_ALIAS, "a source buffer overlaps a destination buffer");
      (x.dst ? end_dst : end_src) = std::max(x.dst ? end_dst : end_src, x.e);
    }
  }
  rb->table = ns > kArgBuffers || nd > kArgBuffers;
  if (rb->table) {
    rb->ptrs.resize((size_t)ns + nd);
    for (uint32_t i = 0; i < ns; ++i) rb->ptrs[i] = reinterpret_cast<uint64_t>(src_bases[i]);
    for (uint32_t i = 0; i < nd; ++i) rb->ptrs[ns + i] = reinterpret_cast<uint64_t>(dst_bases[i]);
  } else {
    for (uint32_t i = 0; i < ns; ++i) rb->src.p[i] = static_cast<char *>(src_bases[i]);
    for (uint32_t i = 0; i < nd; ++i) rb->dst.p[i] = static_cast<char *>(dst_bases[i]);
  }
  return EMRS_OK;
}

// The device pointer table of an execution or comparison (nullptr when the
// bases travel in kernel arguments).  The plan keeps, per device, the table of
// the first call and reuses it while the bases are the same: it is uploaded
// synchronously and never written again, so any stream may read it.  Calls
// with other bases get a stream-ordered table of their own (*owned = true),
// which the caller frees on the same stream after the launch.
int pointer_table(emrs_plan *plan, int dev, const ResolvedBases &rb, hipStream_t st, uint64_t **out, bool *owned) {
  *out = nullptr;
  *owned = false;
  if (!rb.table) return EMRS_OK;
  const size_t bytes = rb.ptrs.size() * sizeof(uint64_t);
  {
    std::lock_guard<std::mutex> lk(plan->mu);
    if ((int)plan->ptr_tables.size() <= dev) {
      plan->ptr_tables.resize(dev + 1, nullptr);
      plan->ptr_contents.resize(dev + 1);
    }
    if (plan->ptr_tables[dev]) {
      if (plan->ptr_contents[dev] == rb.ptrs) {
        *out = plan->ptr_tables[dev];
        return EMRS_OK;
      }
    } else {
      if (int rc = refuse_capture(st, "the first call of a plan on a device")) return rc;
      uint64_t *t = nullptr;
      if (int rc = table_upload(reinterpret_cast<void **>(&t), rb.ptrs.data(), bytes, st, "uploading the pointer table"))
        return rc;
      plan->ptr_tables[dev] = t;
      plan->ptr_contents[dev] = rb.ptrs;
      *out = t;
      return EMRS_OK;
    }
  }
  // Other bases than the cached ones: a table of this call's own, which a
  // captured graph could not replay (its host copy is this call's).
  if (int rc = refuse_capture(st, "a call whose base pointers differ from the plan's first call")) return rc;
  *owned = true;
  hipError_t e = hipMallocAsync(reinterpret_cast<void **>(out), bytes, st);
  if (e != hipSuccess) {
    *out = nullptr;
    return hip_fail(e, "hipMallocAsync(pointer table)");
  }
  e = hipMemcpyAsync(*out, rb.ptrs.data(), bytes, hipMemcpyHostToDevice, st);
  if (e != hipSuccess) {
    (void)hipFreeAsync(*out, st);
    *out = nullptr;
    return hip_fail(e, "hipMemcpyAsync(pointer table)");
  }
  return EMRS_OK;
}

// The plan's segment table on device `dev` resolved against the bases of its
// cached pointer table: every offset counts units from *common, the lowest
// referenced base, and every buffer id is 0, so the copy kernel looks up no
// base pointer at all.  Built and uploaded synchronously on first use, like
// the pointer table, and never written again.  *out = nullptr when the bases
// are not the cached ones (the caller then uses the pointer table).
int resolved_table(emrs_plan *plan, int dev, const ResolvedBases &rb, hipStream_t st, DevSeg **out,
                   char **common) {
  *out = nullptr;
  std::lock_guard<std::mutex> lk(plan->mu);
  if ((int)plan->ptr_tables.size() <= dev || !plan->ptr_tables[dev] || plan->ptr_contents[dev] != rb.ptrs)
    return EMRS_OK;
  if ((int)plan->abs_tables.size() <= dev) {
    plan->abs_tables.resize(dev + 1, nullptr);
    plan->abs_base.resize(dev + 1, 0);
  }
  if (!plan->abs_tables[dev]) {
    if (int rc = refuse_capture(st, "the first call of a plan on a device")) return rc;
    const uint32_t ns = plan->stats.n_src_bufs, nd = plan->stats.n_dst_bufs;
    uint64_t lo = ~0ull;
    for (uint32_t i = 0; i < ns; ++i)
      if (plan->src_used[i]) lo = std::min(lo, rb.ptrs[i]);
    for (uint32_t i = 0; i < nd; ++i)
      if (plan->dst_used[i]) lo = std::min(lo, rb.ptrs[ns + i]);
    // Referenced bases are 16-byte aligned, so every difference is a whole
    // number of units.  Unreferenced buffers (a zero fill's source) may be
    // NULL; their offsets are never used.
    auto units_from_lo = [lo](uint64_t p, uint32_t log2) -> uint64_t { return p >= lo ? (p - lo) >> log2 : 0; };
    std::vector<DevSeg> segs = plan->segs;
    for (DevSeg &d : segs) {
      const uint32_t ul = d.off_log2(), ops = d.ops();
      const uint32_t aux_log2 = (ops & 1) ? ul - 1 : ul;  // a bf16 image unit is half a unit
      d.src_off = (ops & 2) ? 0 : d.src_off + units_from_lo(rb.ptrs[d.src_buf()], ul);
      d.dst_off += units_from_lo(rb.ptrs[ns + d.dst_buf()], ul);
      d.aux_off += units_from_lo(rb.ptrs[ns + d.aux_buf()], aux_log2);
      d.set_bufs(0, 0, 0);
    }
    const size_t bytes = segs.size() * sizeof(DevSeg);
    DevSeg *t = nullptr;
    if (int rc = table_upload(reinterpret_cast<void **>(&t), segs.data(), bytes, st, "uploading the resolved plan table"))
      return rc;
    plan->abs_tables[dev] = t;
    plan->abs_base[dev] = lo;
  }
  *out = plan->abs_tables[dev];
  *common = reinterpret_cast<char *>(plan->abs_base[dev]);
  return EMRS_OK;
}

// The device segment of every chunk on device `dev`, written on the device
// from its segment table `segs` on first use and never written again.
int chunk_table(emrs_plan *plan, int dev, hipStream_t st, const DevSeg *segs, uint32_t **out) {
  std::lock_guard<std::mutex> lk(plan->mu);
  if ((int)plan->chunk_tables.size() <= dev) plan->chunk_tables.resize(dev + 1, nullptr);
  if (!plan->chunk_tables[dev]) {
    // The table only spares each workgroup its search.  While the stream captures a graph it
    // cannot be built (that would record an allocation), so the launch searches instead; a
    // later call outside a capture builds it.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t ce = hipStreamIsCapturing(st, &cs);
    if (ce != hipSuccess) return hip_fail(ce, "hipStreamIsCapturing");
    if (cs != hipStreamCaptureStatusNone) {
      *out = nullptr;
      return EMRS_OK;
    }
    if (plan->segs.size() > 0xffffffffull) return fail(EMRS_ERR_INVALID_ARGUMENT, "too many device segments");
    const size_t bytes = plan->n_chunks * sizeof(uint32_t);
    uint32_t *t = nullptr;
    hipError_t e = table_alloc(reinterpret_cast<void **>(&t), bytes, st);
    if (e == hipErrorOutOfMemory) {
      // The table only spares each workgroup its search: with no room for it,
      // this launch searches instead, and the next call tries again.
      (void)hipGetLastError();
      *out = nullptr;
      return EMRS_OK;
    }
    if (e != hipSuccess) return hip_fail(e, "hipMallocAsync(chunk table)");
    const uint32_t nseg = (uint32_t)plan->segs.size();
    hipLaunchKernelGGL(fill_chunk_table_kernel, dim3(std::min<uint32_t>(nseg, 65535)), dim3(256), 0, st, segs, nseg,
                       plan->n_chunks, t);
    e = hipGetLastError();
    // Later calls may come on other streams: the table is complete before it is published.
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
      (void)hipFreeAsync(t, st);
      (void)hipStreamSynchronize(st);
      return hip_fail(e, "building the chunk table");
    }
    plan->chunk_tables[dev] = t;
  }
  *out = plan->chunk_tables[dev];
  return EMRS_OK;
}

// The chunk table already on device `dev`, or nullptr: allocates nothing.
const uint32_t *existing_chunk_table(emrs_plan *plan, int dev) {
  std::lock_guard<std::mutex> lk(plan->mu);
  return (int)plan->chunk_tables.size() > dev ? plan->chunk_tables[dev] : nullptr;
}

// The plan's segment table on device `dev`, uploaded on first use.
int device_table(emrs_plan *plan, int dev, hipStream_t st, DevSeg **table) {
  std::lock_guard<std::mutex> lk(plan->mu);
  if ((int)plan->dev_tables.size() <= dev) plan->dev_tables.resize(dev + 1, nullptr);
  if (!plan->dev_tables[dev]) {
    if (int rc = refuse_capture(st, "the first call of a plan on a device")) return rc;
    const size_t bytes = plan->segs.size() * sizeof(DevSeg);
    DevSeg *t = nullptr;
    if (int rc = table_upload(reinterpret_cast<void **>(&t), plan->segs.data(), bytes, st, "uploading the plan table"))
      return rc;
    plan->dev_tables[dev] = t;
  }
  *table = plan->dev_tables[dev];
  return EMRS_OK;
}

// ---------------------------------------------------------------------------
// Compare kernel
// ---------------------------------------------------------------------------

// Device accumulators of one group (emrs_compare_stats minus the element
// count, which the host knows).  Maxima are non-negative floats, ordered as
// their bit patterns.
struct GroupAcc {
  unsigned long long mismatches;
  unsigned long long nonfinite;
  double sum_sq_diff;
  double sum_sq_expected;
  unsigned int max_abs_bits;
  unsigned int max_rel_bits;
};

struct LaneAcc {
  uint32_t mismatches = 0, nonfinite = 0;
  double sq_diff = 0.0, sq_exp = 0.0;
  float max_abs = 0.0f, max_rel = 0.0f;
};

__device__ __forceinline__ void cmp_float(LaneAcc &a, uint32_t e_bits, uint32_t g_bits) {
  const float e = __uint_as_float(e_bits), g = __uint_as_float(g_bits);
  if (fabsf(e) <= 3.402823466e38f) a.sq_exp += (double)e * (double)e;
  if (e_bits == g_bits) return;
  ++a.mismatches;
  const float d = fabsf(g - e);
  if (!(d <= 3.402823466e38f)) {  // NaN or infinite difference
    ++a.nonfinite;
    return;
  }
  a.sq_diff += (double)d * (double)d;
  a.max_abs = fmaxf(a.max_abs, d);
  a.max_rel = fmaxf(a.max_rel, d / (fabsf(e) + 1e-12f));
}

// Compare one unit (1, 2, 4, 8 or 16 bytes held in w[0..3]) element by element: its elements [first, last).
__device__ __forceinline__ void cmp_words(LaneAcc &a, const uint32_t *e, const uint32_t *g, uint32_t unit_bytes,
                                          uint32_t elem_log2, uint32_t first = 0, uint32_t last = 16) {
  switch (elem_log2) {
    case 2:  // fp32
      for (uint32_t k = 0; k < unit_bytes / 4; ++k)
        if (k >= first && k < last) cmp_float(a, e[k], g[k]);
      break;
    case 1:  // bf16
      for (uint32_t k = 0; k < unit_bytes / 2; ++k) {
        if (k < first || k >= last) continue;
        const uint32_t sh = (k & 1) * 16;
        cmp_float(a, ((e[k >> 1] >> sh) & 0xffffu) << 16, ((g[k >> 1] >> sh) & 0xffffu) << 16);
      }
      break;
    case 0:  // bytes: bits only
      for (uint32_t k = 0; k < unit_bytes; ++k) {
        const uint32_t sh = (k & 3) * 8;
        a.mismatches += ((e[k >> 2] >> sh) & 0xffu) != ((g[k >> 2] >> sh) & 0xffu);
      }
      break;
    default:  // 8-byte elements: bits only
      for (uint32_t k = 0; k < unit_bytes / 8; ++k)
        if (k >= first && k < last) a.mismatches += (e[2 * k] != g[2 * k]) || (e[2 * k + 1] != g[2 * k + 1]);
      break;
  }
}

template <typename T>
__device__ __forceinline__ void words_of(const T &v, uint32_t *w) {
  if constexpr (sizeof(T) == 16) {
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
  } else if constexpr (sizeof(T) == 8) {
    w[0] = (uint32_t)v; w[1] = (uint32_t)(v >> 32);
  } else {
    w[0] = (uint32_t)v;
  }
}

template <typename A>
__device__ __forceinline__ void aux_words_of(const A &v, uint32_t *w) {
  if constexpr (sizeof(A) == 8) {
    w[0] = v.x; w[1] = v.y;
  } else {
    w[0] = (uint32_t)v;
  }
}

// Compare units [u0, u_end) of segment s (at most kStepUnits); with a cast,
// also its bf16 image; with a duplicate, also the second copy.
template <typename T>
__device__ __forceinline__ void compare_chunk(const DevSeg &s, const char *sbase, const char *dbase,
                                              const char *abase, uint32_t u0, uint32_t u_end, LaneAcc &m,
                                              LaneAcc &x) {
  typedef typename std::conditional<sizeof(T) == 16 || sizeof(T) == 4, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename C::type A;
  const T *src = reinterpret_cast<const T *>(sbase);
  const T *dst = reinterpret_cast<const T *>(dbase);
  const A *aux = reinterpret_cast<const A *>(abase);
  for (uint32_t j = 0; j < kUnroll; ++j) {
    const uint32_t u = u0 + j * kThreads + threadIdx.x;
    if (u >= u_end) break;
    uint64_t so = s.src_off + u, dof = s.dst_off + u, ao = s.aux_off + u;
    if (s.rows > 1) {
      const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2()), col = u - row * s.len;
      so = s.src_off + (uint64_t)row * s.src_stride + col;
      dof = s.dst_off + (uint64_t)row * s.dst_stride + col;
      ao = s.aux_off + (uint64_t)row * s.aux_stride + col;
    }
    const uint32_t ops = s.ops();
    const T e = (ops & 2) ? T{} : ld<T, true>(src + so);
    const T g = ld<T, true>(dst + dof);
    uint32_t ew[4] = {0, 0, 0, 0}, gw[4] = {0, 0, 0, 0};
    words_of(e, ew);
    words_of(g, gw);
    cmp_words(m, ew, gw, (uint32_t)sizeof(T), s.elem_log2());
    if (ops & 4) {
      uint32_t dw[4] = {0, 0, 0, 0};
      words_of(ld<T, true>(reinterpret_cast<const T *>(abase) + ao), dw);
      cmp_words(x, ew, dw, (uint32_t)sizeof(T), s.elem_log2());
    }
    if constexpr (sizeof(T) == 16 || sizeof(T) == 4) {
      if (ops & 1) {
        uint32_t ea[2] = {0, 0}, ga[2] = {0, 0};
        aux_words_of(C::cast(e), ea);
        aux_words_of(ld<A, true>(aux + ao), ga);
        cmp_words(x, ea, ga, (uint32_t)sizeof(A), 1);
      }
    }
  }
}

// compare_chunk for row units: every element of a row once, whichever units hold it.
__device__ __forceinline__ void compare_rows(const DevSeg &s, const char *sbase, const char *dbase, const char *abase,
                                             uint32_t u0, uint32_t u_end, LaneAcc &m, LaneAcc &x) {
  const uint32_t ops = s.ops(), lg = s.elem_log2();
  for (uint32_t j = 0; j < kUnroll; ++j) {
    const RowUnit r = row_unit(s, dbase, u0 + j * kThreads + threadIdx.x, u_end);
    if (!r.on) continue;
    u32x4 e = u32x4{};
    if (!(ops & 2)) e = ld16<true>(sbase + (r.src << lg));
    const u32x4 g = ld16<true>(dbase + (r.dst << lg));
    uint32_t ew[4], gw[4];
    words_of(e, ew);
    words_of(g, gw);
    cmp_words(m, ew, gw, 16, lg, r.first, r.last);
    if (ops & 4) {
      const u32x4 d = ld16<true>(abase + (r.aux << lg));
      words_of(d, gw);
      cmp_words(x, ew, gw, 16, lg, r.first, r.last);
    }
    if (ops & 1) {
      const CastOf<u32x4>::type a = ld8<true>(abase + (r.aux << 1));
      uint32_t ea[2], ga[2];
      aux_words_of(CastOf<u32x4>::cast(e), ea);
      aux_words_of(a, ga);
      cmp_words(x, ea, ga, 8, 1, r.first, r.last);
    }
  }
}

// Bits of a that differ from b, folded into one word (0: the units are equal).
__device__ __forceinline__ uint32_t differ(const u32x4 &a, const u32x4 &b) {
  return (a.x ^ b.x) | (a.y ^ b.y) | (a.z ^ b.z) | (a.w ^ b.w);
}
__device__ __forceinline__ uint32_t differ(uint64_t a, uint64_t b) {
  const uint64_t d = a ^ b;
  return (uint32_t)d | (uint32_t)(d >> 32);
}
__device__ __forceinline__ uint32_t differ(uint32_t a, uint32_t b) { return a ^ b; }
__device__ __forceinline__ uint32_t differ(uint16_t a, uint16_t b) { return (uint32_t)(a ^ b); }
__device__ __forceinline__ uint32_t differ(uint8_t a, uint8_t b) { return (uint32_t)(a ^ b); }
__device__ __forceinline__ uint32_t differ(const CastOf<u32x4>::type &a, const CastOf<u32x4>::type &b) {
  return (a.x ^ b.x) | (a.y ^ b.y);
}

// The bit-level pass over units [u0, u_end) of segment s: `dm` collects the
// bits in which the destination differs from the source, `dx` those of the
// second destination (bf16 image or duplicate).  Loads, addresses and order
// are compare_chunk's; only the arithmetic is left out.
template <typename T>
__device__ __forceinline__ void differ_chunk(const DevSeg &s, const char *sbase, const char *dbase,
                                             const char *abase, uint32_t u0, uint32_t u_end, uint32_t &dm,
                                             uint32_t &dx) {
  typedef typename std::conditional<sizeof(T) == 16 || sizeof(T) == 4, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename C::type A;
  const T *src = reinterpret_cast<const T *>(sbase);
  const T *dst = reinterpret_cast<const T *>(dbase);
  const A *aux = reinterpret_cast<const A *>(abase);
  const T *dup = reinterpret_cast<const T *>(abase);
  const uint32_t ops = s.ops();
  for (uint32_t j = 0; j < kUnroll; ++j) {
    const uint32_t u = u0 + j * kThreads + threadIdx.x;
    if (u >= u_end) break;
    uint64_t so = s.src_off + u, dof = s.dst_off + u, ao = s.aux_off + u;
    if (s.rows > 1) {
      const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2()), col = u - row * s.len;
      so = s.src_off + (uint64_t)row * s.src_stride + col;
      dof = s.dst_off + (uint64_t)row * s.dst_stride + col;
      ao = s.aux_off + (uint64_t)row * s.aux_stride + col;
    }
    const T e = (ops & 2) ? T{} : ld<T, true>(src + so);
    dm |= differ(e, ld<T, true>(dst + dof));
    if (ops & 4) dx |= differ(e, ld<T, true>(dup + ao));
    if constexpr (sizeof(T) == 16 || sizeof(T) == 4) {
      if (ops & 1) dx |= differ(C::cast(e), ld<A, true>(aux + ao));
    }
  }
}

// The bit-level pass over units [u0, u0 + 64 * U) of segment s (clipped to its
// `total` units) by one wave.  Every lane issues all its units' loads, the
// second destination's (kAux: 1 a bf16 image, 2 a duplicate) among them, before
// it compares: one round trip to HBM per workgroup.
template <typename T, int U, int kAux>
__device__ __forceinline__ void differ_units(const DevSeg &s, const char *sbase, const char *dbase,
                                             const char *abase, uint32_t u0, uint32_t total, uint32_t &dm,
                                             uint32_t &dx) {
  typedef typename std::conditional<kAux == 1, CastOf<T>, CastOf<uint32_t>>::type C;
  typedef typename std::conditional<kAux == 1, typename C::type, T>::type X;
  const T *src = reinterpret_cast<const T *>(sbase);
  const T *dst = reinterpret_cast<const T *>(dbase);
  const X *aux = reinterpret_cast<const X *>(abase);
  const bool zero = (s.ops() & 2) != 0;
  T e[U], g[U];
  X x[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const uint32_t u = u0 + j * 64 + threadIdx.x;
    e[j] = T{};
    g[j] = T{};
    x[j] = X{};
    if (u < total) {
      uint64_t so = s.src_off + u, dof = s.dst_off + u, ao = s.aux_off + u;
      if (s.rows > 1) {
        const uint32_t row = magic_div(u, s.magic, s.sh1(), s.sh2()), col = u - row * s.len;
        so = s.src_off + (uint64_t)row * s.src_stride + col;
        dof = s.dst_off + (uint64_t)row * s.dst_stride + col;
        ao = s.aux_off + (uint64_t)row * s.aux_stride + col;
      }
      if (!zero) e[j] = ld<T, true>(src + so);
      g[j] = ld<T, true>(dst + dof);
      if constexpr (kAux != 0) x[j] = ld<X, true>(aux + ao);
    }
  }
  // Units past the end are zero on every side, and so is the image of zero.
#pragma unroll
  for (int j = 0; j < U; ++j) {
    dm |= differ(e[j], g[j]);
    if constexpr (kAux == 1) dx |= differ(C::cast(e[j]), x[j]);
    if constexpr (kAux == 2) dx |= differ(e[j], x[j]);
  }
}

// differ_units for the segment's second destination, if it has one.
template <typename T, int U>
__device__ __forceinline__ void dispatch_differ(const DevSeg &s, const char *sb, const char *db, const char *ab,
                                                uint32_t u0, uint32_t total, uint32_t &dm, uint32_t &dx) {
  const uint32_t ops = s.ops();
  if (ops & 4) {
    differ_units<T, U, 2>(s, sb, db, ab, u0, total, dm, dx);
    return;
  }
  if constexpr (sizeof(T) == 16 || sizeof(T) == 4) {
    if (ops & 1) {
      differ_units<T, U, 1>(s, sb, db, ab, u0, total, dm, dx);
      return;
    }
  }
  differ_units<T, U, 0>(s, sb, db, ab, u0, total, dm, dx);
}

// What a comparison's first pass finds: per device segment, bit 0 where its
// destination differs and bit 1 where its second destination does; and, if
// `any` is not null, a word of host memory set once something differs.
struct DifferMarks {
  uint32_t *flags;
  uint32_t *any;
};

// Mark a segment that differs; one lane per wave that saw a difference calls it.  Nothing is written
// where the segment is marked already, so that a destination that differs all over stays cheap.
__device__ __forceinline__ void mark_segment(const DifferMarks &m, uint32_t seg, uint32_t bits) {
  if ((__hip_atomic_load(m.flags + seg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bits) == bits) return;
  atomicOr(m.flags + seg, bits);
  if (m.any) __hip_atomic_store(m.any, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The bit-level pass over row units [u0, u0 + L * U) (clipped to u_end), every
// load of the source and the destination issued before the comparison, the second destination's after
// it.  Elements that two units hold are looked at twice.
template <int L, int U>
__device__ __forceinline__ void differ_rows(const DevSeg &s, const char *sbase, const char *dbase, const char *abase,
                                            uint32_t u0, uint32_t u_end, uint32_t &dm, uint32_t &dx) {
  const uint32_t ops = s.ops(), lg = s.elem_log2();
  u32x4 e[U], g[U];
#pragma unroll
  for (int j = 0; j < U; ++j) {
    const RowUnit r = row_unit(s, dbase, u0 + j * L + threadIdx.x, u_end);
    e[j] = g[j] = u32x4{};
    if (r.on) {
      if (!(ops & 2)) e[j] = ld16<true>(sbase + (r.src << lg));
      g[j] = ld16<true>(dbase + (r.dst << lg));
    }
  }
#pragma unroll
  for (int j = 0; j < U; ++j) {
    dm |= differ(e[j], g[j]);
    if (!(ops & 5)) continue;
    const RowUnit r = row_unit(s, dbase, u0 + j * L + threadIdx.x, u_end);
    if (!r.on) continue;
    if (ops & 4) {
      const u32x4 d = ld16<true>(abase + (r.aux << lg));
      dx |= differ(e[j], d);
    } else {
      const CastOf<u32x4>::type a = ld8<true>(abase + (r.aux << 1));
      dx |= differ(CastOf<u32x4>::cast(e[j]), a);
    }
  }
}

// First pass of a comparison on the copy kernel's schedule and with its short
// chain of scalar loads (see copy_pieces_kernel): the first workgroups read the
// tables, then one 64-lane workgroup per piece of U units a lane takes its
// segment from the plan's chunk table, dispatched in order, the XCDs in runs
// (xcd_order).  Faster than the persistent grid on
// every full-size switch (2-4%, same allocations): a segment's rows or gathered
// runs are spread over many workgroups in flight.  Bound by reading HBM.  Whole
// calls before the pre-read, the preloaded arguments, two units a lane and the
// marks in place of accumulators, and with them (one process, same
// allocations): 1 MB 52 and 31 us, 1.0 GB 194 and 174, 9.2 GB in short rows
// 1567 and 1338, 28 GB 4016 and 3975, 44 GB 6437 and 6412.
template <bool kTable, int U, typename B>
__global__ __launch_bounds__(64) void differ_piece_kernel(
    const uint32_t *__restrict__ chunk_seg, const DevSeg *__restrict__ segs, uint64_t n_chunks, uint64_t xcd_end,
    uint32_t gx, uint32_t n_warm, uint32_t xcd_log2, const uint64_t *__restrict__ src_tab, const uint64_t *__restrict__ dst_tab, B src,
    B dst, uint32_t n_segs, DifferMarks marks) {
  constexpr uint32_t kPieces = kChunkUnits / (64 * U);
  uint64_t w = (uint64_t)blockIdx.y * gx + blockIdx.x - n_warm;
  if ((int32_t)(w >> 32) < 0) {  // the sign: among the first n_warm
    warm_tables<64>(chunk_seg, segs, n_chunks, n_segs, blockIdx.x);
    return;
  }
  w = xcd_order(w, xcd_end, xcd_log2);
  const uint64_t c = w / kPieces;
  if (c >= n_chunks) return;
  const uint32_t lo = chunk_seg[c];
  const DevSeg s = load_seg(segs + lo);
  const uint32_t total = s.units();
  const uint32_t u0 = (uint32_t)(c - s.chunk_begin) * kChunkUnits + (uint32_t)(w % kPieces) * (64 * U);
  const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
  const char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
  const char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
  if (kPieces > 1 && u0 >= total) return;
  uint32_t dm = 0, dx = 0;
  switch (s.unit_log2()) {
    case kRowUnits: differ_rows<64, U>(s, sb, db, ab, u0, total, dm, dx); break;
    case 4: dispatch_differ<u32x4, U>(s, sb, db, ab, u0, total, dm, dx); break;
    case 3: dispatch_differ<uint64_t, U>(s, sb, db, ab, u0, total, dm, dx); break;
    case 2: dispatch_differ<uint32_t, U>(s, sb, db, ab, u0, total, dm, dx); break;
    case 1: dispatch_differ<uint16_t, U>(s, sb, db, ab, u0, total, dm, dx); break;
    default: dispatch_differ<uint8_t, U>(s, sb, db, ab, u0, total, dm, dx); break;
  }
  const uint32_t bits = (__any(dm != 0) ? 1u : 0u) | (__any(dx != 0) ? 2u : 0u);
  if (bits && threadIdx.x == 0) mark_segment(marks, lo, bits);
}

// First pass of a comparison when the plan has no chunk table on the device
// (it did not fit, or emrs_plan_compare_static meets a plan that has never
// run there): which segments differ at all, on compare_plan_kernel's persistent
// schedule.  Per lane only two words of differing bits are kept.  Only the
// groups of the segments it marks are compared again for compare_ckpt's figures
// (compare_plan_kernel), whose per-element fp64 work costs about 4% more time
// on Llama-2-7B than reading alone.
template <bool kTable>
__global__ __launch_bounds__(kThreads) void differ_plan_kernel(
    const DevSeg *__restrict__ segs, uint32_t n_segs, uint64_t n_chunks, uint32_t run, Bases src, Bases dst,
    const uint64_t *__restrict__ src_tab, const uint64_t *__restrict__ dst_tab, DifferMarks marks) {
  const uint64_t xcd = blockIdx.x & 7;
  const uint64_t c1 = n_chunks * (xcd + 1) / 8;
  const uint64_t step = (uint64_t)(gridDim.x >> 3) * run;
  uint32_t dm = 0, dx = 0, cur = 0;
  // Each wave marks on its own: no barrier.
  auto mark = [&](uint32_t seg) {
    const uint32_t bits = (__any(dm != 0) ? 1u : 0u) | (__any(dx != 0) ? 2u : 0u);
    if (bits && (threadIdx.x & 63) == 0) mark_segment(marks, seg, bits);
    dm = dx = 0;
  };
  for (uint64_t c = n_chunks * xcd / 8 + (uint64_t)(blockIdx.x >> 3) * run; c < c1; c += step) {
    const uint64_t c_end = min(c + run, c1);
    uint32_t lo = 0, hi = n_segs - 1;
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (segs[mid].chunk_begin <= c) lo = mid;
      else hi = mid - 1;
    }
    uint32_t si = lo;
    uint64_t s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;
    for (uint64_t q = c, nq; q < c_end; q += nq) {
      while (q >= s_end) {
        ++si;
        s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;
      }
      nq = min(min(c_end, s_end) - q, (uint64_t)kUnroll);
      const DevSeg s = segs[si];
      if (si != cur) mark(cur);
      cur = si;
      const uint32_t total = s.units();
      const uint32_t u0 = (uint32_t)(q - s.chunk_begin) * kChunkUnits;
      const uint32_t u_end = min(u0 + (uint32_t)nq * kChunkUnits, total);
      const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
      const char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
      const char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
      switch (s.unit_log2()) {
        case kRowUnits:
#pragma unroll 1
          for (uint32_t u = u0; u < u_end; u += kThreads * kRowStep)
            differ_rows<kThreads, kRowStep>(s, sb, db, ab, u, u_end, dm, dx);
          break;
        case 4: differ_chunk<u32x4>(s, sb, db, ab, u0, u_end, dm, dx); break;
        case 3: differ_chunk<uint64_t>(s, sb, db, ab, u0, u_end, dm, dx); break;
        case 2: differ_chunk<uint32_t>(s, sb, db, ab, u0, u_end, dm, dx); break;
        case 1: differ_chunk<uint16_t>(s, sb, db, ab, u0, u_end, dm, dx); break;
        default: differ_chunk<uint8_t>(s, sb, db, ab, u0, u_end, dm, dx); break;
      }
    }
  }
  mark(cur);
}

// Sum / max over the workgroup; the result is valid in thread 0.
__device__ void block_reduce(LaneAcc &a, double *lds_d, uint32_t *lds_u, float *lds_f) {
  for (int off = 32; off > 0; off >>= 1) {
    a.mismatches += __shfl_xor(a.mismatches, off, 64);
    a.nonfinite += __shfl_xor(a.nonfinite, off, 64);
    a.sq_diff += __shfl_xor(a.sq_diff, off, 64);
    a.sq_exp += __shfl_xor(a.sq_exp, off, 64);
    a.max_abs = fmaxf(a.max_abs, __shfl_xor(a.max_abs, off, 64));
    a.max_rel = fmaxf(a.max_rel, __shfl_xor(a.max_rel, off, 64));
  }
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  __syncthreads();
  if (lane == 0) {
    lds_u[2 * wave] = a.mismatches;
    lds_u[2 * wave + 1] = a.nonfinite;
    lds_d[2 * wave] = a.sq_diff;
    lds_d[2 * wave + 1] = a.sq_exp;
    lds_f[2 * wave] = a.max_abs;
    lds_f[2 * wave + 1] = a.max_rel;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kThreads / 64; ++w) {
      a.mismatches += lds_u[2 * w];
      a.nonfinite += lds_u[2 * w + 1];
      a.sq_diff += lds_d[2 * w];
      a.sq_exp += lds_d[2 * w + 1];
      a.max_abs = fmaxf(a.max_abs, lds_f[2 * w]);
      a.max_rel = fmaxf(a.max_rel, lds_f[2 * w + 1]);
    }
  }
}

__device__ void flush(const LaneAcc &a, GroupAcc *g) {
  if (a.mismatches) atomicAdd(&g->mismatches, (unsigned long long)a.mismatches);
  if (a.nonfinite) atomicAdd(&g->nonfinite, (unsigned long long)a.nonfinite);
  if (a.sq_diff != 0.0) atomicAdd(&g->sum_sq_diff, a.sq_diff);
  if (a.sq_exp != 0.0) atomicAdd(&g->sum_sq_expected, a.sq_exp);
  if (a.max_abs > 0.0f) atomicMax(&g->max_abs_bits, __float_as_uint(a.max_abs));
  if (a.max_rel > 0.0f) atomicMax(&g->max_rel_bits, __float_as_uint(a.max_rel));
}

// Add the workgroup's lane sums to their groups and clear them: the values
// compared, and with `aux` the second destination's.  Every thread calls it.
__device__ void flush_block(LaneAcc &m, LaneAcc &x, uint32_t g, uint32_t ga, bool aux, GroupAcc *acc,
                            const uint8_t *active, double *lds_d, uint32_t *lds_u, float *lds_f) {
  if (active[g]) {
    block_reduce(m, lds_d, lds_u, lds_f);
    if (threadIdx.x == 0) flush(m, acc + g);
  }
  if (aux && active[ga]) {
    block_reduce(x, lds_d, lds_u, lds_f);
    if (threadIdx.x == 0) flush(x, acc + ga);
  }
  __syncthreads();  // the LDS slots are reused by the next reduction
  m = LaneAcc();
  x = LaneAcc();
}

// Workgroups take runs of `run` consecutive chunks, each XCD sweeping its own
// eighth of the plan (workgroup b runs on XCD b % 8; the grid is a multiple of
// 8), and compare up to kUnroll chunks of one segment per step, so that every
// lane has several loads in flight.  Lane sums stay in registers while consecutive
// chunks share their (group, aux group); they are reduced over the workgroup
// only when that pair changes and at the end.  Every decision depends on the
// segment alone, so it is uniform across the workgroup, and every thread
// reaches every barrier.  Only segments with a group marked in `active` are
// compared, and only marked groups are accumulated: the second pass of a
// comparison, over the groups the first pass (differ_plan_kernel) found to differ.
template <bool kTable>
__global__ __launch_bounds__(kThreads) void compare_plan_kernel(
    const DevSeg *__restrict__ segs, const uint32_t *__restrict__ groups, const uint32_t *__restrict__ aux_groups,
    uint32_t n_segs, uint64_t n_chunks, uint32_t run, Bases src, Bases dst, const uint64_t *__restrict__ src_tab,
    const uint64_t *__restrict__ dst_tab, GroupAcc *__restrict__ acc, const uint8_t *__restrict__ active) {
  __shared__ double lds_d[2 * kThreads / 64];
  __shared__ uint32_t lds_u[2 * kThreads / 64];
  __shared__ float lds_f[2 * kThreads / 64];
  const uint64_t xcd = blockIdx.x & 7;
  const uint64_t c1 = n_chunks * (xcd + 1) / 8;
  const uint64_t step = (uint64_t)(gridDim.x >> 3) * run;
  LaneAcc m, x;
  uint32_t cur_g = 0, cur_ga = 0;
  bool open = false, cur_aux = false;
  for (uint64_t c = n_chunks * xcd / 8 + (uint64_t)(blockIdx.x >> 3) * run; c < c1; c += step) {
    const uint64_t c_end = min(c + run, c1);
    uint32_t lo = 0, hi = n_segs - 1;
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (segs[mid].chunk_begin <= c) lo = mid;
      else hi = mid - 1;
    }
    uint32_t si = lo;
    uint64_t s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;
    for (uint64_t q = c, nq; q < c_end; q += nq) {
      while (q >= s_end) {
        ++si;
        s_end = (si + 1 < n_segs) ? segs[si + 1].chunk_begin : n_chunks;
      }
      nq = min(min(c_end, s_end) - q, (uint64_t)kUnroll);  // chunks of this segment in this step
      const DevSeg s = segs[si];
      const uint32_t g = groups[si], ga = aux_groups[si];
      const bool aux = (s.ops() & 5) != 0;  // cast or duplicate
      if (!active[g] && !(aux && active[ga])) continue;  // no group of this segment differs
      if (open && (g != cur_g || aux != cur_aux || (aux && ga != cur_ga)))
        flush_block(m, x, cur_g, cur_ga, cur_aux, acc, active, lds_d, lds_u, lds_f);
      open = true;
      cur_g = g;
      cur_ga = ga;
      cur_aux = aux;
      const uint32_t total = s.units();
      const uint32_t u0 = (uint32_t)(q - s.chunk_begin) * kChunkUnits;
      const uint32_t u_end = min(u0 + (uint32_t)nq * kChunkUnits, total);
      const char *sb = base_of<kTable>(src, src_tab, s.src_buf());
      const char *db = base_of<kTable>(dst, dst_tab, s.dst_buf());
      const char *ab = base_of<kTable>(dst, dst_tab, s.aux_buf());
      switch (s.unit_log2()) {
        case kRowUnits: compare_rows(s, sb, db, ab, u0, u_end, m, x); break;
        case 4: compare_chunk<u32x4>(s, sb, db, ab, u0, u_end, m, x); break;
        case 3: compare_chunk<uint64_t>(s, sb, db, ab, u0, u_end, m, x); break;
        case 2: compare_chunk<uint32_t>(s, sb, db, ab, u0, u_end, m, x); break;
        case 1: compare_chunk<uint16_t>(s, sb, db, ab, u0, u_end, m, x); break;
        default: compare_chunk<uint8_t>(s, sb, db, ab, u0, u_end, m, x); break;
      }
    }
  }
  if (open) flush_block(m, x, cur_g, cur_ga, cur_aux, acc, active, lds_d, lds_u, lds_f);
}

// Zero n 32-bit words (accumulators are cleared by a kernel rather than a memset).
__global__ void clear_words_kernel(uint32_t *p, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

// The groups that a first pass's flags mark, into `active` (all zero before); leaves the flags zero.
__global__ void mark_groups_kernel(uint32_t *__restrict__ flags, const uint32_t *__restrict__ groups,
                                   const uint32_t *__restrict__ aux_groups, uint32_t n_segs,
                                   uint8_t *__restrict__ active) {
  for (uint64_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n_segs; k += gridDim.x * blockDim.x) {
    const uint32_t f = flags[k];
    if (!f) continue;
    if (f & 1u) active[groups[k]] = 1;
    if (f & 2u) active[aux_groups[k]] = 1;
    flags[k] = 0;
  }
}

// A grid of `n_wg` workgroups of `lanes` lanes, with fewer than 8 more per row:
// one row up to the 2^32 - 1 lanes that a dimension holds, else as many equal
// rows as that takes, each a multiple of 8 workgroups long so that a
// workgroup's XCD follows from its number.  Rows of 65536 workgroups were used
// before: the last one, half empty on average, still cost its launch, 0.4 ns a
// workgroup (a 383 MB switch 65.9 us, of which 14 us for the 36,000 empty
// workgroups of its last row).  False when 65535 rows do not hold them.
bool tight_grid(uint64_t n_wg, uint32_t lanes, dim3 *grid) {
  const uint64_t max_x = 0xffffffffull / lanes / 8 * 8;
  const uint64_t rows = std::max<uint64_t>(1, (n_wg + max_x - 1) / max_x);
  if (rows > kMaxGridY) return false;
  const uint64_t gx = rows == 1 ? n_wg : std::min(max_x, ((n_wg + rows - 1) / rows + 7) / 8 * 8);
  *grid = dim3((uint32_t)gx, (uint32_t)((n_wg + gx - 1) / gx));
  return true;
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Workgroups that read a plan's tables ahead of the pieces, a multiple of 8 so that the pieces keep their XCDs.
uint32_t warm_groups(uint64_t n_chunks, uint64_t n_segs, uint32_t lanes) {
  const uint64_t units = n_chunks / 4 + n_segs * (sizeof(DevSeg) / sizeof(u32x4));
  const uint64_t n = ((units + kWarmUnits * lanes - 1) / (kWarmUnits * lanes) + 7) / 8 * 8;
  return n > 0xffffffffull ? 0 : (uint32_t)n;
}

// What both comparison entry points prepare on the host: checked bases and the
// element counts per group.
struct CompareJob {
  ResolvedBases rb;
  const uint32_t *groups = nullptr, *aux_groups = nullptr;  // the caller's, one per input segment, or null
  int cus = 0;
  const uint32_t *cseg = nullptr;  // the plan's chunk table on this device, if there is one

  // Group of device segment k's destination, and of its second destination.
  uint32_t group(const emrs_plan *plan, size_t k) const { return groups ? groups[plan->origin[k]] : 0; }
  uint32_t aux_group(const emrs_plan *plan, size_t k) const {
    return aux_groups ? aux_groups[plan->origin[k]] : group(plan, k);
  }
  // Per device segment its group, then its aux group.
  std::vector<uint32_t> group_table(const emrs_plan *plan) const {
    const size_t nd = plan->segs.size();
    std::vector<uint32_t> t(2 * nd);
    for (size_t k = 0; k < nd; ++k) t[k] = group(plan, k), t[nd + k] = aux_group(plan, k);
    return t;
  }
  // The groups that the first pass's flags mark; false when there is none.
  bool marked_groups(const emrs_plan *plan, const std::vector<uint32_t> &flags, std::vector<uint8_t> *mark) const {
    bool any = false;
    for (size_t k = 0; k < flags.size(); ++k) {
      if (flags[k] & 1u) (*mark)[group(plan, k)] = 1;
      if (flags[k] & 2u) (*mark)[aux_group(plan, k)] = 1;
      any = any || flags[k];
    }
    return any;
  }
};

int compare_setup(emrs_plan *plan, void *const *src_bases, void *const *dst_bases, const uint32_t *groups,
                  const uint32_t *aux_groups, uint32_t n_groups, emrs_compare_stats *stats, CompareJob *job) {
  if (!plan || !stats) return fail(EMRS_ERR_INVALID_ARGUMENT, "NULL argument");
  if (n_groups == 0) return fail(EMRS_ERR_INVALID_ARGUMENT, "n_groups must be >= 1");
  const uint64_t n_in = plan->stats.n_segments;
  for (uint64_t i = 0; i < n_in; ++i)
    if ((groups && groups[i] >= n_groups) || (aux_groups && aux_groups[i] >= n_groups))
      return fail(EMRS_ERR_INVALID_ARGUMENT, "group id >= n_groups");
  int rc = resolve_bases(plan, src_bases, dst_bases, &job->rb, /*out_of_place=*/false);
  if (rc) return rc;
  job->groups = groups;
  job->aux_groups = aux_groups;
  std::vector<uint64_t> elements(n_groups, 0);
  for (size_t k = 0; k < plan->segs.size(); ++k) {
    const DevSeg &d = plan->segs[k];
    const uint64_t n = ((uint64_t)d.len * d.rows) << (d.off_log2() - d.elem_log2());
    elements[job->group(plan, k)] += n;
    if (d.ops() & 5) elements[job->aux_group(plan, k)] += n;
  }
  for (uint32_t g = 0; g < n_groups; ++g) {
    stats[g] = emrs_compare_stats{};
    stats[g].elements = elements[g];
  }
  return EMRS_OK;
}

// The current device and its CU count.
int compare_device(CompareJob *job, int *dev) {
  int resident_nt = 0, resident_t = 0;
  return current_device(dev, &job->cus, &resident_nt, &resident_t);
}

// Workgroups per CU that a persistent comparison kernel can hold.
template <typename K>
int resident_of(K kernel) {
  int v = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, kernel, kThreads, 0) != hipSuccess || v <= 0) {
    (void)hipGetLastError();
    v = 4;
  }
  return v;
}

// A persistent grid of resident workgroups, a multiple of 8 (one eighth of
// the plan per XCD), in runs of up to 32 steps: at most a quarter of each
// workgroup's share, so that small plans still spread out.
void persistent_grid(const emrs_plan *plan, const CompareJob &job, int per_cu, dim3 *grid, uint32_t *run) {
  uint64_t blocks = std::min<uint64_t>(plan->n_chunks, (uint64_t)job.cus * per_cu);
  blocks = std::max<uint64_t>(8, blocks / 8 * 8);
  *run = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(32 * kUnroll, plan->n_chunks / (blocks * 4)));
  *grid = dim3((uint32_t)blocks);
}

// First pass: marks what differs.  differ_piece_kernel with the plan's chunk table, else differ_plan_kernel.
hipError_t differ_launch(const emrs_plan *plan, const CompareJob &job, const DevSeg *table, const uint64_t *tab,
                         const DifferMarks &marks, hipStream_t st) {
  const uint32_t nd = (uint32_t)plan->segs.size();
  const uint64_t *dtab = tab ? tab + plan->stats.n_src_bufs : nullptr;
  if (job.cseg) {
    constexpr int U = kDifferUnits;
    const uint64_t n_pieces = plan->n_chunks * (kChunkUnits / (64 * U));
    const uint32_t n_warm = g_tuning.warm_tables.load() ? warm_groups(plan->n_chunks, nd, 64) : 0;
    dim3 grid;
    if (!tight_grid(n_warm + n_pieces, 64, &grid)) return hipErrorInvalidConfiguration;
    const XcdRuns xcd = xcd_runs(g_tuning.xcd_remap.load(), plan->n_chunks, kChunkUnits / (64 * U));
    FewBases src{}, dst{};
    if (!job.rb.table)
      for (uint32_t i = 0; i < kFewBuffers; ++i) src.p[i] = job.rb.src.p[i], dst.p[i] = job.rb.dst.p[i];
    if (job.rb.table)
      hipLaunchKernelGGL((differ_piece_kernel<true, U, FewBases>), grid, dim3(64), 0, st, job.cseg, table,
                         plan->n_chunks, xcd.end, grid.x, n_warm, xcd.log2, tab, dtab, src, dst, nd, marks);
    else if (std::max(plan->stats.n_src_bufs, plan->stats.n_dst_bufs) <= kFewBuffers)
      hipLaunchKernelGGL((differ_piece_kernel<false, U, FewBases>), grid, dim3(64), 0, st, job.cseg, table,
                         plan->n_chunks, xcd.end, grid.x, n_warm, xcd.log2, tab, dtab, src, dst, nd, marks);
    else
      hipLaunchKernelGGL((differ_piece_kernel<false, U, Bases>), grid, dim3(64), 0, st, job.cseg, table,
                         plan->n_chunks, xcd.end, grid.x, n_warm, xcd.log2, tab, dtab, job.rb.src, job.rb.dst, nd, marks);
    return hipGetLastError();
  }
  // It could hold 8 workgroups per CU; 3-6 read at the plain read rate and 8 is up to
  // 7% slower (Llama-2-7B, Mixtral and Group-ZeRO switches, same allocations): 4.
  dim3 grid;
  uint32_t run = 0;
  persistent_grid(plan, job, std::min(resident_of(differ_plan_kernel<false>), kDifferBlocksPerCu), &grid, &run);
  if (job.rb.table)
    hipLaunchKernelGGL(differ_plan_kernel<true>, grid, dim3(kThreads), 0, st, table, nd, plan->n_chunks, run,
                       job.rb.src, job.rb.dst, tab, dtab, marks);
  else
    hipLaunchKernelGGL(differ_plan_kernel<false>, grid, dim3(kThreads), 0, st, table, nd, plan->n_chunks, run,
                       job.rb.src, job.rb.dst, tab, dtab, marks);
  return hipGetLastError();
}

// Zero 32-bit words with a kernel (no memset node if the stream's work is ever captured).
hipError_t clear_words(void *p, uint64_t words, hipStream_t st) {
  hipLaunchKernelGGL(clear_words_kernel, dim3((uint32_t)std::min<uint64_t>(1024, (words + 255) / 256)), dim3(256), 0,
                     st, static_cast<uint32_t *>(p), words);
  return hipGetLastError();
}

// Second pass of a comparison, when the first has marked segments: every figure
// of their groups, on device buffers the caller provides (acc: n_groups
// accumulators; grp: two group ids per device segment; active: n_groups bytes,
// in whole words), leaving the accumulators in `host`.  The groups are those of
// `mark` or, where it is null, those that `flags` mark on the device, which are
// zero afterwards: read back to the host, they cost a comparison that finds
// something one more wait (4 KB 57 us, and 76 with the wait; 240 MB in 60,000
// segments 489 and 553).  Waits for the stream: `mark` and the group table are read by the copies.
hipError_t compare_marked(const emrs_plan *plan, const CompareJob &job, const DevSeg *table, uint32_t *grp,
                          const uint64_t *tab, GroupAcc *acc, uint8_t *active, const std::vector<uint8_t> *mark,
                          uint32_t *flags, hipStream_t st, std::vector<GroupAcc> &host) {
  const uint32_t nd = (uint32_t)plan->segs.size();
  const uint64_t *dtab = tab ? tab + plan->stats.n_src_bufs : nullptr;
  const std::vector<uint32_t> gt = job.group_table(plan);
  dim3 grid;
  uint32_t run = 0;
  persistent_grid(plan, job, resident_of(compare_plan_kernel<false>), &grid, &run);
  hipError_t e = hipMemcpyAsync(grp, gt.data(), gt.size() * sizeof(uint32_t), hipMemcpyHostToDevice, st);
  if (mark) {
    if (e == hipSuccess) e = hipMemcpyAsync(active, mark->data(), mark->size(), hipMemcpyHostToDevice, st);
  } else {
    if (e == hipSuccess) e = clear_words(active, (host.size() + 3) / 4, st);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(mark_groups_kernel, dim3(std::min<uint32_t>(1024, (nd + 255) / 256)), dim3(256), 0, st, flags,
                         grp, grp + nd, nd, active);
      e = hipGetLastError();
    }
  }
  if (e == hipSuccess) e = clear_words(acc, host.size() * sizeof(GroupAcc) / sizeof(uint32_t), st);
  if (e == hipSuccess) {
    if (job.rb.table)
      hipLaunchKernelGGL(compare_plan_kernel<true>, grid, dim3(kThreads), 0, st, table, grp, grp + nd, nd,
                         plan->n_chunks, run, job.rb.src, job.rb.dst, tab, dtab, acc, active);
    else
      hipLaunchKernelGGL(compare_plan_kernel<false>, grid, dim3(kThreads), 0, st, table, grp, grp + nd, nd,
                         plan->n_chunks, run, job.rb.src, job.rb.dst, tab, dtab, acc, active);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(host.data(), acc, host.size() * sizeof(GroupAcc), hipMemcpyDeviceToHost, st);
  const hipError_t se = hipStreamSynchronize(st);
  return e == hipSuccess ? se : e;
}

// Words of pinned host memory that comparisons in flight are told a difference
// through: one page for the process, one 64-byte slot per comparison.  Null
// when all are in use or the page could not be made: the comparison then
// reads its flags back.
struct AnySlots {
  static constexpr int kSlots = 64;
  std::mutex mu;
  uint32_t *page = nullptr;
  bool tried = false;
  uint64_t used = 0;
};
AnySlots g_any;

uint32_t *take_any_slot() {
  std::lock_guard<std::mutex> lk(g_any.mu);
  if (!g_any.tried) {
    g_any.tried = true;
    void *p = nullptr;
    if (hipHostMalloc(&p, AnySlots::kSlots * 64,
                      hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess)
      g_any.page = static_cast<uint32_t *>(p);
    else
      (void)hipGetLastError();
  }
  if (!g_any.page) return nullptr;
  for (int i = 0; i < AnySlots::kSlots; ++i)
    if (!((g_any.used >> i) & 1u)) {
      g_any.used |= 1ull << i;
      return g_any.page + i * 16;
    }
  return nullptr;
}

void give_any_slot(uint32_t *slot) {
  if (!slot) return;
  std::lock_guard<std::mutex> lk(g_any.mu);
  g_any.used &= ~(1ull << ((slot - g_any.page) / 16));
}

// The plan's flags on device `dev`, all zero: one array is kept between
// comparisons (a comparison has waited for its stream when it gives the array
// back, and has cleared what it marked), and concurrent ones get arrays of
// their own.
int take_flags(emrs_plan *plan, int dev, hipStream_t st, uint32_t **out) {
  {
    std::lock_guard<std::mutex> lk(plan->mu);
    if ((int)plan->differ_flags.size() <= dev) plan->differ_flags.resize(dev + 1, nullptr);
    *out = plan->differ_flags[dev];
    plan->differ_flags[dev] = nullptr;
  }
  if (*out) return EMRS_OK;
  const uint64_t nd = plan->segs.size();
  hipError_t e = table_alloc(reinterpret_cast<void **>(out), nd * sizeof(uint32_t), st);
  if (e != hipSuccess) return hip_fail(e, "hipMallocAsync(compare flags)");
  e = clear_words(*out, nd, st);
  if (e == hipSuccess) return EMRS_OK;
  (void)hipFreeAsync(*out, st);
  *out = nullptr;
  return hip_fail(e, "clearing the compare flags");
}

// `clean`: the array is all zero again and no launch uses it.
void give_flags(emrs_plan *plan, int dev, hipStream_t st, uint32_t *flags, bool clean) {
  if (clean) {
    std::lock_guard<std::mutex> lk(plan->mu);
    if (!plan->differ_flags[dev]) {
      plan->differ_flags[dev] = flags;
      return;
    }
  }
  (void)hipFreeAsync(flags, st);
}

void compare_finish(const std::vector<GroupAcc> &host, emrs_compare_stats *stats) {
  for (size_t g = 0; g < host.size(); ++g) {
    stats[g].mismatches = host[g].mismatches;
    stats[g].nonfinite = host[g].nonfinite;
    stats[g].sum_sq_diff = host[g].sum_sq_diff;
    stats[g].sum_sq_expected = host[g].sum_sq_expected;
    uint32_t ma = host[g].max_abs_bits, mr = host[g].max_rel_bits;
    memcpy(&stats[g].max_abs_diff, &ma, 4);
    memcpy(&stats[g].max_rel_diff, &mr, 4);
  }
}

// Per device: the address of `scratch` (the array's host-side name is not a
// device address), looked up once with that device current, and the mutex
// that serialises the calls sharing it.
std::mutex g_scratch_mu;
std::vector<unsigned char *> g_scratch_ptr;
std::vector<std::unique_ptr<std::mutex>> g_scratch_call_mu;

int scratch_of(int dev, unsigned char **out) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize(dev + 1, nullptr);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(EMRS_ERR_HIP, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_ptr[dev] = static_cast<unsigned char *>(p);
  }
  *out = g_scratch_ptr[dev];
  return EMRS_OK;
}

std::mutex *scratch_call_mutex(int dev) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  while ((int)g_scratch_call_mu.size() <= dev) g_scratch_call_mu.emplace_back(new std::mutex);
  return g_scratch_call_mu[dev].get();
}

}  // namespace

extern "C" {

const char *emrs_last_error(void) { return g_last_error.c_str(); }

int emrs_abi_version(void) { return EMRS_ABI_VERSION; }

int emrs_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

int emrs_plan_create(const emrs_segment *segs, uint64_t n_segs, const uint64_t *src_buf_bytes,
                     uint32_t n_src_bufs, const uint64_t *dst_buf_bytes, uint32_t n_dst_bufs,
                     uint32_t flags, emrs_plan **out_plan) {
  g_last_error.clear();
  if (!out_plan) return fail(EMRS_ERR_INVALID_ARGUMENT, "out_plan is NULL");
  *out_plan = nullptr;
  if (n_segs && !segs) return fail(EMRS_ERR_INVALID_ARGUMENT, "segs is NULL");
  if (n_src_bufs > EMRS_MAX_BUFFERS || n_dst_bufs > EMRS_MAX_BUFFERS)
    return fail(EMRS_ERR_TOO_MANY_BUFFERS, "more than EMRS_MAX_BUFFERS buffers on one side");
  if ((n_src_bufs && !src_buf_bytes) || (n_dst_bufs && !dst_buf_bytes))
    return fail(EMRS_ERR_INVALID_ARGUMENT, "buffer size array is NULL");
  if (flags & ~EMRS_PLAN_CHECK_DISJOINT) return fail(EMRS_ERR_INVALID_ARGUMENT, "unknown flags");
  if (n_segs > 0xffffffffull) return fail(EMRS_ERR_INVALID_ARGUMENT, "more than 2^32 - 1 segments");

  Builder bld;
  bld.out.reserve(n_segs);
  uint64_t payload = 0, read = 0;
  std::vector<uint8_t> src_used(n_src_bufs, 0), dst_used(n_dst_bufs, 0);
  for (uint64_t i = 0; i < n_segs; ++i) {
    const emrs_segment &s = segs[i];
    char where[64];
    snprintf(where, sizeof where, "segment %llu: ", (unsigned long long)i);
    const std::string at(where);
    const int lg = log2_of(s.elem_bytes);
    const bool cast = (s.flags & EMRS_SEG_CAST_BF16) != 0;
    const bool zero = (s.flags & EMRS_SEG_ZERO_FILL) != 0;
    const bool dup = (s.flags & EMRS_SEG_DUP) != 0;
    const bool has_aux = cast || dup;
    if (lg < 0) return fail(EMRS_ERR_INVALID_ARGUMENT, at + "elem_bytes must be 1, 2, 4 or 8");
    if ((s.flags & ~(EMRS_SEG_CAST_BF16 | EMRS_SEG_ZERO_FILL | EMRS_SEG_DUP)) || s.reserved)
      return fail(EMRS_ERR_INVALID_ARGUMENT, at + "unknown flags");
    if (cast && dup) return fail(EMRS_ERR_INVALID_ARGUMENT, at + "a segment carries a bf16 image or a duplicate, not both");
    if (cast && s.elem_bytes != 4) return fail(EMRS_ERR_INVALID_ARGUMENT, at + "a bf16 cast needs fp32 elements");
    if (s.src_buf >= n_src_bufs || s.dst_buf >= n_dst_bufs || (has_aux && s.aux_buf >= n_dst_bufs))
      return fail(EMRS_ERR_INVALID_ARGUMENT, at + "buffer id out of range");
    if (s.rows == 0) return fail(EMRS_ERR_INVALID_ARGUMENT, at + "rows must be >= 1");
    if (s.len == 0) continue;
    if (s.rows > 1 && (s.dst_stride < s.len || (has_aux && s.aux_stride < s.len)))
      return fail(EMRS_ERR_INVALID_ARGUMENT, at + "a destination stride < len makes rows overlap");
    if (!zero && extent_end(s.src_off, s.len, s.rows, s.rows > 1 ? s.src_stride : 0, s.elem_bytes) >
                     src_buf_bytes[s.src_buf])
      return fail(EMRS_ERR_OUT_OF_BOUNDS, at + "source range exceeds its buffer");
    if (extent_end(s.dst_off, s.len, s.rows, s.rows > 1 ? s.dst_stride : 0, s.elem_bytes) > dst_buf_bytes[s.dst_buf])
      return fail(EMRS_ERR_OUT_OF_BOUNDS, at + "destination range exceeds its buffer");
    // Bytes per aux element: a bf16 image, or a duplicate of the element.
    const uint64_t aeb = cast ? 2 : (dup ? s.elem_bytes : 0);
    if (has_aux && extent_end(s.aux_off, s.len, s.rows, s.rows > 1 ? s.aux_stride : 0, (uint32_t)aeb) >
                       dst_buf_bytes[s.aux_buf])
      return fail(EMRS_ERR_OUT_OF_BOUNDS, at + (cast ? "bf16 range exceeds its buffer" : "duplicate range exceeds its buffer"));
    if (!zero) read += s.len * s.rows * s.elem_bytes;
    payload += s.len * s.rows * (s.elem_bytes + aeb);
    if (!zero) src_used[s.src_buf] = 1;
    dst_used[s.dst_buf] = 1;
    if (has_aux) dst_used[s.aux_buf] = 1;

    const uint64_t eb = s.elem_bytes;
    bld.cur_origin = (uint32_t)i;
    bld.cur_elem_log2 = (uint8_t)lg;
    // A zero fill has no source: align its phantom source with the destination.
    const uint64_t so = zero ? s.dst_off * eb : s.src_off * eb, dof = s.dst_off * eb, lb = s.len * eb;
    const uint64_t ds = s.rows > 1 ? s.dst_stride * eb : 0, ss = zero ? ds : (s.rows > 1 ? s.src_stride * eb : 0);
    const uint64_t ao = s.aux_off * aeb, as = s.rows > 1 ? s.aux_stride * aeb : 0;
    Aux ax;
    ax.on = has_aux;
    ax.cast = cast;
    ax.dup = dup;
    ax.zero = zero;
    ax.buf = s.aux_buf;
    // Aux bytes per 16-byte unit: 8 for a bf16 image of fp32, 16 for a duplicate.
    const uint64_t avu = has_aux ? 16 * aeb / eb : 16;
    const bool aux_vec_ok = !has_aux || (ao % avu == 0 && as % avu == 0);
    const bool rows1 = s.rows == 1 || (ss == lb && ds == lb && (!has_aux || as == s.len * aeb));
    const uint64_t L = lb * s.rows;
    // One run of L bytes, or rows of lb bytes.
    const uint64_t run = rows1 ? L : lb;
    const bool all16 = so % 16 == 0 && dof % 16 == 0 && run % 16 == 0 && (rows1 || (ss % 16 == 0 && ds % 16 == 0)) &&
                       aux_vec_ok;
    // Source, destination and aux reach a 16-byte boundary at the same element.
    const bool together = rows1 && so % 16 == dof % 16 && (!has_aux || (ao % avu) * eb / aeb == so % 16);
    const uint64_t head = std::min<uint64_t>((16 - so % 16) % 16, run);
    bld.vec_bytes += all16 ? L : (together ? (L - head) / 16 * 16 : 0);
    bld.scalar_bytes += all16 ? 0 : (together ? L - (L - head) / 16 * 16 : L);
    // Row units (see kRowUnits) wherever 16-byte units do not fit.  Where they
    // do fit they stay, on lines or not: row units for segments off the lines
    // gained 0-1% on switches of 9 GB and more, but cost 2% and 5% on ones of 0.9
    // and 4 GB.  Byte elements stay on the element path: no tensor of a training
    // state has them.
    const bool by_rows = lg > 0 && !all16 && run >= 16;
    const uint32_t ul = by_rows ? (uint32_t)lg : (all16 ? 4u : (uint32_t)lg);
    const uint64_t ub = 1ull << ul, aub = has_aux ? ub * aeb / eb : 1;  // bytes per unit, and per aux unit
    if (has_aux) ax.off = ao / aub;
    if (rows1 && !by_rows && !all16 && together) {  // byte elements: a vector body between two ends
      const uint64_t body = (L - head) / 16 * 16, tail = L - head - body;
      const uint64_t aux_head = head * aeb / eb, aux_body = body * aeb / eb;
      bld.emit(s.src_buf, s.dst_buf, lg, so / eb, dof / eb, head / eb, 1, 0, 0, ax);
      ax.off = has_aux ? (ao + aux_head) / avu : 0;
      bld.emit(s.src_buf, s.dst_buf, 4, (so + head) / 16, (dof + head) / 16, body / 16, 1, 0, 0, ax);
      ax.off = has_aux ? (ao + aux_head + aux_body) / aeb : 0;
      bld.emit(s.src_buf, s.dst_buf, lg, (so + head + body) / eb, (dof + head + body) / eb, tail / eb, 1, 0, 0, ax);
    } else if (rows1) {
      bld.emit(s.src_buf, s.dst_buf, ul, so / ub, dof / ub, L / ub, 1, 0, 0, ax, by_rows);
    } else {
      ax.stride = has_aux ? as / aub : 0;
      bld.emit(s.src_buf, s.dst_buf, ul, so / ub, dof / ub, lb / ub, s.rows, ss / ub, ds / ub, ax, by_rows);
    }
  }
  if (flags & EMRS_PLAN_CHECK_DISJOINT) {
    int rc = check_disjoint(segs, n_segs);
    if (rc) return rc;
  }

  if (bld.out.size() > 0xffffffffull) return fail(EMRS_ERR_INVALID_ARGUMENT, "plan needs more than 2^32 - 1 device segments");
  emrs_plan *p = new (std::nothrow) emrs_plan;
  if (!p) return fail(EMRS_ERR_INVALID_ARGUMENT, "out of host memory");
  p->segs = std::move(bld.out);
  p->origin = std::move(bld.origin);
  p->n_chunks = bld.chunks;
  make_hint(p->segs, p->n_chunks, &p->hint);
  p->src_bytes.assign(src_buf_bytes, src_buf_bytes + n_src_bufs);
  p->dst_bytes.assign(dst_buf_bytes, dst_buf_bytes + n_dst_bufs);
  p->src_used = std::move(src_used);
  p->dst_used = std::move(dst_used);
  p->stats.n_segments = n_segs;
  p->stats.n_device_segments = p->segs.size();
  p->stats.payload_bytes = payload;
  p->stats.read_bytes = read;
  p->stats.vector_bytes = bld.vec_bytes;
  p->stats.scalar_bytes = bld.scalar_bytes;
  p->stats.n_chunks = bld.chunks;
  p->stats.n_src_bufs = n_src_bufs;
  p->stats.n_dst_bufs = n_dst_bufs;
  *out_plan = p;
  return EMRS_OK;
}

}  // extern "C"

namespace {
// One launch of the copy over every piece of a plan.
struct CopyLaunch {
  const ResolvedBases *rb;
  const uint64_t *stab, *dtab;  // device pointer tables when rb->table
  const DevSeg *table;
  uint32_t n_segs, n_bufs;      // n_bufs: buffers on the larger side whose bases rb holds
  uint64_t n_chunks;
  const SegHint *hint;
  const uint32_t *cseg;         // the chunk table, or nullptr: the kernel searches
  bool nt, warm;
  hipStream_t st;
};

template <bool kNT, bool kTable, int L, int U, bool kBuf>
void launch_kernel(const CopyLaunch &c, dim3 grid, const XcdRuns &xcd, uint32_t n_warm) {
  if constexpr (!kBuf) {
    if (c.cseg) {
      if (c.n_bufs <= kFewBuffers || kTable) {
        FewBases src{}, dst{};
        for (uint32_t i = 0; i < kFewBuffers && !kTable; ++i) src.p[i] = c.rb->src.p[i], dst.p[i] = c.rb->dst.p[i];
        hipLaunchKernelGGL((copy_pieces_kernel<kNT, kTable, L, U, FewBases>), grid, dim3(L), 0, c.st, c.cseg, c.table,
                           c.n_chunks, xcd.end, grid.x, n_warm, xcd.log2, c.stab, c.dtab, src, dst, c.n_segs);
      } else if constexpr (!kTable) {
        hipLaunchKernelGGL((copy_pieces_kernel<kNT, false, L, U, Bases>), grid, dim3(L), 0, c.st, c.cseg, c.table,
                           c.n_chunks, xcd.end, grid.x, n_warm, xcd.log2, c.stab, c.dtab, c.rb->src, c.rb->dst, c.n_segs);
      }
      return;
    }
  }
  hipLaunchKernelGGL((copy_plan_kernel<kNT, kTable, L, U, kBuf>), grid, dim3(L), 0, c.st, c.table, c.n_chunks, *c.hint,
                     c.rb->src, c.rb->dst, c.stab, c.dtab, xcd.end, xcd.log2, c.cseg, n_warm, c.n_segs);
}

template <int L, int U, bool kBuf>
int launch_chunks(const CopyLaunch &c) {
  const uint64_t n_pieces = c.n_chunks * (kChunkUnits / (L * U));
  const XcdRuns xcd = xcd_runs(g_tuning.xcd_remap.load(), c.n_chunks, kChunkUnits / (L * U));
  const uint64_t n_warm = c.cseg && c.warm ? warm_groups(c.n_chunks, c.n_segs, L) : 0;
  dim3 grid;
  if (!tight_grid(n_warm + n_pieces, L, &grid))
    return fail(EMRS_ERR_INVALID_ARGUMENT, "plan has too many chunks for one launch");
  if (c.nt && c.rb->table) launch_kernel<true, true, L, U, kBuf>(c, grid, xcd, (uint32_t)n_warm);
  else if (c.nt) launch_kernel<true, false, L, U, kBuf>(c, grid, xcd, (uint32_t)n_warm);
  else if (c.rb->table) launch_kernel<false, true, L, U, kBuf>(c, grid, xcd, (uint32_t)n_warm);
  else launch_kernel<false, false, L, U, kBuf>(c, grid, xcd, (uint32_t)n_warm);
  return EMRS_OK;
}

// The one-workgroup-per-piece launch for `lanes` lanes of `units` units each.
template <bool kBuf>
int launch_pieces(uint32_t lanes, uint32_t units, const CopyLaunch &c) {
  switch (lanes * 8 + units) {
    case 64 * 8 + 1: return launch_chunks<64, 1, kBuf>(c);
    case 64 * 8 + 2: return launch_chunks<64, 2, kBuf>(c);
    case 128 * 8 + 1: return launch_chunks<128, 1, kBuf>(c);
    case 128 * 8 + 2: return launch_chunks<128, 2, kBuf>(c);
    case 256 * 8 + 1: return launch_chunks<256, 1, kBuf>(c);
    default: return launch_chunks<64, 4, kBuf>(c);
  }
}
}  // namespace

extern "C" {

int emrs_plan_stats_get(const emrs_plan *plan, emrs_plan_stats *out) {
  if (!plan || !out) return fail(EMRS_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = plan->stats;
  return EMRS_OK;
}

int emrs_plan_prepare(emrs_plan *plan, void *stream) {
  g_last_error.clear();
  if (!plan) return fail(EMRS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (plan->n_chunks == 0) return EMRS_OK;
  int dev = 0, cus = 0, resident_nt = 0, resident_t = 0;
  int rc = current_device(&dev, &cus, &resident_nt, &resident_t);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if ((rc = refuse_capture(st, "emrs_plan_prepare"))) return rc;
  DevSeg *table = nullptr;
  rc = device_table(plan, dev, st, &table);
  if (rc) return rc;
  if (g_tuning.chunk_index.load() && !g_tuning.persistent.load()) {
    uint32_t *cseg = nullptr;
    rc = chunk_table(plan, dev, st, table, &cseg);
  }
  return rc;
}

int emrs_plan_execute(emrs_plan *plan, void *const *src_bases, void *const *dst_bases,
                      void *stream) {
  g_last_error.clear();
  if (!plan) return fail(EMRS_ERR_INVALID_ARGUMENT, "plan is NULL");
  ResolvedBases rb;
  int rc = resolve_bases(plan, src_bases, dst_bases, &rb);
  if (rc) return rc;
  if (plan->n_chunks == 0) return EMRS_OK;

  int dev = 0, cus = 0, resident_nt = 0, resident_t = 0;
  rc = current_device(&dev, &cus, &resident_nt, &resident_t);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  DevSeg *table = nullptr;
  rc = device_table(plan, dev, st, &table);
  if (rc) return rc;

  const bool nt = g_tuning.nontemporal.load() != 0;
  const uint32_t nseg = (uint32_t)plan->segs.size();
  const dim3 block(kThreads);
  if (!g_tuning.persistent.load()) {
    // One workgroup per piece of lanes * units units.
    const uint32_t lanes = g_tuning.lanes.load(), units = g_tuning.units.load();
    uint64_t *tab = nullptr;
    bool tab_owned = false;
    rc = pointer_table(plan, dev, rb, st, &tab, &tab_owned);
    if (rc) return rc;
    const uint64_t *stab = tab, *dtab = tab ? tab + plan->stats.n_src_bufs : nullptr;
    // The bases of the cached pointer table also have a resolved segment
    // table: no per-workgroup base lookup.
    const ResolvedBases *lb = &rb;
    ResolvedBases flat;
    uint32_t n_bufs = std::max(plan->stats.n_src_bufs, plan->stats.n_dst_bufs);
    if (rb.table && !tab_owned) {
      DevSeg *abs = nullptr;
      char *common = nullptr;
      rc = resolved_table(plan, dev, rb, st, &abs, &common);
      if (rc) return rc;
      if (abs) {
        table = abs;
        flat.src.p[0] = flat.dst.p[0] = common;
        lb = &flat;
        n_bufs = 1;
        stab = dtab = nullptr;
      }
    }
    uint32_t *cseg = nullptr;
    if (g_tuning.chunk_index.load()) {
      rc = chunk_table(plan, dev, st, table, &cseg);
      if (rc) {
        if (tab_owned) (void)hipFreeAsync(tab, st);
        return rc;
      }
    }
    const CopyLaunch launch{lb, stab, dtab, table, nseg, n_bufs, plan->n_chunks, &plan->hint,
                            cseg, nt, g_tuning.warm_tables.load() != 0, st};
    rc = g_tuning.buffer_ops.load() ? launch_pieces<true>(lanes, units, launch) : launch_pieces<false>(lanes, units, launch);
    if (rc) {
      if (tab_owned) (void)hipFreeAsync(tab, st);
      return rc;
    }
    hipError_t le = hipGetLastError();
    if (tab_owned) (void)hipFreeAsync(tab, st);
    if (le != hipSuccess) return hip_fail(le, "copy_plan_kernel launch");
    return note_launch(plan, dev, st);
  }

  // Persistent grid.  A run of N counts N steps of kUnroll chunks.
  const uint32_t bpc = g_tuning.blocks_per_cu.load();
  const uint64_t max_blocks = (uint64_t)cus * (bpc ? bpc : (uint32_t)(nt ? resident_nt : resident_t));
  uint64_t blocks = std::min<uint64_t>(plan->n_chunks, max_blocks);
  uint32_t run = g_tuning.run.load() * kUnroll;
  const bool remap = g_tuning.xcd_remap.load() != 0;
  if (run) {
    // Round-robin runs: at most a quarter of each workgroup's share, so that
    // small plans still spread over the whole grid.
    run = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(run, plan->n_chunks / (blocks * 4)));
    blocks = std::min<uint64_t>(blocks, (plan->n_chunks + run - 1) / run);
  }
  if (remap) blocks = (blocks + 7) / 8 * 8;
  const uint64_t cpb = (plan->n_chunks + blocks - 1) / blocks;
  if (!remap && !run) blocks = (plan->n_chunks + cpb - 1) / cpb;
  const uint32_t xcd_stride = remap ? (uint32_t)(blocks / 8) : 0;
  uint64_t *tab = nullptr;
  bool tab_owned = false;
  rc = pointer_table(plan, dev, rb, st, &tab, &tab_owned);
  if (rc) return rc;
  const uint64_t *stab = tab, *dtab = tab ? tab + plan->stats.n_src_bufs : nullptr;
  const dim3 grid((uint32_t)blocks);
  if (nt && rb.table)
    hipLaunchKernelGGL((copy_plan_persistent_kernel<true, true>), grid, block, 0, st, table, nseg, plan->n_chunks,
                       cpb, xcd_stride, run, rb.src, rb.dst, stab, dtab);
  else if (nt)
    hipLaunchKernelGGL((copy_plan_persistent_kernel<true, false>), grid, block, 0, st, table, nseg, plan->n_chunks,
                       cpb, xcd_stride, run, rb.src, rb.dst, stab, dtab);
  else if (rb.table)
    hipLaunchKernelGGL((copy_plan_persistent_kernel<false, true>), grid, block, 0, st, table, nseg, plan->n_chunks,
                       cpb, xcd_stride, run, rb.src, rb.dst, stab, dtab);
  else
    hipLaunchKernelGGL((copy_plan_persistent_kernel<false, false>), grid, block, 0, st, table, nseg, plan->n_chunks,
                       cpb, xcd_stride, run, rb.src, rb.dst, stab, dtab);
  hipError_t le = hipGetLastError();
  if (tab_owned) (void)hipFreeAsync(tab, st);
  if (le != hipSuccess) return hip_fail(le, "copy_plan_persistent_kernel launch");
  return note_launch(plan, dev, st);
}

int emrs_plan_compare(emrs_plan *plan, void *const *src_bases, void *const *dst_bases, const uint32_t *groups,
                      const uint32_t *aux_groups, uint32_t n_groups, emrs_compare_stats *stats, void *stream) {
  g_last_error.clear();
  CompareJob job;
  int rc = compare_setup(plan, src_bases, dst_bases, groups, aux_groups, n_groups, stats, &job);
  if (rc || plan->n_chunks == 0) return rc;
  int dev = 0;
  rc = compare_device(&job, &dev);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // The comparison allocates its accumulators and waits for the stream.
  rc = refuse_capture(st, "emrs_plan_compare");
  if (rc) return rc;
  DevSeg *table = nullptr;
  rc = device_table(plan, dev, st, &table);
  if (rc) return rc;

  uint64_t *tab = nullptr;
  bool tab_owned = false;
  rc = pointer_table(plan, dev, job.rb, st, &tab, &tab_owned);
  if (rc) return rc;
  uint32_t *cseg = nullptr, *flags = nullptr;  // no chunk table when it does not fit: then a persistent grid
  rc = chunk_table(plan, dev, st, table, &cseg);
  if (rc == EMRS_OK) rc = take_flags(plan, dev, st, &flags);
  if (rc) {
    if (tab_owned) {
      (void)hipFreeAsync(tab, st);
      (void)hipStreamSynchronize(st);  // its upload reads job's vector
    }
    return rc;
  }
  job.cseg = cseg;

  // A switch that is correct, the common case, costs one launch and one wait:
  // no buffer is allocated, uploaded or read back.  A comparison of 1 GB used
  // to allocate, upload the groups, clear, launch, read back and free.
  const size_t nd = plan->segs.size();
  uint32_t *any = take_any_slot();
  if (any) *static_cast<volatile uint32_t *>(any) = 0;
  hipError_t e = differ_launch(plan, job, table, tab, DifferMarks{flags, any}, st);
  const hipError_t se = hipStreamSynchronize(st);
  if (e == hipSuccess) e = se;
  const bool differs = any && *static_cast<volatile uint32_t *>(any) != 0;
  give_any_slot(any);
  std::vector<GroupAcc> host(n_groups);
  bool clean = e == hipSuccess, marked = differs;
  if (e == hipSuccess && !any) {  // no word was set: the flags themselves tell
    std::vector<uint32_t> found(nd);
    e = hipMemcpyAsync(found.data(), flags, nd * sizeof(uint32_t), hipMemcpyDeviceToHost, st);
    const hipError_t fe = hipStreamSynchronize(st);
    if (e == hipSuccess) e = fe;
    clean = e == hipSuccess;
    marked = std::any_of(found.begin(), found.end(), [](uint32_t f) { return f != 0; });
  }
  if (e == hipSuccess && marked) {
    clean = false;
    const size_t acc_bytes = align256((size_t)n_groups * sizeof(GroupAcc));
    const size_t grp_bytes = align256(2 * nd * sizeof(uint32_t));
    char *buf = nullptr;
    e = hipMalloc(&buf, acc_bytes + grp_bytes + align256(n_groups));
    if (e == hipSuccess) {
      e = compare_marked(plan, job, table, reinterpret_cast<uint32_t *>(buf + acc_bytes), tab,
                         reinterpret_cast<GroupAcc *>(buf), reinterpret_cast<uint8_t *>(buf + acc_bytes + grp_bytes),
                         nullptr, flags, st, host);
      (void)hipFree(buf);
      clean = e == hipSuccess;
    }
  }
  give_flags(plan, dev, st, flags, clean);
  if (tab_owned) (void)hipFreeAsync(tab, st);
  if (e != hipSuccess) return hip_fail(e, "compare_plan_kernel");
  compare_finish(host, stats);
  return EMRS_OK;
}

int emrs_plan_compare_static(emrs_plan *plan, void *const *src_bases, void *const *dst_bases,
                             const uint32_t *groups, const uint32_t *aux_groups, uint32_t n_groups,
                             emrs_compare_stats *stats, void *stream) {
  g_last_error.clear();
  CompareJob job;
  int rc = compare_setup(plan, src_bases, dst_bases, groups, aux_groups, n_groups, stats, &job);
  if (rc || plan->n_chunks == 0) return rc;
  // Everything the kernel reads or writes beyond the caller's buffers lives in `scratch`, in
  // 256-byte aligned regions: accumulators, group ids, the segment table, the pointer table.
  const size_t nd = plan->segs.size();
  const size_t acc_bytes = align256((size_t)n_groups * sizeof(GroupAcc));
  const size_t grp_bytes = align256(2 * nd * sizeof(uint32_t));
  const size_t seg_bytes = align256(nd * sizeof(DevSeg));
  const size_t ptr_bytes = job.rb.table ? align256(job.rb.ptrs.size() * sizeof(uint64_t)) : 0;
  const size_t act_bytes = align256(n_groups);
  const size_t need = acc_bytes + grp_bytes + seg_bytes + ptr_bytes + act_bytes;
  if (need > EMRS_STATIC_SCRATCH_BYTES) {
    char msg[200];
    snprintf(msg, sizeof msg,
             "the comparison needs %zu bytes of scratch (%zu segments, %u groups); the allocation-free "
             "entry point holds at most %u: use emrs_plan_compare",
             need, nd, n_groups, (unsigned)EMRS_STATIC_SCRATCH_BYTES);
    return fail(EMRS_ERR_TOO_LARGE, msg);
  }
  int dev = 0;
  rc = compare_device(&job, &dev);
  if (rc) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  rc = refuse_capture(st, "emrs_plan_compare_static");  // it waits for the stream
  if (rc) return rc;
  unsigned char *base = nullptr;
  rc = scratch_of(dev, &base);
  if (rc) return rc;

  // One call at a time per device: the array is shared by every call on it.
  std::lock_guard<std::mutex> lk(*scratch_call_mutex(dev));
  GroupAcc *acc = reinterpret_cast<GroupAcc *>(base);
  uint32_t *grp = reinterpret_cast<uint32_t *>(base + acc_bytes);
  DevSeg *table = reinterpret_cast<DevSeg *>(base + acc_bytes + grp_bytes);
  uint64_t *tab = job.rb.table ? reinterpret_cast<uint64_t *>(base + acc_bytes + grp_bytes + seg_bytes) : nullptr;
  uint8_t *active = base + acc_bytes + grp_bytes + seg_bytes + ptr_bytes;
  hipError_t e = hipMemcpyAsync(table, plan->segs.data(), nd * sizeof(DevSeg), hipMemcpyHostToDevice, st);
  if (e == hipSuccess && tab)
    e = hipMemcpyAsync(tab, job.rb.ptrs.data(), job.rb.ptrs.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st);
  std::vector<GroupAcc> host(n_groups);
  std::vector<uint32_t> found(nd);
  std::vector<uint8_t> mark(n_groups, 0);
  job.cseg = existing_chunk_table(plan, dev);  // never built here: that would allocate
  // The first pass's flags lie where the second pass's group ids go.
  if (e == hipSuccess) e = clear_words(grp, nd, st);
  if (e == hipSuccess) e = differ_launch(plan, job, table, tab, DifferMarks{grp, nullptr}, st);
  if (e == hipSuccess) e = hipMemcpyAsync(found.data(), grp, nd * sizeof(uint32_t), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e == hipSuccess && job.marked_groups(plan, found, &mark))
    e = compare_marked(plan, job, table, grp, tab, acc, active, &mark, nullptr, st, host);
  // The host copies above read job's and plan's vectors: wait before they can go.
  const hipError_t se = hipStreamSynchronize(st);
  if (e == hipSuccess) e = se;
  if (e != hipSuccess) return hip_fail(e, "compare_plan_kernel (static scratch)");
  compare_finish(host, stats);
  return EMRS_OK;
}

int emrs_plan_destroy(emrs_plan *plan) {
  if (!plan) return EMRS_OK;
  int prev = 0;
  (void)hipGetDevice(&prev);
  const size_t n_dev = std::max({plan->dev_tables.size(), plan->ptr_tables.size(), plan->abs_tables.size(),
                                  plan->chunk_tables.size(), plan->launch_events.size(), plan->differ_flags.size()});
  for (size_t d = 0; d < n_dev; ++d) {
    DevSeg *segs = d < plan->dev_tables.size() ? plan->dev_tables[d] : nullptr;
    uint64_t *ptrs = d < plan->ptr_tables.size() ? plan->ptr_tables[d] : nullptr;
    DevSeg *abs = d < plan->abs_tables.size() ? plan->abs_tables[d] : nullptr;
    uint32_t *chunks = d < plan->chunk_tables.size() ? plan->chunk_tables[d] : nullptr;
    std::vector<hipEvent_t> evs = d < plan->launch_events.size() ? plan->launch_events[d] : std::vector<hipEvent_t>();
    uint32_t *flags = d < plan->differ_flags.size() ? plan->differ_flags[d] : nullptr;
    if (!(segs || ptrs || abs || chunks || flags || !evs.empty())) continue;
    (void)hipSetDevice((int)d);
    // A graph may replay the plan's launches at any time: only a drained device is safe.
    if (plan->captured) (void)hipDeviceSynchronize();
    // The tables are freed on the library's stream after the launches that read them, and only
    // after those: work on other streams is not waited for, and the host does not block.
    hipStream_t fs = free_stream((int)d);
    if (!fs) {
      (void)hipDeviceSynchronize();
    } else {
      for (hipEvent_t ev : evs) (void)hipStreamWaitEvent(fs, ev, 0);
    }
    for (hipEvent_t ev : evs) (void)hipEventDestroy(ev);
    for (void *t : {static_cast<void *>(segs), static_cast<void *>(ptrs), static_cast<void *>(abs),
                    static_cast<void *>(chunks), static_cast<void *>(flags)})
      if (t) (void)hipFreeAsync(t, fs);
  }
  (void)hipSetDevice(prev);
  delete plan;
  return EMRS_OK;
}

int emrs_get_tuning(emrs_tuning *out) {
  if (!out) return fail(EMRS_ERR_INVALID_ARGUMENT, "NULL argument");
  out->blocks_per_cu = g_tuning.blocks_per_cu.load();
  out->nontemporal = g_tuning.nontemporal.load();
  out->xcd_remap = g_tuning.xcd_remap.load();
  out->run = g_tuning.run.load();
  out->persistent = g_tuning.persistent.load();
  out->lanes = g_tuning.lanes.load();
  out->units = g_tuning.units.load();
  out->buffer_ops = g_tuning.buffer_ops.load();
  out->chunk_index = g_tuning.chunk_index.load();
  out->warm_tables = g_tuning.warm_tables.load();
  return EMRS_OK;
}

int emrs_set_tuning(const emrs_tuning *t) {
  if (!t) return fail(EMRS_ERR_INVALID_ARGUMENT, "NULL argument");
  if (t->blocks_per_cu > 64) return fail(EMRS_ERR_INVALID_ARGUMENT, "blocks_per_cu must be in [0, 64]");
  if (t->run > (1u << 20)) return fail(EMRS_ERR_INVALID_ARGUMENT, "run must be in [0, 2^20]");
  if (t->xcd_remap > 2) return fail(EMRS_ERR_INVALID_ARGUMENT, "xcd_remap must be 0, 1 or 2");
  if (t->lanes != 0 && t->lanes != 64 && t->lanes != 128 && t->lanes != 256)
    return fail(EMRS_ERR_INVALID_ARGUMENT, "lanes must be 0, 64, 128 or 256");
  const uint32_t lanes = t->lanes ? t->lanes : 64;
  // 0 keeps the pre-existing meaning: one chunk of 256 units per workgroup.
  const uint32_t units = t->units ? t->units : kChunkUnits / lanes;
  if (units != 1 && units != 2 && units != 4) return fail(EMRS_ERR_INVALID_ARGUMENT, "units must be 0, 1, 2 or 4");
  if (kChunkUnits % (lanes * units)) return fail(EMRS_ERR_INVALID_ARGUMENT, "lanes * units must divide 256");
  g_tuning.blocks_per_cu.store(t->blocks_per_cu);
  g_tuning.nontemporal.store(t->nontemporal ? 1 : 0);
  g_tuning.xcd_remap.store(t->xcd_remap);
  g_tuning.run.store(t->run);
  g_tuning.persistent.store(t->persistent ? 1 : 0);
  g_tuning.lanes.store(lanes);
  g_tuning.units.store(units);
  g_tuning.buffer_ops.store(t->buffer_ops ? 1 : 0);
  g_tuning.chunk_index.store(t->chunk_index ? 1 : 0);
  g_tuning.warm_tables.store(t->warm_tables ? 1 : 0);
  return EMRS_OK;
}

}  // extern "C"
