// reshard.hip -- plan-driven pack / unpack engine for Suika state migration on
// MI355X (gfx950).  One source file: the C ABI declared in
// include/suika_reshard.h, the host-side plan builder, and the device kernels.
//
// Reference behaviour reproduced (paths relative to the Suika repository):
//   Suika/migration.py:290-312  get_send_tensor: chunk(n, dim)[k].contiguous()
//   Suika/migration.py:531-541  cat(pieces, dim=slice_dim) / clone()
// Both are pure byte movement.  The Python host lowers every TransferOp x
// sub-field into 2-D region moves (sr_piece); this file validates them, lays
// out the per-peer buffers and executes each phase -- pack (sources -> peer
// buffers), unpack (peer buffers -> destinations) or gather (sources ->
// destinations directly) -- as a single launch.
//
// Device design
//   * A phase is a list of items, one per piece.  An item is
//     a 2-D byte region: `rows` rows of `row_bytes` bytes at a source and a
//     destination stride.  Regions that are contiguous on both sides are
//     collapsed to one long row.
//   * Items are cut into tiles of `tile_bytes` (16 KiB) source bytes; one
//     workgroup (1024 lanes = 16 wave64) moves one tile, 16 bytes per lane,
//     and the grid is the tile count (or a grid-stride loop when capped).
//     Phases of few, small or several-pass tiles have other workgroups (Shape),
//     and some items of large phases two tiles to a workgroup (record_bytes).
//     Tiles balance the work whatever the tensor sizes (8 KB norms to GB
//     embeddings).
//   * A lane loads once, stores once and ends.  Two workgroups fill a compute
//     unit, so 32 KiB of reads are in flight there: HBM moves a flat copy of
//     2 GiB at 6.65 TB/s with that, at 6.1 with twice as much (two loads per
//     lane of 512), and at 4.1-5.4 with waves that go on to another tile,
//     because a load's data is waited for behind the stores issued before it.
//   * So the way from the launch to the load is short: the kernel arguments
//     arrive in registers, a tile's record holds the addresses of a
//     contiguous copy, a record line is read into the die's L2 256 tiles
//     before its workgroup starts, the lines of the next items with it
//     (Ahead), and the forms of large tensors come first in a kernel of 26 KB
//     (one of 46 KB, before the forms were folded: 3% slower).
//   * The tile list follows the tensor address each item starts at and is cut
//     into 8 segments: workgroups go to the 8 XCDs round-robin, so each XCD
//     walks one contiguous eighth of the list (and of its records) and the
//     tiles in flight come from 8 distant regions; a single window of
//     consecutive tiles keeps the read and write streams at a fixed distance
//     and leaves HBM bandwidth idle.
//     Side-by-side strided items (the column bands of one dim -1 `cat`) deal
//     out their tiles row block by row block, so each destination row is
//     written by adjacent tiles.
//   * Lanes move 16-byte vectors where addresses, strides and row widths are
//     multiples of 16 bytes, and at any alignment in contiguous pieces and in
//     long rows of 1- and 2-byte alignment; narrower vectors otherwise
//     (bind_item).  Loads are non-temporal, and how stores are cached follows
//     from whether they write whole lines (Policy).
//   * Strided regions (row-parallel dim -1 slices) map a tile-relative byte
//     position to (row, col) with a multiply-high division by the row width
//     (Granlund-Montgomery invariant-integer division), computed per item
//     on the host.
//   * The unpack RECAST item reads f32 once and writes the f32 copy and the
//     bf16 round-to-nearest-even copy in the same pass.
//   * The copy kernels use no LDS: every region row is >= 768 bytes at the
//     configured shapes, so a direct coalesced copy already issues full-width
//     bursts; a transpose is never needed because no piece changes the
//     element order within a row.
//
// Host design
//   * sr_plan_create is host only and O(pieces): validation, coverage, the
//     buffer layout the API reports, and one pointer-independent descriptor
//     per item.  The CPU test-suite exercises it without a GPU.
//     Each item's first tile is a prefix sum over the items.
//   * Phases of at most kHostTableTiles tiles have their tables written by the
//     host, at each launch on new pointers (run_small).
//   * The O(tiles) work of larger ones runs on the GPU at first use of a
//     phase: an emit kernel writes the tile table, and prefix sums (wave64
//     shuffle scans, wave totals through LDS) give each peer's 256-byte
//     aligned buffer offsets.  The Llama2-7B share has 1.44 M tiles per phase;
//     building them on the host took 0.12 s and a 35 MB upload per phase.
//   * Tile records and items hold absolute addresses.  When the pointers of a
//     larger phase change, only the pointer table is uploaded and the emit
//     kernel writes both again from the descriptors and the device-side buffer
//     offsets (2624 to 16384 tiles 4.1-4.4 us; a table of items alone, bound
//     by a kernel of one lane per item, took 4.2).  Read in place in pinned
//     memory, without the upload, the emit is 1 us a launch slower (4096 tiles
//     33.1 -> 34.1 us).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "suika_reshard.h"
#include "sr_internal.h"

namespace sr_internal {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

const char* last_error() { return g_last_error.c_str(); }

int dtype_size(int32_t dt) {
  switch (dt) {
    case SR_DT_U8: return 1;
    case SR_DT_BF16: return 2;
    case SR_DT_F16: return 2;
    case SR_DT_F32: return 4;
    case SR_DT_F64: return 8;
    case SR_DT_I32: return 4;
    case SR_DT_I64: return 8;
    default: return 0;
  }
}

}  // namespace sr_internal

namespace {

// What the largest copy workgroup, 1024 lanes, moves with one 16-byte vector
// (or as many narrower ones as make 16 bytes) per lane: a tile.
constexpr uint32_t kPassBytes = 16384;
constexpr uint32_t kDefaultTileBytes = kPassBytes;
constexpr uint64_t kBufAlign = 256;
// Segments of the tile list, one per accelerator complex die (XCD) of an
// MI355X; the dies take workgroups round-robin.
constexpr uint32_t kXcds = 8;
// A RECAST item that writes the f32 copy and the bf16 copy moves 2.5x its
// source bytes (a COPY item 2x); its tiles, as plans count them, hold
// tile_bytes >> this many source bytes.  A workgroup takes two of them where
// it has lanes for both (record_bytes).
constexpr uint32_t kRecastTileShift = 1;

// ---------------------------------------------------------------- errors

using sr_internal::fail;

#define SR_HIP_TRY(expr)                                                      \
  do {                                                                        \
    hipError_t e_ = (expr);                                                   \
    if (e_ != hipSuccess)                                                     \
      return fail(SR_EHIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
  } while (0)

using sr_internal::dtype_size;

// ------------------------------------------------ invariant integer division
// Granlund & Montgomery, "Division by invariant integers using
// multiplication" (PLDI 1994), Figure 4.1 with N = 32: for 1 <= d < 2^31 and
// any 32-bit n, q = (t + ((n - t) >> s1)) >> s2 with t = mulhi(m, n).

struct DivMagic {
  uint32_t m;
  uint32_t s1;
  uint32_t s2;
};

DivMagic div_magic(uint32_t d) {
  uint32_t l = 0;
  while ((uint64_t(1) << l) < d) ++l;               // l = ceil(log2 d)
  const uint64_t num = (uint64_t(1) << 32) * ((uint64_t(1) << l) - d);
  DivMagic r;
  r.m = uint32_t(num / d + 1);
  r.s1 = l < 1 ? l : 1;
  r.s2 = l > 1 ? l - 1 : 0;
  return r;
}

__host__ __device__ inline uint32_t div_apply(uint32_t n, uint32_t m, uint32_t s1,
                                              uint32_t s2) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t t = __umulhi(m, n);
#else
  const uint32_t t = uint32_t((uint64_t(m) * n) >> 32);
#endif
  return (t + ((n - t) >> s1)) >> s2;
}

// ------------------------------------------------------- device structures

enum : uint32_t {
  kKindCopy = 0,
  kKindRecast = 1,
  kKindZero = 2,
};

// One piece bound to its objects' addresses: what its tiles read beyond
// their own records.
struct alignas(16) DevItem {
  uint64_t src;           // absolute address of the region origin
  uint64_t dst;
  uint64_t dst2;          // bf16 target of RECAST
  uint64_t src_stride;    // bytes between rows
  uint64_t dst_stride;
  uint64_t dst2_stride;
  uint32_t row_bytes;     // source bytes per row; 0 = contiguous (one row)
  uint32_t magic;         // division by row_bytes
  uint32_t shifts;        // s1 | s2 << 8
  uint32_t flags;         // bits 0-3 kind, 4-7 log2 of the vector bytes, kItemMerge
};
static_assert(sizeof(DevItem) == 64, "DevItem layout");

constexpr uint32_t kItemMerge = 1u << 8;   // partly written lines are left to the L2 to merge

// How a tile is moved; "rows" are strided.  ZERO rows are copied from a source
// of no bytes.  The first seven are the tiles of large tensors; of those the
// first five write whole lines through.
enum : uint32_t {
  kOpCopy = 0,           // contiguous
  kOpRows = 1,           // COPY and ZERO rows of a multiple of 16 bytes
  kOpRecast = 2,         // contiguous f32 -> f32 copy (where there is one) + bf16 copy
  kOpZero = 3,           // contiguous
  kOpRecastRows = 4,     // rows of a multiple of 16 bytes
  kOpCopyStream = 5,     // kOpCopy, streamed
  kOpRowsStream = 6,     // kOpRows, streamed
  kOpRows8 = 7,          // COPY rows in 8-byte vectors, streamed
  kOpRows4 = 8,
  kOpWide = 9,           // COPY and ZERO rows of other widths, in 16-byte vectors
  kOpNarrow = 10,        // vectors of less than 16 bytes otherwise
  kOpRecastRowsPart = 11,   // kOpRecastRows, streamed or left to the L2
  kOpRecastStream = 12,     // kOpRecast, streamed
  kOpZeroStream = 13,       // kOpZero, streamed
  kOpFar = 14,           // rows 2 GiB or more apart
};

// The record of one tile.  A contiguous COPY or ZERO tile needs nothing else.
struct alignas(8) DevTile {
  uint64_t src;      // contiguous: address of its first source byte; strided: first row
  uint64_t dst;      // contiguous: address of its first destination byte (0: none); strided: byte
                     // column of the tile start in its first row
  uint32_t item;
  uint32_t info;     // bits 0-24 source bytes, 25-31 op
};
static_assert(sizeof(DevTile) == 24, "DevTile layout");

constexpr uint32_t kTileOpBit = 25;
constexpr uint32_t kTileBytesMask = (1u << kTileOpBit) - 1;

// -------------------------------------------------------------- device code

template <int VB> struct VecOf;
template <> struct VecOf<16> { typedef unsigned int type __attribute__((ext_vector_type(4))); };
template <> struct VecOf<8> { typedef unsigned int type __attribute__((ext_vector_type(2))); };
template <> struct VecOf<4> { typedef unsigned int type; };
template <> struct VecOf<2> { typedef unsigned short type; };
template <> struct VecOf<1> { typedef unsigned char type; };

// A tile's source or destination bytes as a buffer resource: 32-bit offsets
// from a base in scalar registers, and the hardware drops what lies outside
// `bytes`, so lanes past a tile's end need no branch.
typedef __amdgpu_buffer_rsrc_t Region;

__device__ __forceinline__ Region region(uint64_t addr, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(addr), 0, bytes, 0x00027000);
}

// Bytes of the region a strided tile addresses, and an offset outside it for
// the lanes past the tile's end.
constexpr uint32_t kNearBytes = 1u << 31;
constexpr uint32_t kNowhere = 0xfffffff0u;

// Cache policies: the aux bits of gfx950's buffer instructions (2 = nt,
// 16 = sc1).  Loads are non-temporal.  Stores of whole 64-byte lines write
// through the L2: the lines then do not wait there for an eviction that
// competes with the reads (flat copy of 2 GiB: 6.65 TB/s, nt 6.50; zero fill
// of 4 GiB 7.66, nt 6.90).  Lines that several waves or rows write in parts are left for
// the L2 to merge, as streaming lines or, for short rows, as ordinary ones
// (side by side rows of 4 bytes: through 3.0 TB/s, nt 3.6, ordinary 5.1; of
// 36 kB + 16 bytes: 5.4, 5.9, 5.5).  Where whole lines are streamed all the
// same: stream_whole.
enum Policy : int {
  kCached = 0,
  kStream = 2,
  kThrough = 16,
};

template <int VB, bool NT>
__device__ __forceinline__ typename VecOf<VB>::type ld(Region r, uint32_t off) {
  constexpr int aux = NT ? kStream : kCached;
  typedef typename VecOf<VB>::type V;
  if constexpr (VB == 16) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, aux));
  else if constexpr (VB == 8) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, aux));
  else if constexpr (VB == 4) return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, aux);
  else if constexpr (VB == 2) return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, aux);
  else return __builtin_amdgcn_raw_buffer_load_b8(r, off, 0, aux);
}

template <int VB, Policy POLICY>
__device__ __forceinline__ void st(Region r, uint32_t off, typename VecOf<VB>::type v) {
  if constexpr (VB == 16) __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, POLICY);
  else if constexpr (VB == 8) __builtin_amdgcn_raw_buffer_store_b64(v, r, off, 0, POLICY);
  else if constexpr (VB == 4) __builtin_amdgcn_raw_buffer_store_b32(v, r, off, 0, POLICY);
  else if constexpr (VB == 2) __builtin_amdgcn_raw_buffer_store_b16(v, r, off, 0, POLICY);
  else __builtin_amdgcn_raw_buffer_store_b8(v, r, off, 0, POLICY);
}

// The same through 64-bit addresses (kOpFar).
#define SR_GLOBAL __attribute__((address_space(1)))

template <int VB>
__device__ __forceinline__ typename VecOf<VB>::type ld_far(uint64_t addr) {
  return __builtin_nontemporal_load((const SR_GLOBAL typename VecOf<VB>::type*)addr);
}

template <int VB>
__device__ __forceinline__ void st_far(uint64_t addr, typename VecOf<VB>::type v) {
  __builtin_nontemporal_store(v, (SR_GLOBAL typename VecOf<VB>::type*)addr);
}

// Row and column of the source byte `b` counted from the start of a strided
// tile: a multiply-high division by the row width.
struct RowMap {
  uint32_t c_base, width, magic, s1, s2;

  __host__ __device__ __forceinline__ void at(uint32_t b, uint32_t& row, uint32_t& col) const {
    const uint32_t x = c_base + b;
    row = div_apply(x, magic, s1, s2);
    col = x - row * width;
  }
};

__device__ __forceinline__ RowMap row_map(const DevItem& it, uint32_t column) {
  return {column, it.row_bytes, it.magic, it.shifts & 0xffu, it.shifts >> 8};
}

// The 16-byte vector of a tile of rows of at least 16 bytes that starts at
// tile byte `b`: its row and column, and whether its bytes go on in the next
// row, where another vector starts at column 0.
struct RowVec {
  uint32_t row, col;
  bool in, next;
};

__host__ __device__ __forceinline__ RowVec row_vec(const RowMap& rows, uint32_t b, uint32_t nbytes) {
  RowVec v;
  uint32_t col;
  rows.at(b, v.row, col);
  v.in = b < nbytes;
  v.col = col < rows.width - 16u ? col : rows.width - 16u;
  v.next = v.in && v.col != col && b + (rows.width - col) < nbytes;
  return v;
}

// The offset of the 16-byte vector of a contiguous tile (16 bytes or more)
// that starts at byte `b`; past the tile's end for lanes that have none.
__host__ __device__ __forceinline__ uint32_t contiguous_vec(uint32_t b, uint32_t nbytes) {
  return b < nbytes && b > nbytes - 16 ? nbytes - 16 : b;
}

// Where a vector of a tile goes: its offsets in the source, destination and
// bf16 regions.  Lanes past the tile's end, and second vectors that are not
// there, get an offset outside the regions.
struct Place {
  uint32_t src, dst, half;
};

// The places of the vectors `step` bytes apart in a tile: the first by a
// division, the others by additions.  Width 0: one row.
struct RowWalk {
  uint32_t width, right, col;   // `step` on: some rows down, `right` columns on
  Place at, by, wrap;           // wrap: to the next row's start

  __host__ __device__ __forceinline__ RowWalk(const RowMap& rows, uint32_t b, uint32_t step, uint32_t ss, uint32_t ds,
                                              uint32_t hs)
      : width(0xffffffffu), right(step), col(b) {
    uint32_t row = 0, down = 0;
    if (rows.width) {
      width = rows.width;
      down = div_apply(step, rows.magic, rows.s1, rows.s2);
      right = step - down * width;
      rows.at(b, row, col);
    }
    at = {row * ss + col, row * ds + col, row * hs + (col >> 1)};
    by = {down * ss + right, down * ds + right, down * hs + (right >> 1)};
    wrap = {ss - width, ds - width, hs - (width >> 1)};
  }

  __host__ __device__ __forceinline__ void advance() {
    col += right;
    const bool over = col >= width;
    col -= over ? width : 0;
    at.src += by.src + (over ? wrap.src : 0);
    at.dst += by.dst + (over ? wrap.dst : 0);
    at.half += by.half + (over ? wrap.half : 0);
  }
};

// float -> bfloat16, round to nearest, ties to even; NaN -> 0x7FC0.
// This is the standard integer rounding of the upper half-word: add
// 0x7FFF plus the lowest kept bit, then truncate.
__device__ __forceinline__ uint32_t bf16_rne(uint32_t u) {
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

template <int NE>
__device__ __forceinline__ typename VecOf<2 * NE>::type to_bf16(typename VecOf<4 * NE>::type v) {
  typename VecOf<2 * NE>::type h;
  if constexpr (NE == 4) {
    h.x = bf16_rne(v.x) | (bf16_rne(v.y) << 16);
    h.y = bf16_rne(v.z) | (bf16_rne(v.w) << 16);
  } else {
    h = (unsigned short)bf16_rne(v);
  }
  return h;
}

// What a tile reads and writes; a region of no bytes takes no store.
struct Regions {
  Region src, dst, half;
};

// Stores a loaded vector: COPY the bytes, RECAST also the rounded ones.
template <uint32_t KIND, int VB, Policy POLICY>
__device__ __forceinline__ void put(const Regions& r, const Place& at, typename VecOf<VB>::type v) {
  st<VB, POLICY>(r.dst, at.dst, v);
  if constexpr (KIND == kKindRecast) st<VB / 2, POLICY>(r.half, at.half, to_bf16<VB / 4>(v));
}

// The tile records this far ahead of a workgroup's own are read into the
// die's L2 (one read per kAheadStep records, which span less than a cache
// line), so that a record is there when its workgroup starts.  The read is
// issued behind the tile's loads and done with before its stores: a wait
// after them would hold the wave until they are written.  256 records cover a
// die's tiles in flight twice over (flat copy of 2 GiB: 6.26 TB/s without,
// 6.65 with; 512 ahead gave the same, 2048 3% less).
//
// The same read takes the lines of the next 16 items along, for tiles that
// need theirs: each new item's line otherwise stops all the tiles that are in
// flight on a die (columns split off 64 tiles an item, 1024 items: 381 us
// without, 328 with; 64 items 329 and 329).  One read for both, as a second
// costs every such tile 10%.
constexpr uint32_t kAhead = 256;
constexpr uint32_t kAheadStep = 4;
constexpr uint32_t kAheadItems = 16;

struct Ahead {
  const DevTile* tiles;
  uint32_t i, n, lane;
  const DevItem* items;
  uint32_t item, n_items;   // item: n_items where a tile needs none
  template <int B>
  __device__ __forceinline__ void touch() const {
    if (lane >= B - 64 && i % kAheadStep == 0 && i + kAhead < n) {
      constexpr uint32_t kPerLine = 128 / sizeof(DevItem);
      const uint32_t l = lane - (B - 64), k = item + l * kPerLine;
      const uint32_t* at = l < kAheadItems / kPerLine && k < n_items ? &items[k].flags : &tiles[i + kAhead].info;
      const uint32_t x = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      asm volatile("" ::"v"(x));
    }
  }
};

// A tile of at least 16 contiguous bytes, at any alignment: 16 bytes per
// lane, the last vector moved back to end with the tile (it then writes
// bytes of its neighbour again, with the same values).
template <uint32_t KIND, Policy POLICY, bool NT, int B, int U>
__device__ __forceinline__ void contiguous_tile(const Regions& r, uint32_t nbytes, const Ahead& ahead) {
  for (uint32_t base = 0; base < nbytes; base += B * U * 16) {
    uint32_t off[U];
    VecOf<16>::type v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      off[u] = contiguous_vec(base + (u * B + ahead.lane) * 16, nbytes);
      v[u] = VecOf<16>::type(0);
      if constexpr (KIND != kKindZero) v[u] = ld<16, NT>(r.src, off[u]);
    }
    if (KIND != kKindZero && base == 0) ahead.touch<B>();
#pragma unroll
    for (int u = 0; u < U; ++u) put<KIND, 16, NT ? POLICY : kCached>(r, Place{off[u], off[u], off[u] >> 1}, v[u]);
  }
}

// A tile of rows of a multiple of 16 bytes, at any alignment: 16 bytes per lane.
template <uint32_t KIND, Policy POLICY, bool NT, int B, int U>
__device__ __forceinline__ void rows_tile(const Regions& r, const DevItem& it, uint32_t column, uint32_t nbytes,
                                          const Ahead& ahead) {
  const RowMap rows = row_map(it, column);
  const uint32_t ss = uint32_t(it.src_stride), ds = uint32_t(it.dst_stride), hs = uint32_t(it.dst2_stride);
  for (uint32_t base = 0; base < nbytes; base += B * U * 16) {
    Place at[U];
    VecOf<16>::type v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t b = base + (u * B + ahead.lane) * 16;
      uint32_t row, col;
      rows.at(b, row, col);
      const bool in = b < nbytes;
      at[u] = {in ? row * ss + col : kNowhere, in ? row * ds + col : kNowhere, in ? row * hs + (col >> 1) : kNowhere};
      v[u] = ld<16, NT>(r.src, at[u].src);
    }
    if (base == 0) ahead.touch<B>();
#pragma unroll
    for (int u = 0; u < U; ++u) put<KIND, 16, NT ? POLICY : kCached>(r, at[u], v[u]);
  }
}

// The regions of a strided tile (or of a contiguous piece that is one tile,
// from its origin).
__device__ __forceinline__ Regions row_regions(const DevItem& it, uint64_t row) {
  return {region(it.src + row * it.src_stride, it.src ? kNearBytes : 0),
          region(it.dst + row * it.dst_stride, it.dst ? kNearBytes : 0),
          region(it.dst2 + row * it.dst2_stride, it.dst2 ? kNearBytes : 0)};
}

// The regions of a contiguous RECAST tile.
__device__ __forceinline__ Regions recast_regions(const DevItem& it, const DevTile& t, uint32_t nbytes) {
  return {region(t.src, nbytes), region(t.dst, t.dst ? nbytes : 0),
          region(it.dst2 + ((t.src - it.src) >> 1), nbytes >> 1)};
}

// COPY and ZERO rows of at least 16 bytes at any alignment, in 16-byte vectors.
// A vector that runs over the end of its row becomes two, the last 16 bytes of
// that row and the first 16 of the next; the bytes that neighbouring lanes
// write too have the same values.
template <Policy POLICY, bool NT, int B>
__device__ __forceinline__ void wide_tile(const DevItem& it, const DevTile& t, uint32_t nbytes, const Ahead& ahead) {
  const Regions r = row_regions(it, t.src);
  const RowMap rows = row_map(it, uint32_t(t.dst));
  const uint32_t ss = uint32_t(it.src_stride), ds = uint32_t(it.dst_stride);
  for (uint32_t base = 0; base < nbytes; base += B * 16) {
    const RowVec x = row_vec(rows, base + ahead.lane * 16, nbytes);
    const uint32_t from = x.in ? x.row * ss + x.col : kNowhere, to = x.in ? x.row * ds + x.col : kNowhere;
    const uint32_t from2 = x.next ? (x.row + 1) * ss : kNowhere, to2 = x.next ? (x.row + 1) * ds : kNowhere;
    const VecOf<16>::type v = ld<16, NT>(r.src, from), w = ld<16, NT>(r.src, from2);
    if (base == 0) ahead.touch<B>();
    st<16, NT ? POLICY : kCached>(r.dst, to, v);
    st<16, NT ? POLICY : kCached>(r.dst, to2, w);
  }
}

// Vectors of the widest aligned type that divides the rows (RECAST: one
// element).  A wave takes consecutive bytes, W vectors per lane a wave's
// width apart: each vector's lines are then written by one wave (side by
// side f32 rows of 16396 bytes: 5.7 TB/s, with the vectors of a lane a
// workgroup's width apart 5.2).
template <uint32_t KIND, int VB, Policy POLICY, bool NT, int B, int W = VB == 8 ? 2 : 4>
__device__ __forceinline__ void narrow_tile(const DevItem& it, const DevTile& t, uint32_t nbytes, const Ahead& ahead) {
  constexpr uint32_t kStep = 64 * VB;
  const bool strided = it.row_bytes != 0;
  const Regions r = row_regions(it, strided ? t.src : 0);
  const RowMap rows = row_map(it, strided ? uint32_t(t.dst) : 0);
  for (uint32_t base = 0; base < nbytes; base += B * VB * W) {
    uint32_t b = base + (ahead.lane >> 6) * (W * kStep) + (ahead.lane & 63) * VB;
    RowWalk walk(rows, b, kStep, uint32_t(it.src_stride), uint32_t(it.dst_stride), uint32_t(it.dst2_stride));
    Place at[W];
    typename VecOf<VB>::type v[W];
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const bool in = b < nbytes;
      at[u] = {kNowhere, in ? walk.at.dst : kNowhere, in ? walk.at.half : kNowhere};
      v[u] = ld<VB, NT>(r.src, in ? walk.at.src : kNowhere);
      b += kStep;
      walk.advance();
    }
    if (base == 0) ahead.touch<B>();
#pragma unroll
    for (int u = 0; u < W; ++u) put<KIND, VB, NT ? POLICY : kCached>(r, at[u], v[u]);
  }
}

// kOpNarrow.  A body for each policy here and above: one that branches before
// its stores is 10% slower (rows of 17 bytes 458 us, so 398; of 2 bytes 319 /
// 290), and large shares 0.4% where their forms branch.
template <bool NT, int B>
__device__ __forceinline__ void narrow_forms(const DevItem& it, const DevTile& t, uint32_t nbytes, const Ahead& ahead) {
  const uint32_t lv = (it.flags >> 4) & 0xfu;
  const bool merge = it.flags & kItemMerge;
  if ((it.flags & 0xfu) == kKindRecast) {
    if (merge) narrow_tile<kKindRecast, 4, kCached, NT, B>(it, t, nbytes, ahead);
    else narrow_tile<kKindRecast, 4, kStream, NT, B>(it, t, nbytes, ahead);
  } else if (lv == 3) {   // streamed: kOpRows8, kOpRows4, or one small piece
    narrow_tile<kKindCopy, 8, kCached, NT, B>(it, t, nbytes, ahead);
  } else if (lv == 2) {
    narrow_tile<kKindCopy, 4, kCached, NT, B>(it, t, nbytes, ahead);
  } else if (lv == 1) {
    if (merge) narrow_tile<kKindCopy, 2, kCached, NT, B>(it, t, nbytes, ahead);
    else narrow_tile<kKindCopy, 2, kStream, NT, B>(it, t, nbytes, ahead);
  } else {
    if (merge) narrow_tile<kKindCopy, 1, kCached, NT, B>(it, t, nbytes, ahead);
    else narrow_tile<kKindCopy, 1, kStream, NT, B>(it, t, nbytes, ahead);
  }
}

// One vector at a time through 64-bit addresses: strided items whose tiles
// span 2 GiB or more of an object (a few bytes of very long rows).
template <int B>
__device__ __forceinline__ void far_tile(const DevItem& it, const DevTile& t, uint32_t nbytes, uint32_t lane) {
  const uint32_t lv = (it.flags >> 4) & 0xfu, kind = it.flags & 0xfu;
  const RowMap rows = row_map(it, uint32_t(t.dst));
  for (uint32_t b = lane << lv; b < nbytes; b += B << lv) {
    uint32_t row, col;
    rows.at(b, row, col);
    const uint64_t q = t.src + row;
    const uint64_t from = it.src + q * it.src_stride + col, to = it.dst + q * it.dst_stride + col;
    const uint64_t half = it.dst2 + q * it.dst2_stride + (col >> 1);
    if (kind == kKindRecast) {
      if (lv == 4) {
        const VecOf<16>::type v = ld_far<16>(from);
        if (it.dst) st_far<16>(to, v);
        st_far<8>(half, to_bf16<4>(v));
      } else {
        const uint32_t v = ld_far<4>(from);
        if (it.dst) st_far<4>(to, v);
        st_far<2>(half, to_bf16<1>(v));
      }
    } else if (lv == 4) {
      st_far<16>(to, kind == kKindZero ? VecOf<16>::type(0) : ld_far<16>(from));
    } else if (lv == 3) {
      st_far<8>(to, kind == kKindZero ? VecOf<8>::type(0) : ld_far<8>(from));
    } else if (lv == 2) {
      st_far<4>(to, kind == kKindZero ? 0u : ld_far<4>(from));
    } else if (lv == 1) {
      st_far<2>(to, kind == kKindZero ? (unsigned short)0 : ld_far<2>(from));
    } else {
      st_far<1>(to, kind == kKindZero ? (unsigned char)0 : ld_far<1>(from));
    }
  }
}

// The tile at each position of the grid.  With `seg` non-zero the list is
// cut into kXcds segments of `seg` tiles and position p takes tile p / kXcds
// of segment p % kXcds: each die walks one contiguous part of the list, and
// of the records.  Positions p, p + stride, ... below n_pos are this
// workgroup's; `stride` is the grid.
template <bool NT, int B, int U>
__device__ __forceinline__ void exec_tiles(const DevItem* __restrict__ items, const DevTile* __restrict__ tiles,
                                           uint32_t n_tiles, uint32_t seg, uint32_t n_pos, uint32_t stride,
                                           uint32_t n_ahead, uint32_t n_items) {
  uint32_t p = blockIdx.x;
  do {
    const uint32_t i = seg ? (p % kXcds) * seg + p / kXcds : p;
    if (i < n_tiles) {
      const DevTile t = tiles[i];
      // made anew for each tile: what a path derives from it would otherwise
      // be computed for all paths before the loop, and held
      uint32_t lane = threadIdx.x;
      asm volatile("" : "+v"(lane));
      const uint32_t op = t.info >> kTileOpBit, nbytes = t.info & kTileBytesMask;
      const Ahead ahead{tiles, i, n_ahead, lane, items, op == kOpCopy ? n_items : t.item, n_items};
      const Region none = region(0, 0);
      if (__builtin_expect(op == kOpCopy, 1)) {
        contiguous_tile<kKindCopy, kThrough, NT, B, U>(Regions{region(t.src, nbytes), region(t.dst, nbytes), none},
                                                       nbytes, ahead);
      } else if (__builtin_expect(op == kOpRows, 1)) {
        const DevItem it = items[t.item];
        rows_tile<kKindCopy, kThrough, NT, B, U>(
            Regions{region(it.src + t.src * it.src_stride, it.src ? kNearBytes : 0),
                    region(it.dst + t.src * it.dst_stride, kNearBytes), none},
            it, uint32_t(t.dst), nbytes, ahead);
      } else if (__builtin_expect(op == kOpRecast, 1)) {
        contiguous_tile<kKindRecast, kThrough, NT, B, U>(recast_regions(items[t.item], t, nbytes), nbytes, ahead);
      } else if (__builtin_expect(op == kOpZero, 1)) {
        contiguous_tile<kKindZero, kThrough, NT, B, U>(Regions{none, region(t.dst, nbytes), none}, nbytes, ahead);
      } else if (__builtin_expect(op == kOpRecastRows, 1)) {
        const DevItem it = items[t.item];
        rows_tile<kKindRecast, kThrough, NT, B, U>(row_regions(it, t.src), it, uint32_t(t.dst), nbytes, ahead);
      } else if (op == kOpCopyStream) {
        contiguous_tile<kKindCopy, kStream, NT, B, U>(Regions{region(t.src, nbytes), region(t.dst, nbytes), none},
                                                      nbytes, ahead);
      } else if (op == kOpRowsStream) {
        const DevItem it = items[t.item];
        rows_tile<kKindCopy, kStream, NT, B, U>(row_regions(it, t.src), it, uint32_t(t.dst), nbytes, ahead);
      } else if (op == kOpRows8) {
        // a body of four vectors in the workgroups of large phases too costs their merged rows 1%
        if (U == 2 && nbytes > B * 16) narrow_tile<kKindCopy, 8, kStream, NT, B, 2 * U>(items[t.item], t, nbytes, ahead);
        else narrow_tile<kKindCopy, 8, kStream, NT, B>(items[t.item], t, nbytes, ahead);
      } else if (op == kOpRows4) {
        narrow_tile<kKindCopy, 4, kStream, NT, B>(items[t.item], t, nbytes, ahead);
      } else if (op == kOpWide) {
        const DevItem it = items[t.item];
        if (it.flags & kItemMerge) wide_tile<kCached, NT, B>(it, t, nbytes, ahead);
        else wide_tile<kStream, NT, B>(it, t, nbytes, ahead);
      } else if (op == kOpNarrow) {
        const DevItem it = items[t.item];
        narrow_forms<NT, B>(it, t, nbytes, ahead);
      } else if (op == kOpRecastRowsPart) {
        const DevItem it = items[t.item];
        const Regions r = row_regions(it, t.src);
        if (it.flags & kItemMerge) rows_tile<kKindRecast, kCached, NT, B, U>(r, it, uint32_t(t.dst), nbytes, ahead);
        else rows_tile<kKindRecast, kStream, NT, B, U>(r, it, uint32_t(t.dst), nbytes, ahead);
      } else if (op == kOpRecastStream) {
        contiguous_tile<kKindRecast, kStream, NT, B, U>(recast_regions(items[t.item], t, nbytes), nbytes, ahead);
      } else if (op == kOpZeroStream) {
        contiguous_tile<kKindZero, kStream, NT, B, U>(Regions{none, region(t.dst, nbytes), none}, nbytes, ahead);
      } else {
        far_tile<B>(items[t.item], t, nbytes, lane);
      }
    }
    p += stride;
  } while (p < n_pos);
}

// Three entry points with one body, so profiles tell the phases apart.  Eight
// waves per SIMD (2048 lanes per compute unit) need at most 64 vector
// registers and, the trap handler's 16 included, 96 scalar ones each: with
// 84 of its own the kernel ran half the waves and lost 15%.
#define SR_COPY_KERNEL(NAME)                                                                                 \
  template <bool NT, int B, int U>                                                                           \
  __global__ __launch_bounds__(B) __attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(8))) void NAME(    \
      const DevItem* __restrict__ items, const DevTile* __restrict__ tiles, uint32_t n_tiles, uint32_t seg,  \
      uint32_t n_pos, uint32_t stride, uint32_t n_ahead, uint32_t n_items) {                                 \
    exec_tiles<NT, B, U>(items, tiles, n_tiles, seg, n_pos, stride, n_ahead, n_items);                       \
  }
SR_COPY_KERNEL(sr_pack_kernel)
SR_COPY_KERNEL(sr_unpack_kernel)
SR_COPY_KERNEL(sr_gather_kernel)
#undef SR_COPY_KERNEL

// The kernels' workgroups: lanes, and 16-byte vectors that a lane holds at
// once.  One vector in each of 1024 lanes is the best for the tiles of a large
// phase; the others are for
//   * tiles of few vectors, whose workgroups cost more to start than to run:
//     256 lanes for a mean of 7 KiB or less (us; 1024 / 512 / 256 lanes:
//     60000 pieces of 1000 bytes 135 / 87 / 46, 4096-byte tiles of 1 GiB
//     744 / 473 / 325, 8192-byte ones 404 / 329 / 340), 512 lanes for 12 KiB
//     or less (pieces of 10000 bytes 88 / 76 / 76; of 14000 77 / 75 / 77;
//     60000 pieces of 1000 bytes among 1 GiB, mean 9 KiB, 425 / 372 / 399);
//   * few tiles, where each compute unit takes a handful in turn and more of
//     them side by side hide the way to a tile's first load: 512 lanes of two
//     vectors up to 5120 tiles (strided, 2624 tiles 18.2 / 15.7 us, 4000
//     24.5 / 21.7, 6000 36.5 / 36.5), and up to 16384 where most are COPY
//     rows, which then are streamed (1024 lanes of one / 512 of two: 8192
//     tiles 50.8 / 49.1, 16384 91.8 / 89.1; contiguous ones 46.9 / 48.8);
//   * grids capped at 512 workgroups or less, the same (1 GiB of columns
//     merged, 64 workgroups 1198 / 1000 us, 256 405 / 370, 512 448 / 421);
//   * tiles of more than one pass: two vectors in each of 1024 lanes (64 KiB
//     tiles, columns merged 381 / 356 us with one / two).
enum Shape { kWide, kSmall, kTiny, kLong };

constexpr uint32_t shape_lanes(Shape s) { return s == kSmall ? 512 : s == kTiny ? 256 : 1024; }

constexpr uint64_t kFewTiles = 5120, kManyTiles = 16384;
constexpr uint32_t kFewBlocks = 512;

// More bytes than kManyTiles whole tiles.
bool large_phase(uint64_t bytes, uint32_t tile_bytes) { return bytes / tile_bytes > kManyTiles; }

// The phase's tiles number more than a few, but not many, and are not small.
bool middling(uint64_t n_recs, uint64_t bytes, uint32_t tile_bytes) {
  return n_recs > kFewTiles && !large_phase(bytes, tile_bytes) && bytes / n_recs > 12 * 1024;
}

// `rows`: the tiles of COPY rows of 512 bytes and more and of a multiple of 16
// (of 16 bytes, 16384 tiles: 117 us with 1024 lanes, 132 with 512), or of 8
// where they are written end to end (9000 tiles, rows of 4104 bytes split off
// 55.6 / 53.2, but merged 56.4 / 56.7, of 1032 merged 57.7 / 61.4), and of
// RECAST into bf16 alone (9000 tiles 43.2 / 38.3).  `recast`: those of RECAST
// with an f32 copy, which count twice as few (4000 tiles 29.3 / 31.2).
Shape pick_shape(uint64_t n_recs, uint64_t bytes, uint64_t rows, uint64_t recast, const sr_plan_options& opt) {
  const uint64_t mean = bytes / n_recs;
  if (mean <= 7 * 1024) return kTiny;
  if (opt.tile_bytes > kPassBytes) return kLong;
  if (mean <= 12 * 1024 || n_recs + recast <= kFewTiles) return kSmall;
  if (opt.max_blocks != 0 && opt.max_blocks <= kFewBlocks) return kSmall;
  return middling(n_recs, bytes, opt.tile_bytes) && 2 * rows > n_recs ? kSmall : kWide;
}

// ------------------------------------------------- device-side plan binding
// The host keeps O(pieces) descriptors and the prefix sum of their tile
// counts; for phases above kHostTableTiles the per-tile table, the per-peer
// buffer offsets and the absolute-address item table are computed on the GPU
// from them:
//   sr_offsets_kernel   per peer: exclusive prefix sum of the 256-byte
//                       rounded payloads of its pieces, in piece order;
//   sr_tile_emit_kernel one workgroup per chunk of an item's tiles writes
//                       their records, bound to the caller's pointers; again
//                       for other pointers.

// Pointer-independent item descriptor (device resident, uploaded once).
enum : uint32_t {
  kRelSrcBuf = 1u << 16,   // source side is a peer buffer at the piece's offset
  kRelDstBuf = 1u << 17,   // destination side is a peer buffer at the piece's offset
  kRelFar = 1u << 18,      // kOpFar
  kRelStream = 1u << 19,   // whole lines are streamed too (stream_whole)
  kRelShiftBit = 20,       // bits 20-24: log2 of the source bytes of a tile record
};

struct alignas(8) DevRel {
  uint64_t src_off;        // byte offset of the region origin in its object
  uint64_t dst_off;
  uint64_t dst2_off;
  uint64_t src_stride;
  uint64_t dst_stride;
  uint64_t dst2_stride;
  uint64_t total;          // source bytes (destination bytes for ZERO)
  uint32_t row_bytes;      // 0 = contiguous
  uint32_t magic;
  uint32_t shifts;
  uint32_t kind;           // bits 0-7 kind, 8-15 element bytes, kRelSrcBuf ... kRelShiftBit
  int32_t src_slot;        // index into the phase's pointer table, -1 = none
  int32_t dst_slot;
  int32_t dst2_slot;
  int32_t piece;           // piece whose buffer offset the buffer side uses
  uint32_t group_size;     // items whose tiles are dealt out row block by row block
  uint32_t group_index;    // this item's place in its group
};
static_assert(sizeof(DevRel) == 96, "DevRel layout");

// Exclusive prefix sum across a workgroup of NT lanes: an inclusive scan
// inside each wave64 by shuffles, then the wave totals through LDS.  Every
// lane of the workgroup must call it (it synchronises).  `total` receives
// the sum over the workgroup.
template <int NT>
__device__ uint64_t block_exclusive_scan(uint64_t v, uint64_t& total) {
  constexpr int kWaves = NT / 64;
  __shared__ uint64_t wave_sum[kWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) wave_sum[wave] = x;
  __syncthreads();
  uint64_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint64_t s = wave_sum[w];
    if (w < wave) before += s;
    all += s;
  }
  __syncthreads();   // wave_sum is reused by the next call
  total = all;
  return before + x - v;
}

constexpr int kSetupBlock = 256;
// Tiles one workgroup of the emit kernel writes at most (16 per lane): a
// large item's tiles are spread over several workgroups.
constexpr uint32_t kEmitTiles = 4096;
// Phases of at most this many tiles set up on the caller's stream even
// while earlier work still runs there: their setup takes a few microseconds
// of GPU time, less than a wait across streams costs the host.
constexpr uint64_t kInlineSetupTiles = 65536;

// Phases of at most this many tiles have their tables written by the host
// and read from its memory at the first launch on new pointers, which saves
// the emit kernel.  Above, the tiles' reads over the host link and the host's
// writes cost more.  A call with new pointers, us, upload and emit / host
// tables (f32 rows of 8 KiB split off): 8 tiles 17.4 / 7.7, 512 17.8 / 9.2,
// 1024 18.8 / 12.9, 2048 24.8 / 21.2, 4096 36.0 / 38.7.  Launches that repeat the pointers
// read device memory, as 2048 tiles take 21.4 from the host's and 14.4 from
// the device's.
constexpr uint64_t kHostTableTiles = 2048;

// `vectors` 16-byte vectors of a table from pinned host memory to the device:
// bound by the host link's latency, one read per lane in flight.
__global__ __launch_bounds__(kSetupBlock) void sr_table_copy_kernel(const unsigned char* __restrict__ from,
                                                                    unsigned char* __restrict__ to,
                                                                    uint32_t vectors) {
  typedef VecOf<16>::type V;
  const uint32_t i = blockIdx.x * kSetupBlock + threadIdx.x;
  if (i < vectors) reinterpret_cast<V*>(to)[i] = reinterpret_cast<const V*>(from)[i];
}

// An empty kernel: launching it loads the library's GPU code (sr_prepare).
__global__ void sr_prepare_kernel() {}

struct EmitChunk {
  uint32_t item;
  uint32_t chunk;   // the item's tiles [chunk * kEmitTiles, (chunk + 1) * kEmitTiles)
};
static_assert(sizeof(EmitChunk) == 8, "EmitChunk layout");

// One workgroup per peer.  peer_begin[p]..peer_begin[p+1] indexes
// peer_list, the peer's pieces in piece order.
__global__ __launch_bounds__(kSetupBlock) void sr_offsets_kernel(
    const uint32_t* __restrict__ peer_begin, const uint32_t* __restrict__ peer_list,
    const uint64_t* __restrict__ payload, uint64_t* __restrict__ offset) {
  const uint32_t b = peer_begin[blockIdx.x];
  const uint32_t e = peer_begin[blockIdx.x + 1];
  uint64_t carry = 0;
  for (uint32_t base = b; base < e; base += kSetupBlock) {
    const uint32_t i = base + threadIdx.x;
    const bool ok = i < e;
    const uint32_t k = ok ? peer_list[i] : 0u;
    const uint64_t v = ok ? (payload[k] + kBufAlign - 1) / kBufAlign * kBufAlign : 0;
    uint64_t total;
    const uint64_t ex = block_exclusive_scan<kSetupBlock>(v, total);
    if (ok) offset[k] = carry + ex;
    carry += total;
  }
}

// Largest power-of-two vector width (<= 16, >= esize) dividing every value
// OR-ed into `acc`.
__host__ __device__ inline uint32_t pick_vb(uint64_t acc, uint32_t esize) {
  uint32_t vb = 16;
  while (vb > esize && (acc & (vb - 1))) vb >>= 1;
  return vb;
}

__host__ __device__ inline uint32_t log2u(uint32_t v) {
  uint32_t l = 0;
  while ((1u << l) < v) ++l;
  return l;
}

// The narrowest rows that move as 16-byte vectors at any alignment rather
// than as aligned vectors of `vb` bytes, by whether the destination is dense.
// Measured on 1 GiB halves of bf16 (vb 2) and u8 (vb 1) rows, TB/s, narrow
// against 16-byte: side by side rows of 66 bytes 3.2 / 3.7-4.0, 514 bytes
// 3.2 / 4.8; dense rows of 202 bytes 4.0 / 3.6, 514 bytes 4.2 / 4.9; u8 side
// by side of 17 bytes 2.0 / 3.1, dense of 33 bytes 2.5 / 2.4, 101 bytes
// 2.5 / 2.7.  Rows that are 4-byte aligned stay narrow at every width (f32
// rows of 2732 bytes, dense: 5.6 / 5.2).
__host__ __device__ inline uint32_t ragged_from(uint32_t vb, bool dense) {
  if (vb == 1) return dense ? 64 : 16;
  if (vb == 2) return dense ? 400 : 64;
  return 0xffffffffu;
}

// Rows of a destination that is not dense leave their lines to be merged
// when they are shorter than this, RECAST with an f32 copy or in single
// elements at any width: f32 rows of 260 bytes streamed 4.4, merged 4.9 TB/s;
// of 800 bytes 5.7 / 5.5; ZERO rows of 192 bytes 2.9 / 3.5, of 400 bytes 4.7 /
// 3.5; RECAST of 800 bytes 5.1 / 6.0, of 16400 bytes 5.7 / 6.0, into bf16 alone
// of 400 bytes 5.8 / 6.0, of 1600 bytes 6.3 / 5.9.
constexpr uint32_t kMergeBelow = 512, kMergeZeroBelow = 384;

// The item of descriptor `h`: its object addresses resolved from `ptrs`,
// the phase's pointer table (source objects, then destination objects),
// and `offset`, the per-piece buffer offsets from sr_offsets_kernel; the
// vector and the op of its tiles.
__host__ __device__ __forceinline__ DevItem bind_item(const DevRel& h, const uint64_t* __restrict__ ptrs,
                                             const uint64_t* __restrict__ offset, uint32_t& op) {
  const uint32_t kind = h.kind & 0xffu;
  const bool contiguous = h.row_bytes == 0;
  const bool far = (h.kind & kRelFar) != 0;
  DevItem d;
  d.src = h.src_slot >= 0 ? ptrs[h.src_slot] + ((h.kind & kRelSrcBuf) ? offset[h.piece] : h.src_off) : 0;
  d.dst = h.dst_slot >= 0 ? ptrs[h.dst_slot] + ((h.kind & kRelDstBuf) ? offset[h.piece] : h.dst_off) : 0;
  d.dst2 = h.dst2_slot >= 0 ? ptrs[h.dst2_slot] + h.dst2_off : 0;
  d.src_stride = h.src_stride;
  d.dst_stride = h.dst_stride;
  d.dst2_stride = h.dst2_stride;
  d.row_bytes = h.row_bytes;
  d.magic = h.magic;
  d.shifts = h.shifts;
  const uint64_t width = contiguous ? h.total : h.row_bytes;
  // the destination's rows lie end to end
  const bool dense = contiguous || ((h.dst_slot < 0 || h.dst_stride == h.row_bytes) &&
                                    (h.dst2_slot < 0 || h.dst2_stride * 2 == h.row_bytes));

  // the widest vector that all addresses and sizes are aligned for (RECAST:
  // four elements, or one), or 16 bytes at any alignment
  uint64_t at = d.src | d.dst | width;
  if (!contiguous) at |= h.src_stride | h.dst_stride;
  uint32_t lv = log2u(pick_vb(at, kind == kKindRecast ? 4 : (h.kind >> 8) & 0xffu));
  if (kind == kKindRecast) {
    const uint64_t half = d.dst2 | (contiguous ? 0 : h.dst2_stride);
    if (lv < 4 || (half & 7)) lv = contiguous && width >= 16 ? 4 : 2;
  } else if (!far && width >= (contiguous || kind == kKindZero ? 16 : ragged_from(1u << lv, dense))) {
    lv = 4;
  }

  // 16-byte vectors into whole lines: of each row, or of a dense destination
  uint64_t line = d.dst | d.dst2;
  if (!dense) {
    line |= h.row_bytes | h.dst_stride | h.dst2_stride;
    if (kind == kKindRecast) line |= h.row_bytes >> 1;
  }
  const bool whole = (line & 63) == 0, rows16 = !contiguous && h.row_bytes % 16 == 0;
  const bool merge = !dense && (kind == kKindRecast ? lv < 4 || h.dst_slot >= 0 || h.row_bytes < kMergeBelow
                                                    : h.row_bytes < (kind == kKindZero ? kMergeZeroBelow : kMergeBelow));
  const bool through = whole && !(h.kind & kRelStream);
  if (far) op = kOpFar;
  else if (lv < 4 && (contiguous || merge || kind == kKindRecast || lv < 2)) op = kOpNarrow;
  else if (lv < 4) op = lv == 3 ? kOpRows8 : kOpRows4;
  else if (contiguous && through) op = kind == kKindCopy ? kOpCopy : kind == kKindZero ? kOpZero : kOpRecast;
  else if (contiguous) op = kind == kKindCopy ? kOpCopyStream : kind == kKindZero ? kOpZeroStream : kOpRecastStream;
  else if (kind == kKindRecast) op = through ? kOpRecastRows : kOpRecastRowsPart;
  else if (rows16 && through) op = kOpRows;
  else if (rows16 && (whole || !merge)) op = kOpRowsStream;
  else op = kOpWide;
  d.flags = kind | (lv << 4) | (merge && !whole ? kItemMerge : 0u);
  return d;
}

// Tile `j` of item `k` with descriptor `h`, bound as `item`.
__host__ __device__ __forceinline__ DevTile tile_record(const DevItem& item, const DevRel& h, uint32_t k, uint32_t op,
                                                        uint64_t j) {
  const uint32_t width = item.row_bytes, tile_shift = (h.kind >> kRelShiftBit) & 0x1fu;
  const uint64_t total = h.total;
  uint64_t start = j << tile_shift;
  uint64_t n = total - start < (uint64_t(1) << tile_shift) ? total - start : (uint64_t(1) << tile_shift);
  if (width == 0 && total >= 16 && n < 16) {   // a whole vector, from the tile before
    start -= 16 - n;
    n = 16;
  }
  DevTile t;
  t.item = k;
  t.info = op << kTileOpBit | uint32_t(n);
  if (width == 0) {
    t.src = item.src + start;
    t.dst = item.dst ? item.dst + start : 0;
  } else {
    const uint64_t row = start / width;
    t.src = row;
    t.dst = start - row * width;
  }
  return t;
}

// One workgroup per emit chunk -- up to kEmitTiles consecutive tiles of one
// item (chunks[c] = {item, chunk index}; every item has at least one) --
// writes those tiles' records, in list order (tile_base[k] = tiles of items
// 0..k-1, computed with the descriptors on the host), bound to the pointer
// table `ptrs` (and the buffer offsets `offset`).  Lane 0 of an item's first
// chunk also writes the bound item.
__global__ __launch_bounds__(kSetupBlock) void sr_tile_emit_kernel(
    const DevRel* __restrict__ rel, const uint64_t* __restrict__ tile_base, const EmitChunk* __restrict__ chunks,
    uint32_t n_chunks, DevTile* __restrict__ tiles, const uint64_t* __restrict__ ptrs,
    const uint64_t* __restrict__ offset, DevItem* __restrict__ items) {
  for (uint32_t c = blockIdx.x; c < n_chunks; c += gridDim.x) {
    const uint32_t k = chunks[c].item;
    const uint64_t j0 = uint64_t(chunks[c].chunk) * kEmitTiles;
    const uint64_t cnt = tile_base[k + 1] - tile_base[k];
    // Items of a group have equal tile counts; tile j of member m goes to
    // group_start + j*M + m, so the members' tiles over the same rows are
    // adjacent in the list.
    const uint64_t gm = rel[k].group_index;
    const uint64_t gsize = rel[k].group_size;
    const uint64_t b = tile_base[k] - gm * cnt + gm;
    uint32_t op;
    const DevItem item = bind_item(rel[k], ptrs, offset, op);
    if (j0 == 0 && threadIdx.x == 0) items[k] = item;
    const uint64_t j1 = cnt < j0 + kEmitTiles ? cnt : j0 + kEmitTiles;
    for (uint64_t j = j0 + threadIdx.x; j < j1; j += kSetupBlock) {
      tiles[b + j * gsize] = tile_record(item, rel[k], k, op, j);
    }
  }
}

// ----------------------------------------------------------- host structures

// Pointer-independent description of one item of a phase.
struct HostItem {
  uint32_t kind;
  int32_t src_slot;       // pack: src tensor slot; unpack: peer index
  int32_t dst_slot;       // pack: peer index; unpack: dst slot (-1: none)
  int32_t dst2_slot;      // unpack RECAST: bf16 slot, else -1
  uint64_t src_off;       // byte offset of region origin in the source object
  uint64_t dst_off;
  uint64_t dst2_off;
  uint64_t src_stride;
  uint64_t dst_stride;
  uint64_t dst2_stride;
  uint64_t rows;
  uint64_t row_bytes;     // source bytes per row (dst bytes for ZERO)
  bool contiguous;        // collapsed to one row of rows*row_bytes bytes
  uint32_t esize;         // element bytes of the source (dst for ZERO)
  int32_t piece;          // the sr_piece this item moves
};

struct Phase {
  std::vector<HostItem> items;          // in piece order while the plan is built
  std::vector<DevRel> rel;              // items in dispatch (tile) order
  std::vector<uint64_t> tile_base;      // records of rel[0..k-1]; tile_base[n] = n_recs
  std::vector<EmitChunk> emit_chunks;   // the emit kernel's work: every item's tiles in chunks
  uint64_t n_tiles = 0;                 // as the plan reports them
  uint64_t n_recs = 0;                  // tile records, one per workgroup: at most n_tiles
  uint64_t rec_bytes = 0;               // their source bytes
  uint32_t n_src_base = 0;              // pointer table: sources, then destinations
  uint32_t n_dst_base = 0;
  std::vector<uint64_t> obj_bytes;      // per pointer-table slot: object size
  std::vector<uint8_t> obj_use;         // per slot: 1 read, 2 written (0: unused)
  const char* src_name = "src_ptrs";    // caller-side names of the two tables
  const char* dst_name = "dst_ptrs";
  bool interleave = false;
  Shape shape = kWide;
  uint64_t bytes_read = 0;
  uint64_t bytes_written = 0;
  // device state, created on first use: one device allocation carved into
  // the tables, one pinned host buffer for their uploads
  bool ready = false;
  void* d_mem = nullptr;
  size_t d_cap = 0;                     // bytes of d_mem / h_staging as allocated
  size_t h_cap = 0;
  DevRel* d_rel = nullptr;              // uploaded: descriptors, tile prefix, pointer table
  uint64_t* d_tile_base = nullptr;
  uint64_t* d_ptrs = nullptr;
  EmitChunk* d_chunks = nullptr;
  DevItem* d_items = nullptr;           // built on the device
  DevTile* d_tiles = nullptr;
  unsigned char* h_staging = nullptr;   // pinned: the uploaded part, in the same layout
  uint64_t* h_ptrs = nullptr;           // the pointer-table part of h_staging
  std::vector<uint64_t> bound;          // pointer table of the last bind
  bool bound_valid = false;
  hipEvent_t ev_setup = nullptr;        // tile table, offsets and the first bind written
  hipEvent_t ev_staging = nullptr;      // a later bind done (its copy out of h_staging too)
  hipEvent_t ev_kernel = nullptr;       // last copy kernel reading the device's tables, and all before it
  hipEvent_t ev_bound = nullptr;        // the latest bind: ev_setup, ev_staging or ev_kernel (not owned)
  hipEvent_t ev_tail = nullptr;         // the latest bind or copy kernel (not owned)
  // small phases (kHostTableTiles): two pinned tables, written in turn, and a
  // device copy of the latest.  Memory of their own: a first use on a
  // capturing stream takes the blocks above, of other sizes, and may fail
  // after it did.
  unsigned char* h_tables = nullptr;
  unsigned char* d_tables = nullptr;
  size_t h_tables_cap = 0;
  size_t d_tables_cap = 0;
  int slot = 0;
  hipEvent_t ev_slot[2] = {};           // last kernel reading the table
  bool on_device = false;               // the tables are in d_tables too
};

}  // namespace

struct sr_plan {
  std::vector<sr_tensor> src;
  std::vector<sr_tensor> dst;
  std::vector<sr_piece> pieces;
  std::vector<uint64_t> piece_offset;   // buffer offset, UINT64_MAX for ZERO
  std::vector<uint64_t> peer_bytes;
  int32_t n_peers = 0;
  sr_plan_options opt{};
  Phase pack;
  Phase unpack;
  Phase gather;   // direct source -> destination, no buffers
  // alignment each gather pointer must satisfy: its element size; 0 = the
  // slot is not used by the gather
  std::vector<uint32_t> gather_src_align, gather_dst_align;
  int device = -1;
  // Buffer offsets recomputed on the device: per-peer piece lists (CSR).
  std::vector<uint32_t> peer_begin;
  std::vector<uint32_t> peer_list;
  std::vector<uint64_t> payload;        // per piece, 0 for ZERO
  bool offsets_ready = false;
  void* d_offmem = nullptr;             // carved: offsets, payloads, peer lists
  unsigned char* h_offmem = nullptr;    // pinned upload of payloads and peer lists
  size_t d_offcap = 0;
  size_t h_offcap = 0;
  uint64_t* d_offset = nullptr;
  uint32_t* d_peer_begin = nullptr;
  uint32_t* d_peer_list = nullptr;
  uint64_t* d_payload = nullptr;
  hipEvent_t ev_offsets = nullptr;
};

namespace sr_internal {
PlanView plan_view(const sr_plan* p) {
  return PlanView{p->src.data(), p->src.size(), p->pieces.data(), p->pieces.size(), p->piece_offset.data(),
                  p->peer_bytes.data(), p->n_peers, p->peer_begin.data(), p->peer_list.data()};
}
}  // namespace sr_internal

namespace {

int check_tensor(const sr_tensor& t, const char* what, int32_t idx) {
  if (t.reserved != 0) return fail(SR_EINVAL, "%s[%d]: reserved field must be 0", what, idx);
  const int es = dtype_size(t.dtype);
  if (es == 0) return fail(SR_EINVAL, "%s[%d]: unknown dtype %d", what, idx, t.dtype);
  if (t.rows == 0 || t.cols == 0)
    return fail(SR_EINVAL, "%s[%d]: empty tensor [%llu, %llu]", what, idx,
                (unsigned long long)t.rows, (unsigned long long)t.cols);
  const uint64_t lim = uint64_t(1) << 62;
  uint64_t n, bytes;
  if (__builtin_mul_overflow(t.rows, t.cols, &n) || __builtin_mul_overflow(n, uint64_t(es), &bytes) || bytes > lim)
    return fail(SR_EINVAL, "%s[%d]: tensor too large", what, idx);
  return SR_OK;
}

int check_region(const sr_tensor& t, uint64_t r0, uint64_t c0, uint64_t rows, uint64_t cols,
                 const char* what, int32_t piece) {
  if (r0 > t.rows || rows > t.rows - r0 || c0 > t.cols || cols > t.cols - c0)
    return fail(SR_EBOUNDS,
                "piece %d: %s region rows [%llu,+%llu) cols [%llu,+%llu) outside tensor [%llu, %llu]",
                piece, what, (unsigned long long)r0, (unsigned long long)rows,
                (unsigned long long)c0, (unsigned long long)cols, (unsigned long long)t.rows,
                (unsigned long long)t.cols);
  return SR_OK;
}

struct Box {
  uint64_t r0, r1, c0, c1;
  int32_t piece;
  int32_t slot;   // destination slot written
};

// Every destination slot must be written exactly once: boxes pairwise
// disjoint and their areas summing to the slot's area.  `boxes` holds the
// regions of all slots (any order; sorted here by slot, row, column).
int check_coverage(std::vector<Box>& boxes, const std::vector<sr_tensor>& dst) {
  std::sort(boxes.begin(), boxes.end(), [](const Box& x, const Box& y) {
    if (x.slot != y.slot) return x.slot < y.slot;
    return x.r0 != y.r0 ? x.r0 < y.r0 : x.c0 < y.c0;
  });
  size_t at = 0;
  for (size_t s = 0; s < dst.size(); ++s) {
    size_t end = at;
    while (end < boxes.size() && boxes[end].slot == int32_t(s)) ++end;
    unsigned __int128 area = 0;
    for (size_t i = at; i < end; ++i) {
      const Box& bi = boxes[i];
      area += (unsigned __int128)(bi.r1 - bi.r0) * (bi.c1 - bi.c0);
      for (size_t j = i + 1; j < end && boxes[j].r0 < bi.r1; ++j) {
        if (boxes[j].c0 < bi.c1 && bi.c0 < boxes[j].c1)
          return fail(SR_EOVERLAP, "dst[%zu]: pieces %d and %d write overlapping regions", s, bi.piece,
                      boxes[j].piece);
      }
    }
    const unsigned __int128 full = (unsigned __int128)dst[s].rows * dst[s].cols;
    if (area != full)
      return fail(SR_EOVERLAP, "dst[%zu]: pieces cover %llu of %llu elements", s,
                  (unsigned long long)area, (unsigned long long)full);
    at = end;
  }
  return SR_OK;
}

// Device descriptors of a phase, in `order`.  Pointer-table slots: sources
// first, then destinations (offset by n_src_base).  `buf_src` / `buf_dst`
// mark the side that is a peer buffer (its address is the buffer base plus
// the piece's offset, computed on the device).
//
// With `row_groups`, runs of consecutive strided items that sit side by side
// on the ordering side (the source for pack, the destination otherwise:
// same tensor, rows, row width and stride, each starting where the previous
// one's rows end) form a group whose tiles are dealt out row block by row
// block.  A destination row assembled from several pieces (a dim -1 `cat`)
// is then written by adjacent tiles instead of once per piece, far apart in
// time, so each DRAM page is opened once rather than once per piece.
// Tile size reduction of an item (log2): RECAST items writing both copies.
uint32_t tile_reduce(const HostItem& h) {
  return (h.kind == kKindRecast && h.dst_slot >= 0) ? kRecastTileShift : 0;
}

// Source bytes of a tile record: what a workgroup moves in one pass, or
// tile_bytes where that is more; for RECAST with an f32 copy the tile as plans
// count it (16 MiB tiles of such rows: 911 us with twice as much, 692 so).
// In phases that are `large`, two passes for
//   * RECAST into bf16 alone, which moves 1.5 x its source bytes, too little
//     for a workgroup's start (rows of 16 KiB split off 139 us with one, 123
//     with two; merged 278 / 244; rows of 2732 bytes merged 359 / 285);
//   * COPY rows that only 8-byte vectors divide, of 4 KiB and more written end
//     to end (1 GiB of rows of 4104 bytes split off 375 us with one, 369 with
//     two; of 1032 bytes 385 / 413) and of 16 KiB and more otherwise (of
//     4104 bytes merged 368 / 374, of 32776 bytes 366 / 355).
uint32_t record_bytes(const HostItem& h, uint32_t tile_bytes, bool large) {
  if (large && tile_bytes <= kPassBytes) {
    if (h.kind == kKindRecast && h.dst_slot < 0) return tile_bytes * 2;
    if (h.kind == kKindCopy && !h.contiguous && h.row_bytes >= (h.dst_stride == h.row_bytes ? 4096 : 16384) &&
        ((h.row_bytes | h.src_stride | h.dst_stride) & 15) == 8)
      return tile_bytes * 2;
  }
  return std::max(tile_bytes >> tile_reduce(h), std::min(tile_bytes, kPassBytes));
}

// Whether a tile of a strided item may span 2 GiB or more of an object: its
// rows are then addressed with 64-bit offsets.
bool spans_far(const HostItem& h, uint32_t bytes) {
  const uint64_t rows = std::min<uint64_t>(h.rows, (uint64_t(bytes) + h.row_bytes - 2) / h.row_bytes + 1);
  const uint64_t stride = std::max({h.src_stride, h.dst_stride, h.dst2_stride});
  return stride >= kNearBytes || rows * stride + h.row_bytes > kNearBytes;
}

// Whether an item's whole lines are streamed rather than written through the
// L2 (Policy).  ZERO rows always are (1 GiB of rows of 1024 bytes 166 us,
// through 201).  Others written through are faster in large phases and in
// those of few tiles (us, through / streamed: columns merged, 1500 tiles
// 9.4 / 13.1, 40000 209 / 213; flat, 40000 tiles 200 / 203), but not
//   * between, where much of the phase fits the memory-side cache, for RECAST
//     and rows of 512 bytes and more (columns merged, 6000 tiles 36.5 / 35.7, 9000 53.2 / 51.6,
//     20000 108.7 / 108.8; RECAST, merged, 6000 tiles 46.2 / 43.2, 40000
//     264.8 / 267.1);
//   * into rows that the launch does not write side by side from end to end
//     (a band of wider rows, 9000 tiles 58.5 / 52.1, 80000 476 / 428);
//   * where a workgroup goes on to other tiles and so waits for its stores:
//     contiguous pieces under a capped grid or in tiles of several passes
//     (1 GiB, 64 workgroups 1026 / 934, 1 MiB tiles 405 / 400).
bool stream_whole(const HostItem& h, uint32_t group_size, const Phase& ph, const sr_plan_options& opt) {
  if (h.kind == kKindZero) return !h.contiguous;
  if (h.kind == kKindRecast) return middling(ph.n_recs, ph.rec_bytes, opt.tile_bytes);
  const bool loops = opt.tile_bytes > kPassBytes || (opt.max_blocks != 0 && opt.max_blocks <= kFewBlocks);
  if (h.contiguous && loops) return true;
  if (h.contiguous || ph.n_recs <= kFewTiles) return false;
  const bool side_by_side = h.dst_stride == h.row_bytes || h.dst_stride == h.row_bytes * group_size;
  return !side_by_side || (h.row_bytes >= 512 && middling(ph.n_recs, ph.rec_bytes, opt.tile_bytes));
}

void build_rel(Phase& ph, const std::vector<uint32_t>& order, const sr_plan_options& opt, bool buf_src,
               bool buf_dst, bool group_by_src) {
  const uint32_t tile_bytes = opt.tile_bytes;
  const bool row_groups = !(opt.flags & SR_OPT_NO_ROW_GROUPS);
  ph.rel.clear();
  ph.rel.reserve(order.size());
  ph.tile_base.clear();
  ph.tile_base.reserve(order.size() + 1);
  ph.n_tiles = ph.n_recs = ph.rec_bytes = 0;
  uint64_t row_recs = 0, recast_recs = 0, all_bytes = 0;
  for (const HostItem& h : ph.items) all_bytes += h.rows * h.row_bytes;
  const bool large = large_phase(all_bytes, tile_bytes);
  for (uint32_t k : order) {
    ph.tile_base.push_back(ph.n_recs);
    const HostItem& h = ph.items[k];
    DevRel r{};
    r.src_off = h.src_off;
    r.dst_off = h.dst_off;
    r.dst2_off = h.dst2_off;
    r.src_stride = h.src_stride;
    r.dst_stride = h.dst_stride;
    r.dst2_stride = h.dst2_stride;
    r.total = h.rows * h.row_bytes;
    if (h.contiguous) {
      r.row_bytes = 0;
    } else {
      r.row_bytes = uint32_t(h.row_bytes);
      const DivMagic m = div_magic(uint32_t(h.row_bytes));
      r.magic = m.m;
      r.shifts = m.s1 | (m.s2 << 8);
    }
    r.kind = h.kind | (h.esize << 8);
    if (buf_src && h.src_slot >= 0) r.kind |= kRelSrcBuf;
    if (buf_dst && h.dst_slot >= 0) r.kind |= kRelDstBuf;
    const uint32_t rec_bytes = record_bytes(h, tile_bytes, large);
    r.kind |= log2u(rec_bytes) << kRelShiftBit;
    if (!h.contiguous && spans_far(h, rec_bytes)) r.kind |= kRelFar;
    r.src_slot = h.src_slot;
    r.dst_slot = h.dst_slot >= 0 ? int32_t(ph.n_src_base) + h.dst_slot : -1;
    r.dst2_slot = h.dst2_slot >= 0 ? int32_t(ph.n_src_base) + h.dst2_slot : -1;
    ph.obj_use.resize(size_t(ph.n_src_base) + ph.n_dst_base, 0);
    if (r.src_slot >= 0) ph.obj_use[r.src_slot] |= 1;
    if (r.dst_slot >= 0) ph.obj_use[r.dst_slot] |= 2;
    if (r.dst2_slot >= 0) ph.obj_use[r.dst2_slot] |= 2;
    r.piece = h.piece;
    r.group_size = 1;
    r.group_index = 0;
    ph.rel.push_back(r);
    const uint64_t item_tile = uint64_t(tile_bytes) >> tile_reduce(h);
    ph.n_tiles += (r.total + item_tile - 1) / item_tile;
    const uint64_t recs = (r.total + rec_bytes - 1) / rec_bytes;
    const bool half_only = h.kind == kKindRecast && h.dst_slot < 0;
    const bool rows = !h.contiguous && h.kind == kKindCopy && h.row_bytes >= 512 &&
                      h.row_bytes % (h.dst_stride == h.row_bytes ? 8 : 16) == 0;
    if (half_only || rows) row_recs += recs;
    else if (h.kind == kKindRecast) recast_recs += recs;
    ph.n_recs += recs;
    ph.rec_bytes += r.total;
  }
  ph.tile_base.push_back(ph.n_recs);
  if (ph.n_recs > 0) ph.shape = pick_shape(ph.n_recs, ph.rec_bytes, row_recs, recast_recs, opt);
  ph.emit_chunks.clear();
  for (size_t k = 0; k < ph.rel.size(); ++k) {
    const uint64_t cnt = ph.tile_base[k + 1] - ph.tile_base[k];
    for (uint64_t c = 0; c * kEmitTiles < cnt; ++c) ph.emit_chunks.push_back(EmitChunk{uint32_t(k), uint32_t(c)});
  }
  struct Side {
    int64_t slot;
    uint64_t off, stride, width;
  };
  auto side = [&](const HostItem& h) -> Side {
    if (group_by_src) return {h.src_slot, h.src_off, h.src_stride, h.row_bytes};
    if (h.dst_slot >= 0) return {h.dst_slot, h.dst_off, h.dst_stride, h.row_bytes};
    return {h.dst2_slot, h.dst2_off, h.dst2_stride, h.row_bytes / 2};
  };
  size_t first = 0;
  for (size_t i = 1; i <= order.size(); ++i) {
    bool chain = false;
    if (row_groups && i < order.size()) {
      const HostItem& a = ph.items[order[i - 1]];
      const HostItem& b = ph.items[order[i]];
      const Side sa = side(a), sb = side(b);
      chain = !a.contiguous && !b.contiguous && a.kind == b.kind && a.rows == b.rows &&
              a.row_bytes == b.row_bytes && record_bytes(a, tile_bytes, large) == record_bytes(b, tile_bytes, large) && sa.slot >= 0 && sa.slot == sb.slot &&
              sa.stride == sb.stride && sb.off == sa.off + sa.width;
    }
    if (!chain) {
      const uint32_t m = uint32_t(i - first);
      for (size_t g = first; g < i; ++g) {
        ph.rel[g].group_size = m;
        ph.rel[g].group_index = uint32_t(g - first);
        if (stream_whole(ph.items[order[g]], m, ph, opt)) ph.rel[g].kind |= kRelStream;
      }
      first = i;
    }
  }
}

// Order a phase's items by the tensor address they start at: the source
// side for pack, the destination side for unpack.  Pieces of one tensor then
// run next to each other (tiles are generated in this order).
std::vector<uint32_t> item_order(const Phase& ph, bool by_src) {
  struct Key {
    int64_t slot;
    uint64_t off;
    uint32_t idx;
  };
  std::vector<Key> keys(ph.items.size());
  for (uint32_t i = 0; i < ph.items.size(); ++i) {
    const HostItem& it = ph.items[i];
    if (by_src) keys[i] = {it.src_slot, it.src_off, i};
    else if (it.dst_slot >= 0) keys[i] = {it.dst_slot, it.dst_off, i};
    else keys[i] = {it.dst2_slot, it.dst2_off * 2, i};
  }
  std::stable_sort(keys.begin(), keys.end(), [](const Key& x, const Key& y) {
    return x.slot != y.slot ? x.slot < y.slot : x.off < y.off;
  });
  std::vector<uint32_t> order(keys.size());
  for (size_t i = 0; i < keys.size(); ++i) order[i] = keys[i].idx;
  return order;
}

// ---------------------------------------------------------------- table memory
//
// One drop-in call builds and destroys several short-lived plans.  Their
// table memory (a device block and a pinned block per phase, one of each for
// the buffer offsets) and their events are kept for reuse instead of being
// freed: each allocation or free costs tens of microseconds on the host and
// hipFree synchronizes the device, and the last launch group of a call waits
// for them.  Blocks come in power-of-two sizes (at least 64 KiB) so plans of
// different sizes share them; at most kCacheDeviceBytes / kCacheHostBytes
// stay cached per process and the rest is freed as before.  A block goes back
// only after the events of the launches that used it have completed.
constexpr size_t kCacheDeviceBytes = size_t(256) << 20;
constexpr size_t kCacheHostBytes = size_t(64) << 20;
constexpr size_t kCacheEvents = 256;

size_t block_class(size_t bytes) {
  size_t c = size_t(64) << 10;
  while (c < bytes) c <<= 1;
  return c;
}

class TableCache {
 public:
  int get(bool pinned, int device, size_t bytes, void** out, size_t* cap) {
    const size_t want = block_class(bytes);
    {
      std::lock_guard<std::mutex> lock(mu_);
      std::vector<Block>& list = pinned ? host_ : dev_;
      for (size_t i = 0; i < list.size(); ++i)
        if (list[i].device == device && list[i].bytes == want) {
          *out = list[i].p;
          *cap = want;
          (pinned ? host_bytes_ : dev_bytes_) -= want;
          list[i] = list.back();
          list.pop_back();
          return SR_OK;
        }
    }
    // coherent: kernels read what the host wrote last, from its memory
    if (pinned) SR_HIP_TRY(hipHostMalloc(out, want, hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent));
    else SR_HIP_TRY(hipMalloc(out, want));
    *cap = want;
    return SR_OK;
  }

  void put(bool pinned, int device, void* p, size_t cap) {
    if (!p) return;
    {
      std::lock_guard<std::mutex> lock(mu_);
      size_t& held = pinned ? host_bytes_ : dev_bytes_;
      if (held + cap <= (pinned ? kCacheHostBytes : kCacheDeviceBytes)) {
        (pinned ? host_ : dev_).push_back(Block{p, cap, device});
        held += cap;
        return;
      }
    }
    if (pinned) (void)hipHostFree(p);
    else (void)hipFree(p);
  }

  // Events are created on the current device, which must be `device`.
  int get_event(int device, hipEvent_t* ev) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      for (size_t i = events_.size(); i-- > 0;)
        if (events_[i].first == device) {
          *ev = events_[i].second;
          events_.erase(events_.begin() + i);
          return SR_OK;
        }
    }
    SR_HIP_TRY(hipEventCreateWithFlags(ev, hipEventDisableTiming));
    return SR_OK;
  }

  // One stream per device for the first-use setup of plans (table uploads,
  // tile scan/emit, first bind): default priority, non-blocking, kept for
  // the process.  It lets a launch group's setup run while the previous
  // group's copy kernel still occupies the caller's stream.
  int setup_stream(int device, hipStream_t* out) {
    std::lock_guard<std::mutex> lock(mu_);
    for (const auto& ds : streams_)
      if (ds.first == device) {
        *out = ds.second;
        return SR_OK;
      }
    hipStream_t s = nullptr;
    SR_HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    streams_.emplace_back(device, s);
    *out = s;
    return SR_OK;
  }

  void put_event(int device, hipEvent_t ev) {
    if (!ev) return;
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (events_.size() < kCacheEvents) {
        events_.emplace_back(device, ev);
        return;
      }
    }
    (void)hipEventDestroy(ev);
  }

 private:
  struct Block {
    void* p;
    size_t bytes;
    int device;
  };
  std::mutex mu_;
  std::vector<Block> dev_, host_;
  std::vector<std::pair<int, hipEvent_t>> events_;
  std::vector<std::pair<int, hipStream_t>> streams_;
  size_t dev_bytes_ = 0, host_bytes_ = 0;
};

// Never destroyed: cached blocks live until the process exits, so no HIP call
// runs from a static destructor after the runtime may have shut down.
TableCache& table_cache() {
  static TableCache* cache = new TableCache();
  return *cache;
}

int ensure_device(sr_plan* p) {
  int dev = -1;
  SR_HIP_TRY(hipGetDevice(&dev));
  if (p->device < 0) {
    p->device = dev;
  } else if (p->device != dev) {
    return fail(SR_EINVAL, "plan was first used on device %d, current device is %d", p->device, dev);
  }
  return SR_OK;
}

enum PhaseKind { kPack, kUnpack, kGather };

// Next 256-byte aligned offset for a carved sub-buffer of `bytes`.
size_t carve(size_t& end, size_t bytes) {
  const size_t at = (end + 255) & ~size_t(255);
  end = at + bytes;
  return at;
}

// Per-peer buffer offsets on the device (shared by pack and unpack).  The
// inputs go up asynchronously on `stream` from pinned memory, so the call
// never waits for earlier work on the stream.
int setup_offsets(sr_plan* p, hipStream_t stream) {
  if (p->offsets_ready) return SR_OK;
  int rc;
  if (!p->ev_offsets && (rc = table_cache().get_event(p->device, &p->ev_offsets)) != SR_OK) return rc;
  if (p->n_peers > 0 && !p->peer_list.empty()) {
    const size_t np = p->pieces.size();
    size_t in_end = 0;   // layout of the uploaded part: payloads, peer_begin, peer_list
    const size_t o_pay = carve(in_end, np * sizeof(uint64_t));
    const size_t o_beg = carve(in_end, p->peer_begin.size() * sizeof(uint32_t));
    const size_t o_lst = carve(in_end, p->peer_list.size() * sizeof(uint32_t));
    size_t dev_end = in_end;
    const size_t o_off = carve(dev_end, np * sizeof(uint64_t));
    // allocations survive a failed attempt and are reused by the retry
    if (!p->d_offmem && (rc = table_cache().get(false, p->device, dev_end, &p->d_offmem, &p->d_offcap)) != SR_OK)
      return rc;
    if (!p->h_offmem &&
        (rc = table_cache().get(true, p->device, in_end, reinterpret_cast<void**>(&p->h_offmem),
                                &p->h_offcap)) != SR_OK)
      return rc;
    unsigned char* d = static_cast<unsigned char*>(p->d_offmem);
    p->d_payload = reinterpret_cast<uint64_t*>(d + o_pay);
    p->d_peer_begin = reinterpret_cast<uint32_t*>(d + o_beg);
    p->d_peer_list = reinterpret_cast<uint32_t*>(d + o_lst);
    p->d_offset = reinterpret_cast<uint64_t*>(d + o_off);
    std::memcpy(p->h_offmem + o_pay, p->payload.data(), np * sizeof(uint64_t));
    std::memcpy(p->h_offmem + o_beg, p->peer_begin.data(), p->peer_begin.size() * sizeof(uint32_t));
    std::memcpy(p->h_offmem + o_lst, p->peer_list.data(), p->peer_list.size() * sizeof(uint32_t));
    SR_HIP_TRY(hipMemcpyAsync(p->d_offmem, p->h_offmem, in_end, hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(sr_offsets_kernel, dim3(uint32_t(p->n_peers)), dim3(kSetupBlock), 0, stream,
                       p->d_peer_begin, p->d_peer_list, p->d_payload, p->d_offset);
    SR_HIP_TRY(hipGetLastError());
  }
  SR_HIP_TRY(hipEventRecord(p->ev_offsets, stream));
  p->offsets_ready = true;
  return SR_OK;
}

// The tile and item tables of a phase, from its descriptors and the pointer
// table, all on the device.
int emit_tables(sr_plan* p, Phase& ph, hipStream_t stream) {
  const uint32_t n_chunks = uint32_t(ph.emit_chunks.size());
  hipLaunchKernelGGL(sr_tile_emit_kernel, dim3(std::min<uint32_t>(n_chunks, 65535u)), dim3(kSetupBlock), 0, stream,
                     ph.d_rel, ph.d_tile_base, ph.d_chunks, n_chunks, ph.d_tiles, ph.d_ptrs, p->d_offset, ph.d_items);
  SR_HIP_TRY(hipGetLastError());
  return SR_OK;
}

// First use of a phase: its descriptors, tile prefix and pointer table go
// up in one copy from pinned memory, then one kernel builds the tile table
// and binds the items to `ptrs`, stream-ordered on `stream`.  With
// `mark`, ev_setup marks completion (for a copy kernel on another stream);
// else the phase's next copy kernel follows on `stream` and its ev_kernel
// stands for the bind.
int setup_phase(sr_plan* p, Phase& ph, bool needs_offsets, const std::vector<uint64_t>& ptrs,
                hipStream_t stream, bool mark) {
  if (ph.ready) return SR_OK;
  TableCache& cache = table_cache();
  int rc;
  if (mark && !ph.ev_setup && (rc = cache.get_event(p->device, &ph.ev_setup)) != SR_OK) return rc;
  if (!ph.ev_kernel && (rc = cache.get_event(p->device, &ph.ev_kernel)) != SR_OK) return rc;
  const uint32_t n = uint32_t(ph.rel.size());
  if (n > 0) {
    const size_t nptr = std::max<size_t>(1, size_t(ph.n_src_base) + ph.n_dst_base);
    size_t end = 0;   // the first three are uploaded (pinned staging, same layout)
    const size_t o_rel = carve(end, n * sizeof(DevRel));
    const size_t o_base = carve(end, (size_t(n) + 1) * sizeof(uint64_t));
    const size_t o_chunk = carve(end, ph.emit_chunks.size() * sizeof(EmitChunk));
    const size_t o_ptr = carve(end, nptr * sizeof(uint64_t));
    const size_t up_end = o_ptr + nptr * sizeof(uint64_t);
    const size_t o_items = carve(end, n * sizeof(DevItem));
    const size_t o_tiles = carve(end, ph.n_recs * sizeof(DevTile));
    // allocations survive a failed attempt and are reused by the retry
    if (!ph.d_mem && (rc = cache.get(false, p->device, end, &ph.d_mem, &ph.d_cap)) != SR_OK) return rc;
    if (!ph.h_staging &&
        (rc = cache.get(true, p->device, up_end, reinterpret_cast<void**>(&ph.h_staging), &ph.h_cap)) != SR_OK)
      return rc;
    unsigned char* d = static_cast<unsigned char*>(ph.d_mem);
    ph.d_rel = reinterpret_cast<DevRel*>(d + o_rel);
    ph.d_tile_base = reinterpret_cast<uint64_t*>(d + o_base);
    ph.d_ptrs = reinterpret_cast<uint64_t*>(d + o_ptr);
    ph.d_chunks = reinterpret_cast<EmitChunk*>(d + o_chunk);
    ph.d_items = reinterpret_cast<DevItem*>(d + o_items);
    ph.d_tiles = reinterpret_cast<DevTile*>(d + o_tiles);
    ph.h_ptrs = reinterpret_cast<uint64_t*>(ph.h_staging + o_ptr);
    std::memcpy(ph.h_staging + o_rel, ph.rel.data(), n * sizeof(DevRel));
    std::memcpy(ph.h_staging + o_base, ph.tile_base.data(), (size_t(n) + 1) * sizeof(uint64_t));
    std::memcpy(ph.h_staging + o_chunk, ph.emit_chunks.data(), ph.emit_chunks.size() * sizeof(EmitChunk));
    std::memcpy(ph.h_ptrs, ptrs.data(), ptrs.size() * sizeof(uint64_t));
    SR_HIP_TRY(hipMemcpyAsync(ph.d_mem, ph.h_staging, up_end, hipMemcpyHostToDevice, stream));
    if (needs_offsets) {
      rc = setup_offsets(p, stream);
      if (rc != SR_OK) return rc;
      SR_HIP_TRY(hipStreamWaitEvent(stream, p->ev_offsets, 0));
    }
    if ((rc = emit_tables(p, ph, stream)) != SR_OK) return rc;
  }
  if (mark) {
    SR_HIP_TRY(hipEventRecord(ph.ev_setup, stream));
    ph.ev_bound = ph.ev_tail = ph.ev_setup;
  } else {
    ph.ev_bound = ph.ev_tail = ph.ev_kernel;   // recorded after the copy kernel, which follows on `stream`
  }
  ph.bound = ptrs;
  ph.bound_valid = true;
  ph.ready = true;
  return SR_OK;
}

// One launch reads and writes the caller's objects concurrently: objects it
// writes must be pairwise disjoint and must not overlap any object it reads.
int check_disjoint(const Phase& ph, const std::vector<uint64_t>& ptrs) {
  struct Span {
    uint64_t lo, hi;
    size_t slot;
  };
  std::vector<Span> w, r;
  for (size_t i = 0; i < ph.obj_use.size(); ++i) {
    if (!ph.obj_use[i]) continue;
    const Span sp{ptrs[i], ptrs[i] + ph.obj_bytes[i], i};
    if (ph.obj_use[i] & 2) w.push_back(sp);
    if (ph.obj_use[i] & 1) r.push_back(sp);
  }
  auto name = [&](size_t slot, char* buf, size_t n) {
    if (slot < ph.n_src_base) snprintf(buf, n, "%s[%zu]", ph.src_name, slot);
    else snprintf(buf, n, "%s[%zu]", ph.dst_name, slot - ph.n_src_base);
    return buf;
  };
  char a[64], b[64];
  std::sort(w.begin(), w.end(), [](const Span& x, const Span& y) { return x.lo < y.lo; });
  for (size_t k = 1; k < w.size(); ++k)
    if (w[k].lo < w[k - 1].hi)
      return fail(SR_EOVERLAP, "%s and %s are written by one launch and overlap",
                  name(w[k - 1].slot, a, sizeof a), name(w[k].slot, b, sizeof b));
  for (const Span& x : r) {
    // the written span starting last below x.hi is the only candidate
    auto it = std::lower_bound(w.begin(), w.end(), x.hi,
                               [](const Span& s, uint64_t v) { return s.lo < v; });
    if (it != w.begin() && std::prev(it)->hi > x.lo)
      return fail(SR_EOVERLAP, "%s is read while %s, which overlaps it, is written",
                  name(x.slot, a, sizeof a), name(std::prev(it)->slot, b, sizeof b));
  }
  return SR_OK;
}

// The copy kernel of a phase over its tables.
int launch_copy(const sr_plan_options& opt, const Phase& ph, PhaseKind kind, const DevItem* items,
                const DevTile* tiles, bool read_ahead, hipStream_t stream) {
  const uint32_t n_tiles = uint32_t(ph.n_recs);
  const uint32_t seg = ph.interleave ? (n_tiles + kXcds - 1) / kXcds : 0u;
  const uint32_t n_pos = seg ? seg * kXcds : n_tiles;
  const uint32_t lanes = shape_lanes(ph.shape);
  uint32_t grid = n_pos;
  if (opt.max_blocks != 0) grid = std::min(grid, opt.max_blocks);
  grid = std::min(grid, 0xffffffffu / lanes);   // grid work-items stay below 2^32
  // A capped grid strides over the positions; a multiple of the segment
  // count keeps every segment on one die.
  if (seg && grid >= kXcds) grid -= grid % kXcds;
  typedef void (*KernelFn)(const DevItem*, const DevTile*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t);
#define SR_PHASES(NT, B, U) {sr_pack_kernel<NT, B, U>, sr_unpack_kernel<NT, B, U>, sr_gather_kernel<NT, B, U>}
#define SR_SHAPES(NT) {SR_PHASES(NT, 1024, 1), SR_PHASES(NT, 512, 2), SR_PHASES(NT, 256, 1), SR_PHASES(NT, 1024, 2)}
  static const KernelFn kernels[2][4][3] = {SR_SHAPES(true), SR_SHAPES(false)};   // by Shape, PhaseKind
#undef SR_SHAPES
#undef SR_PHASES
  const KernelFn fn = kernels[(opt.flags & SR_OPT_TEMPORAL) ? 1 : 0][ph.shape][kind];
  hipLaunchKernelGGL(fn, dim3(grid), dim3(lanes), 0, stream, items, tiles, n_tiles, seg, n_pos, grid,
                     read_ahead ? n_tiles : 0u, uint32_t(ph.rel.size()));
  SR_HIP_TRY(hipGetLastError());
  return SR_OK;
}

// The launch of a phase of at most kHostTableTiles tiles.  On new pointers the
// host writes the items and tile records, bound, to pinned memory and the copy
// kernel reads them there.  A second launch with the same pointers copies the
// tables to the device first and reads them there, as the ones after it do.
// Other pointers go to the other of two pinned tables, so the host waits only
// for a launch two bindings ago.
int run_small(sr_plan* p, Phase& ph, PhaseKind kind, const std::vector<uint64_t>& ptrs, bool rebind,
              hipStream_t stream) {
  TableCache& cache = table_cache();
  const size_t n = ph.rel.size();
  size_t end = 0;
  const size_t o_items = carve(end, n * sizeof(DevItem));
  const size_t o_tiles = carve(end, ph.n_recs * sizeof(DevTile));
  const size_t half = carve(end, 0);
  int rc;
  if (!ph.h_tables &&
      (rc = cache.get(true, p->device, 2 * half, reinterpret_cast<void**>(&ph.h_tables), &ph.h_tables_cap)) != SR_OK)
    return rc;
  const int slot = rebind ? ph.slot ^ 1 : ph.slot;
  unsigned char* table = ph.h_tables + slot * half;
  if (rebind) {
    if (ph.ev_slot[slot]) SR_HIP_TRY(hipEventSynchronize(ph.ev_slot[slot]));
    else if ((rc = cache.get_event(p->device, &ph.ev_slot[slot])) != SR_OK) return rc;
    ph.bound_valid = ph.on_device = false;
    DevItem* items = reinterpret_cast<DevItem*>(table + o_items);
    DevTile* tiles = reinterpret_cast<DevTile*>(table + o_tiles);
    for (uint32_t k = 0; k < n; ++k) {
      const DevRel& h = ph.rel[k];
      uint32_t op;
      const DevItem item = bind_item(h, ptrs.data(), p->piece_offset.data(), op);
      items[k] = item;
      const uint64_t cnt = ph.tile_base[k + 1] - ph.tile_base[k];
      DevTile* t = tiles + (ph.tile_base[k] - h.group_index * cnt + h.group_index);
      for (uint64_t j = 0; j < cnt; ++j) t[j * h.group_size] = tile_record(item, h, k, op, j);
    }
    ph.slot = slot;
    ph.bound = ptrs;
    ph.bound_valid = true;
  }
  if (!rebind) {
    // Each launch that reads the device's tables follows the one before it,
    // whichever streams they are on: the event stands for all of them.
    if (!ph.ev_kernel && (rc = cache.get_event(p->device, &ph.ev_kernel)) != SR_OK) return rc;
    SR_HIP_TRY(hipStreamWaitEvent(stream, ph.ev_kernel, 0));
    if (!ph.on_device) {
      if (!ph.d_tables &&
          (rc = cache.get(false, p->device, half, reinterpret_cast<void**>(&ph.d_tables), &ph.d_tables_cap)) != SR_OK)
        return rc;
      // the first launch, on whichever stream: the event stands for both readers from here on
      SR_HIP_TRY(hipStreamWaitEvent(stream, ph.ev_slot[slot], 0));
      const uint32_t vectors = uint32_t(half / 16);
      hipLaunchKernelGGL(sr_table_copy_kernel, dim3((vectors + kSetupBlock - 1) / kSetupBlock), dim3(kSetupBlock), 0,
                         stream, table, ph.d_tables, vectors);
      SR_HIP_TRY(hipGetLastError());
      SR_HIP_TRY(hipEventRecord(ph.ev_slot[slot], stream));
    }
    table = ph.d_tables;
  }
  rc = launch_copy(p->opt, ph, kind, reinterpret_cast<DevItem*>(table + o_items),
                   reinterpret_cast<DevTile*>(table + o_tiles), !rebind, stream);
  if (rc != SR_OK) return rc;
  SR_HIP_TRY(hipEventRecord(rebind ? ph.ev_slot[slot] : ph.ev_kernel, stream));
  ph.on_device = !rebind;
  return SR_OK;
}

int run_phase(sr_plan* p, Phase& ph, PhaseKind kind, const std::vector<uint64_t>& ptrs,
              hipStream_t stream) {
  if (ph.rel.empty()) return SR_OK;
  const bool rebind = !ph.bound_valid || ptrs != ph.bound;
  int rc;
  if (rebind && (rc = check_disjoint(ph, ptrs)) != SR_OK) return rc;
  rc = ensure_device(p);
  if (rc != SR_OK) return rc;
  if (ph.n_recs <= kHostTableTiles && !ph.ready) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) (void)hipGetLastError();   // the launch reports it
    if (cap == hipStreamCaptureStatusNone) return run_small(p, ph, kind, ptrs, rebind, stream);
    // A graph would replay reads of tables that the host writes again; a
    // phase whose first use is captured keeps the device tables below.
    if (ph.h_tables) return fail(SR_EHIP, "a plan that has run before cannot be captured into a graph");
  }
  if (!ph.ready) {
    // A phase's first use builds its tables and binds the pointers.  They
    // are the library's own memory and read no caller data: while earlier
    // work on `stream` (such as the previous launch group's copy) is still
    // going, a large phase's setup runs beside it on the device's setup
    // stream; on an idle `stream`, or for a small phase, it runs on
    // `stream` directly, since a wait across streams costs the host more
    // than the setup kernel takes on the GPU.
    hipStream_t setup = stream;
    if (ph.n_recs > kInlineSetupTiles) {
      const hipError_t busy = hipStreamQuery(stream);
      (void)hipGetLastError();   // "not ready" is an answer, not an error
      if (busy != hipSuccess && busy != hipErrorNotReady)
        return fail(SR_EHIP, "hipStreamQuery failed: %s", hipGetErrorString(busy));
      if (busy == hipErrorNotReady && (rc = table_cache().setup_stream(p->device, &setup)) != SR_OK) return rc;
    }
    rc = setup_phase(p, ph, kind != kGather, ptrs, setup, setup != stream);
    if (rc != SR_OK) return rc;
    if (setup != stream) SR_HIP_TRY(hipStreamWaitEvent(stream, ph.ev_setup, 0));
  } else if (rebind) {
    // Later rebinds run on `stream`.  The latest bind's copy out of the
    // staging buffer must be done before the host rewrites it, and the bind
    // follows the phase's previous launch, which may still read the tables
    // (and followed the bind before it: one wait for both).
    if (!ph.ev_staging && (rc = table_cache().get_event(p->device, &ph.ev_staging)) != SR_OK) return rc;
    SR_HIP_TRY(hipEventSynchronize(ph.ev_bound));
    std::memcpy(ph.h_ptrs, ptrs.data(), ptrs.size() * sizeof(uint64_t));
    SR_HIP_TRY(hipStreamWaitEvent(stream, ph.ev_tail, 0));
    SR_HIP_TRY(hipMemcpyAsync(ph.d_ptrs, ph.h_ptrs, ptrs.size() * sizeof(uint64_t), hipMemcpyHostToDevice,
                              stream));
    if ((rc = emit_tables(p, ph, stream)) != SR_OK) return rc;
    SR_HIP_TRY(hipEventRecord(ph.ev_staging, stream));
    ph.ev_bound = ph.ev_tail = ph.ev_staging;
    ph.bound = ptrs;
    ph.bound_valid = true;
  } else {
    // the launch before, on whichever stream: the next bind, or the plan's
    // end, waits for the latest launch alone
    SR_HIP_TRY(hipStreamWaitEvent(stream, ph.ev_tail, 0));
  }

  if ((rc = launch_copy(p->opt, ph, kind, ph.d_items, ph.d_tiles, true, stream)) != SR_OK) return rc;
  SR_HIP_TRY(hipEventRecord(ph.ev_kernel, stream));
  ph.ev_tail = ph.ev_kernel;
  return SR_OK;
}

// Releases a phase's device tables (to the table cache).  Waits first for
// the last launches that read them (bind, copy kernel, setup), so a plan can
// be destroyed right after an asynchronous call.
void free_phase(Phase& ph, int device) {
  TableCache& cache = table_cache();
  for (hipEvent_t ev : {ph.ev_kernel, ph.ev_staging, ph.ev_setup, ph.ev_slot[0], ph.ev_slot[1]})
    if (ev) (void)hipEventSynchronize(ev);
  cache.put(false, device, ph.d_mem, ph.d_cap);
  cache.put(true, device, ph.h_staging, ph.h_cap);
  cache.put(false, device, ph.d_tables, ph.d_tables_cap);
  cache.put(true, device, ph.h_tables, ph.h_tables_cap);
  for (hipEvent_t ev : {ph.ev_setup, ph.ev_staging, ph.ev_kernel, ph.ev_slot[0], ph.ev_slot[1]}) cache.put_event(device, ev);
  ph = Phase();
}

// The phase's pointer table: source objects, then destination objects.
std::vector<uint64_t> pointer_table(const void* const* a, size_t na, const void* const* b, size_t nb) {
  std::vector<uint64_t> t(na + nb, 0);
  for (size_t i = 0; i < na; ++i) t[i] = reinterpret_cast<uintptr_t>(a ? a[i] : nullptr);
  for (size_t i = 0; i < nb; ++i) t[na + i] = reinterpret_cast<uintptr_t>(b ? b[i] : nullptr);
  return t;
}

int check_ptrs(const void* const* ptrs, size_t n, const std::vector<uint32_t>& align,
               const char* what) {
  if (n > 0 && ptrs == nullptr) return fail(SR_EINVAL, "%s: pointer array is null", what);
  for (size_t i = 0; i < n; ++i) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(ptrs[i]);
    if (align[i] == 0) continue;   // slot unused by this phase
    if (a == 0) return fail(SR_EINVAL, "%s[%zu] is null", what, i);
    if (a & (align[i] - 1))   // element sizes: powers of two
      return fail(SR_EALIGN, "%s[%zu] = %p is not %u-byte aligned", what, i, ptrs[i], align[i]);
  }
  return SR_OK;
}

// Alignment each pointer of a gather must satisfy: its element size; 0 =
// the slot is not used by the phase.  Computed once, when the plan is made.
void gather_alignment(sr_plan* plan) {
  std::vector<uint32_t>& sal = plan->gather_src_align;
  std::vector<uint32_t>& dal = plan->gather_dst_align;
  sal.assign(plan->src.size(), 0);
  dal.assign(plan->dst.size(), 0);
  for (const sr_piece& pc : plan->pieces) {
    if (pc.src >= 0) sal[pc.src] = dtype_size(plan->src[pc.src].dtype);
    if (pc.dst >= 0) dal[pc.dst] = dtype_size(plan->dst[pc.dst].dtype);
    if (pc.dst2 >= 0) dal[pc.dst2] = dtype_size(plan->dst[pc.dst2].dtype);
  }
}

}  // namespace

// ------------------------------------------------------- allocation-free gather
// The device tables of sr_gather_noalloc live in this array, one copy per GPU,
// allocated with the code object when the library is loaded on a device and
// held until the process exits.  On the host, `scratch` names a stand-in, not
// device memory: host code never passes it to a kernel or a copy, only the
// per-device address that hipGetSymbolAddress returns (scratch_base below).
static __device__ __align__(256) unsigned char scratch[SR_SCRATCH_BYTES];

namespace {

constexpr int kMaxScratchDevices = 256;
std::mutex g_scratch_mu;
uint64_t g_scratch_addr[kMaxScratchDevices];   // 0 = not looked up yet

// Address of `scratch` on the current device `device`, looked up once per
// device (with that device current, as hipGetSymbolAddress requires).
int scratch_base(int device, unsigned char** out) {
  if (device < 0 || device >= kMaxScratchDevices)
    return fail(SR_EINVAL, "device %d out of range for the scratch table", device);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_addr[device] == 0) {
    void* p = nullptr;
    SR_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (p == nullptr) return fail(SR_EHIP, "hipGetSymbolAddress(scratch) returned null on device %d", device);
    g_scratch_addr[device] = reinterpret_cast<uintptr_t>(p);
  }
  *out = reinterpret_cast<unsigned char*>(g_scratch_addr[device]);
  return SR_OK;
}

// Where the gather phase's tables sit in the scratch, and how much it needs.
struct ScratchLayout {
  size_t rel, ptrs, items, base, chunks, tiles, end;
};

ScratchLayout scratch_layout(const Phase& ph) {
  const size_t n = ph.rel.size();
  const size_t nptr = std::max<size_t>(1, size_t(ph.n_src_base) + ph.n_dst_base);
  ScratchLayout L{};
  size_t end = 0;
  L.rel = carve(end, n * sizeof(DevRel));
  L.base = carve(end, (n + 1) * sizeof(uint64_t));
  L.chunks = carve(end, ph.emit_chunks.size() * sizeof(EmitChunk));
  L.ptrs = carve(end, nptr * sizeof(uint64_t));
  L.items = carve(end, n * sizeof(DevItem));
  L.tiles = carve(end, size_t(ph.n_tiles) * sizeof(DevTile));
  L.end = end;
  return L;
}

}  // namespace

// ------------------------------------------------------------------ C ABI

extern "C" {

int sr_abi_version(void) { return SR_ABI_VERSION; }

const char* sr_last_error(void) { return sr_internal::last_error(); }

int sr_selftest(void) {
  // Division constants: exhaustive small divisors, then edge divisors, each
  // against numerators at the edges of the range and a pseudo-random sweep.
  uint64_t x = 0x9E3779B97F4A7C15ull;
  auto rnd = [&x]() {
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    return uint32_t(x >> 16);
  };
  std::vector<uint32_t> divisors;
  for (uint32_t d = 1; d <= 4096; ++d) divisors.push_back(d);
  for (uint32_t s = 12; s < 31; ++s) {
    divisors.push_back((1u << s) - 1);
    divisors.push_back(1u << s);
    divisors.push_back((1u << s) + 1);
    divisors.push_back((1u << s) * 3 / 2);
  }
  divisors.push_back(0x7fffffffu);
  for (uint32_t d : divisors) {
    const DivMagic m = div_magic(d);
    const uint32_t edge[] = {0u, 1u, d - 1, d, d + 1, 2 * d - 1, 0x7fffffffu, 0x80000000u,
                             0xfffffffeu, 0xffffffffu};
    for (uint32_t n : edge) {
      if (div_apply(n, m.m, m.s1, m.s2) != n / d)
        return fail(SR_EINVAL, "selftest: %u / %u gave %u", n, d, div_apply(n, m.m, m.s1, m.s2));
    }
    for (int k = 0; k < 64; ++k) {
      const uint32_t n = rnd();
      if (div_apply(n, m.m, m.s1, m.s2) != n / d)
        return fail(SR_EINVAL, "selftest: %u / %u gave %u", n, d, div_apply(n, m.m, m.s1, m.s2));
    }
  }
  // Vectors of ragged tiles: every byte of a tile comes from its own place,
  // no vector leaves the piece, whatever the row width and the tile's start.
  auto check_tile = [](uint32_t width, uint32_t column, uint32_t nbytes, uint32_t piece_end) -> bool {
    const DivMagic m = div_magic(width);
    const RowMap rows{column, width, m.m, m.s1, m.s2};
    std::vector<uint8_t> seen(size_t(column) + piece_end, 0);   // by byte of the rows, from the first row's start
    auto mark = [&](uint32_t row, uint32_t col) {
      if (col + 16 > width || uint64_t(row) * width + col + 16 > column + piece_end) return false;
      for (uint32_t k = 0; k < 16; ++k) seen[size_t(row) * width + col + k] = 1;
      return true;
    };
    for (uint32_t b = 0; b < (nbytes + 63) / 16 * 16; b += 16) {
      const RowVec v = row_vec(rows, b, nbytes);
      if (v.in && !mark(v.row, v.col)) return false;
      if (v.next && !mark(v.row + 1, 0)) return false;
    }
    for (uint32_t b = 0; b < nbytes; ++b)
      if (!seen[column + b]) return false;
    return true;
  };
  for (uint32_t w = 16; w < 200; ++w)
    for (uint32_t k = 0; k < 24; ++k) {
      const uint32_t n_rows = 1 + rnd() % 40, total = w * n_rows, tile = 256;
      const uint32_t start = rnd() % ((total + tile - 1) / tile) * tile;   // a tile of the piece
      const uint32_t column = start % w, nbytes = std::min(tile, total - start);
      if (!check_tile(w, column, nbytes, total - start))
        return fail(SR_EINVAL, "selftest: rows of %u bytes, tile at %u of %u", w, start, total);
    }
  // Narrow vectors: each follows from the one before as a division gives it.
  for (uint32_t w = 1; w < 700; ++w)
    for (uint32_t k = 0; k < 8; ++k) {
      const DivMagic m = div_magic(w);
      const RowMap rows{rnd() % w, w, m.m, m.s1, m.s2};
      const uint32_t step = 64u << (k & 3), ss = w + rnd() % 1000, ds = w + rnd() % 1000, hs = w + rnd() % 1000;
      uint32_t b = rnd() % 4096;
      RowWalk walk(rows, b, step, ss, ds, hs);
      for (int u = 0; u < 4; ++u, b += step, walk.advance()) {
        uint32_t row, col;
        rows.at(b, row, col);
        if (walk.col != col || walk.at.src != row * ss + col || walk.at.dst != row * ds + col ||
            (w % 2 == 0 && rows.c_base % 2 == 0 && b % 2 == 0 && walk.at.half != row * hs + (col >> 1)))
          return fail(SR_EINVAL, "selftest: walk of rows of %u bytes, step %u", w, step);
      }
    }
  for (uint32_t n = 16; n < 300; ++n) {
    std::vector<uint8_t> seen(n, 0);
    for (uint32_t b = 0; b < n + 64; b += 16) {
      const uint32_t off = contiguous_vec(b, n);
      if (b >= n ? off < n : off + 16 > n) return fail(SR_EINVAL, "selftest: vector %u of %u contiguous bytes", b, n);
      if (b < n) std::fill_n(seen.begin() + off, 16, 1);
    }
    if (std::count(seen.begin(), seen.end(), 1) != n) return fail(SR_EINVAL, "selftest: %u contiguous bytes", n);
  }
  return SR_OK;
}

int sr_plan_create(const sr_tensor* src_tensors, int32_t n_src, const sr_tensor* dst_tensors,
                   int32_t n_dst, int32_t n_peers, const sr_piece* pieces, int32_t n_pieces,
                   const sr_plan_options* options, sr_plan** out_plan) {
  if (out_plan == nullptr) return fail(SR_EINVAL, "out_plan is null");
  *out_plan = nullptr;
  if (n_src < 0 || n_dst < 0 || n_peers < 0 || n_pieces < 0)
    return fail(SR_EINVAL, "negative count (n_src=%d n_dst=%d n_peers=%d n_pieces=%d)", n_src,
                n_dst, n_peers, n_pieces);
  if ((n_src > 0 && !src_tensors) || (n_dst > 0 && !dst_tensors) || (n_pieces > 0 && !pieces))
    return fail(SR_EINVAL, "null array with non-zero count");

  sr_plan_options opt{};
  if (options) opt = *options;
  if (opt.reserved != 0) return fail(SR_EINVAL, "options.reserved must be 0");
  if (opt.flags & ~(SR_OPT_TEMPORAL | SR_OPT_SKIP_COVERAGE | SR_OPT_PIECE_ORDER | SR_OPT_NO_XCD_INTERLEAVE |
                    SR_OPT_NO_ROW_GROUPS | SR_OPT_GATHER_ONLY))
    return fail(SR_EINVAL, "unknown option flags 0x%x", opt.flags);
  if (opt.tile_bytes == 0) opt.tile_bytes = kDefaultTileBytes;
  if (opt.tile_bytes < 4096 || opt.tile_bytes > (16u << 20) ||
      (opt.tile_bytes & (opt.tile_bytes - 1)))
    return fail(SR_EINVAL, "tile_bytes %u must be a power of two in [4096, 16 MiB]",
                opt.tile_bytes);

  int rc;
  for (int32_t i = 0; i < n_src; ++i)
    if ((rc = check_tensor(src_tensors[i], "src", i)) != SR_OK) return rc;
  for (int32_t i = 0; i < n_dst; ++i)
    if ((rc = check_tensor(dst_tensors[i], "dst", i)) != SR_OK) return rc;

  sr_plan* p = new (std::nothrow) sr_plan();
  if (!p) return fail(SR_ENOMEM, "out of host memory");
  p->src.assign(src_tensors, src_tensors + n_src);
  p->dst.assign(dst_tensors, dst_tensors + n_dst);
  p->pieces.assign(pieces, pieces + n_pieces);
  p->n_peers = n_peers;
  p->opt = opt;
  p->piece_offset.assign(n_pieces, UINT64_MAX);
  p->peer_bytes.assign(n_peers, 0);

  std::vector<Box> cover;   // every destination region, for the coverage check
  cover.reserve(size_t(n_pieces) * 2);
  const uint64_t max_row = (uint64_t(1) << 31) - opt.tile_bytes;
  const bool buffers = (opt.flags & SR_OPT_GATHER_ONLY) == 0;   // build the pack and unpack phases
  if (buffers) {
    p->pack.items.reserve(size_t(n_pieces));
    p->unpack.items.reserve(size_t(n_pieces));
  }
  p->gather.items.reserve(size_t(n_pieces));

  for (int32_t k = 0; k < n_pieces; ++k) {
    const sr_piece& pc = pieces[k];
    auto bad = [&](int code) {
      delete p;
      return code;
    };
    if (pc.reserved != 0) return bad(fail(SR_EINVAL, "piece %d: reserved field must be 0", k));
    if (pc.rows == 0 || pc.cols == 0) return bad(fail(SR_EINVAL, "piece %d: empty region", k));
    if (pc.kind != SR_PIECE_COPY && pc.kind != SR_PIECE_RECAST && pc.kind != SR_PIECE_ZERO)
      return bad(fail(SR_EINVAL, "piece %d: unknown kind %d", k, pc.kind));

    if (pc.kind == SR_PIECE_ZERO) {
      if (pc.src != -1 || pc.dst2 != -1)
        return bad(fail(SR_EINVAL, "piece %d: ZERO takes no src/dst2", k));
      if (pc.dst < 0 || pc.dst >= n_dst) return bad(fail(SR_EINVAL, "piece %d: bad dst slot %d", k, pc.dst));
      const sr_tensor& dt = p->dst[pc.dst];
      if ((rc = check_region(dt, pc.dst_row, pc.dst_col, pc.rows, pc.cols, "dst", k)) != SR_OK) return bad(rc);
      const uint32_t es = dtype_size(dt.dtype);
      HostItem it{};
      it.kind = kKindZero;
      it.src_slot = -1;
      it.dst_slot = pc.dst;
      it.dst2_slot = -1;
      it.dst_off = (pc.dst_row * dt.cols + pc.dst_col) * es;
      it.dst_stride = dt.cols * es;
      it.rows = pc.rows;
      it.row_bytes = pc.cols * es;
      it.esize = es;
      it.piece = k;
      it.contiguous = pc.rows == 1 || it.dst_stride == it.row_bytes;
      if (it.contiguous) {
        it.row_bytes *= it.rows;
        it.rows = 1;
      } else if (it.row_bytes > max_row) {
        return bad(fail(SR_EINVAL, "piece %d: strided row of %llu bytes too wide", k,
                        (unsigned long long)it.row_bytes));
      }
      if (buffers) p->unpack.items.push_back(it);
      p->unpack.bytes_written += pc.rows * pc.cols * es;
      p->gather.items.push_back(it);
      p->gather.bytes_written += pc.rows * pc.cols * es;
      cover.push_back({pc.dst_row, pc.dst_row + pc.rows, pc.dst_col, pc.dst_col + pc.cols, k, pc.dst});
      continue;
    }

    if (pc.src < 0 || pc.src >= n_src) return bad(fail(SR_EINVAL, "piece %d: bad src slot %d", k, pc.src));
    if (pc.peer < 0 || pc.peer >= n_peers) return bad(fail(SR_EINVAL, "piece %d: bad peer %d", k, pc.peer));
    const sr_tensor& st = p->src[pc.src];
    if ((rc = check_region(st, pc.src_row, pc.src_col, pc.rows, pc.cols, "src", k)) != SR_OK) return bad(rc);
    const uint32_t es = dtype_size(st.dtype);

    int32_t dst = pc.dst, dst2 = -1;
    if (pc.kind == SR_PIECE_COPY) {
      if (pc.dst2 != -1) return bad(fail(SR_EINVAL, "piece %d: COPY takes no dst2", k));
      if (dst < 0 || dst >= n_dst) return bad(fail(SR_EINVAL, "piece %d: bad dst slot %d", k, dst));
      if (p->dst[dst].dtype != st.dtype)
        return bad(fail(SR_EDTYPE, "piece %d: src dtype %d != dst dtype %d", k, st.dtype, p->dst[dst].dtype));
    } else {
      dst2 = pc.dst2;
      if (st.dtype != SR_DT_F32) return bad(fail(SR_EDTYPE, "piece %d: RECAST source must be f32", k));
      if (dst2 < 0 || dst2 >= n_dst) return bad(fail(SR_EINVAL, "piece %d: bad dst2 slot %d", k, dst2));
      if (p->dst[dst2].dtype != SR_DT_BF16)
        return bad(fail(SR_EDTYPE, "piece %d: RECAST dst2 must be bf16", k));
      if (dst < -1 || dst >= n_dst) return bad(fail(SR_EINVAL, "piece %d: bad dst slot %d", k, dst));
      if (dst >= 0 && p->dst[dst].dtype != SR_DT_F32)
        return bad(fail(SR_EDTYPE, "piece %d: RECAST dst must be f32", k));
      if (dst == dst2) return bad(fail(SR_EINVAL, "piece %d: dst and dst2 are the same slot", k));
      if ((rc = check_region(p->dst[dst2], pc.dst_row, pc.dst_col, pc.rows, pc.cols, "dst2", k)) != SR_OK)
        return bad(rc);
      cover.push_back({pc.dst_row, pc.dst_row + pc.rows, pc.dst_col, pc.dst_col + pc.cols, k, dst2});
    }
    if (dst >= 0) {
      if ((rc = check_region(p->dst[dst], pc.dst_row, pc.dst_col, pc.rows, pc.cols, "dst", k)) != SR_OK)
        return bad(rc);
      cover.push_back({pc.dst_row, pc.dst_row + pc.rows, pc.dst_col, pc.dst_col + pc.cols, k, dst});
    }

    // Buffer placement: pieces of a peer in piece order, 256-byte aligned.
    const uint64_t payload = pc.rows * pc.cols * es;
    uint64_t& cur = p->peer_bytes[pc.peer];
    const uint64_t off = (cur + kBufAlign - 1) / kBufAlign * kBufAlign;
    p->piece_offset[k] = off;
    cur = off + payload;

    // Pack item: source region -> contiguous payload.
    HostItem pk{};
    pk.kind = kKindCopy;
    pk.src_slot = pc.src;
    pk.dst_slot = pc.peer;
    pk.dst2_slot = -1;
    pk.src_off = (pc.src_row * st.cols + pc.src_col) * es;
    pk.src_stride = st.cols * es;
    pk.dst_off = off;
    pk.rows = pc.rows;
    pk.row_bytes = pc.cols * es;
    pk.dst_stride = pk.row_bytes;
    pk.esize = es;
    pk.piece = k;
    pk.contiguous = pc.rows == 1 || pk.src_stride == pk.row_bytes;
    if (pk.contiguous) {
      pk.row_bytes *= pk.rows;
      pk.rows = 1;
    } else if (pk.row_bytes > max_row) {
      return bad(fail(SR_EINVAL, "piece %d: strided row of %llu bytes too wide", k,
                      (unsigned long long)pk.row_bytes));
    }
    if (buffers) p->pack.items.push_back(pk);
    p->pack.bytes_read += payload;
    p->pack.bytes_written += payload;

    // Unpack item: contiguous payload -> destination region(s).
    HostItem up{};
    up.kind = pc.kind == SR_PIECE_COPY ? kKindCopy : kKindRecast;
    up.src_slot = pc.peer;
    up.dst_slot = dst;
    up.dst2_slot = dst2;
    up.src_off = off;
    up.rows = pc.rows;
    up.row_bytes = pc.cols * es;
    up.src_stride = up.row_bytes;
    up.esize = es;
    up.piece = k;
    if (dst >= 0) {
      up.dst_off = (pc.dst_row * p->dst[dst].cols + pc.dst_col) * es;
      up.dst_stride = p->dst[dst].cols * es;
    }
    if (dst2 >= 0) {
      up.dst2_off = (pc.dst_row * p->dst[dst2].cols + pc.dst_col) * 2;
      up.dst2_stride = p->dst[dst2].cols * 2;
    }
    up.contiguous = pc.rows == 1 || ((dst < 0 || up.dst_stride == up.row_bytes) &&
                                     (dst2 < 0 || up.dst2_stride * 2 == up.row_bytes));
    if (up.contiguous) {
      up.row_bytes *= up.rows;
      up.rows = 1;
    } else if (up.row_bytes > max_row) {
      return bad(fail(SR_EINVAL, "piece %d: strided row of %llu bytes too wide", k,
                      (unsigned long long)up.row_bytes));
    }
    if (buffers) p->unpack.items.push_back(up);
    p->unpack.bytes_read += payload;
    if (dst >= 0) p->unpack.bytes_written += payload;
    if (dst2 >= 0) p->unpack.bytes_written += payload / 2;

    // Gather item: source region -> destination region(s), no buffer.
    HostItem ga = up;
    ga.src_slot = pc.src;
    ga.src_off = pk.src_off;
    ga.src_stride = st.cols * es;
    ga.rows = pc.rows;
    ga.row_bytes = pc.cols * es;
    ga.contiguous = pc.rows == 1 ||
                    (ga.src_stride == ga.row_bytes && (dst < 0 || ga.dst_stride == ga.row_bytes) &&
                     (dst2 < 0 || ga.dst2_stride * 2 == ga.row_bytes));
    if (ga.contiguous) {
      ga.row_bytes *= ga.rows;
      ga.rows = 1;
    } else if (ga.row_bytes > max_row) {
      return bad(fail(SR_EINVAL, "piece %d: strided row of %llu bytes too wide", k,
                      (unsigned long long)ga.row_bytes));
    }
    p->gather.items.push_back(ga);
    p->gather.bytes_read += payload;
    if (dst >= 0) p->gather.bytes_written += payload;
    if (dst2 >= 0) p->gather.bytes_written += payload / 2;
  }

  if (!(opt.flags & SR_OPT_SKIP_COVERAGE)) {
    if ((rc = check_coverage(cover, p->dst)) != SR_OK) {
      delete p;
      return rc;
    }
  }
  {
    auto identity = [](size_t n) {
      std::vector<uint32_t> o(n);
      for (uint32_t i = 0; i < n; ++i) o[i] = i;
      return o;
    };
    const bool by_piece = (opt.flags & SR_OPT_PIECE_ORDER) != 0;
    p->pack.n_src_base = uint32_t(n_src);
    p->pack.n_dst_base = uint32_t(n_peers);
    p->unpack.n_src_base = uint32_t(n_peers);
    p->unpack.n_dst_base = uint32_t(n_dst);
    p->gather.n_src_base = uint32_t(n_src);
    p->gather.n_dst_base = uint32_t(n_dst);
    if (buffers) {
      build_rel(p->pack, by_piece ? identity(p->pack.items.size()) : item_order(p->pack, true), opt, false, true, true);
      build_rel(p->unpack, by_piece ? identity(p->unpack.items.size()) : item_order(p->unpack, false), opt, true, false,
                false);
    }
    build_rel(p->gather, by_piece ? identity(p->gather.items.size()) : item_order(p->gather, false), opt, false, false,
              false);
  }
  {
    // object sizes of each phase's pointer table, and the caller's names
    std::vector<uint64_t> sb(n_src), db(n_dst);
    for (int32_t i = 0; i < n_src; ++i)
      sb[i] = p->src[i].rows * p->src[i].cols * uint64_t(dtype_size(p->src[i].dtype));
    for (int32_t i = 0; i < n_dst; ++i)
      db[i] = p->dst[i].rows * p->dst[i].cols * uint64_t(dtype_size(p->dst[i].dtype));
    auto fill = [](Phase& ph, const std::vector<uint64_t>& a, const std::vector<uint64_t>& b,
                   const char* an, const char* bn) {
      ph.obj_bytes = a;
      ph.obj_bytes.insert(ph.obj_bytes.end(), b.begin(), b.end());
      ph.obj_use.resize(ph.obj_bytes.size(), 0);
      ph.src_name = an;
      ph.dst_name = bn;
    };
    if (buffers) {
      fill(p->pack, sb, p->peer_bytes, "src_ptrs", "peer_bufs");
      fill(p->unpack, p->peer_bytes, db, "peer_bufs", "dst_ptrs");
    }
    fill(p->gather, sb, db, "src_ptrs", "dst_ptrs");
  }
  for (Phase* ph : {&p->pack, &p->unpack, &p->gather}) {
    if (ph->n_tiles > UINT32_MAX) {
      delete p;
      return fail(SR_EINVAL, "plan has too many tiles; raise tile_bytes");
    }
    ph->interleave = !(opt.flags & SR_OPT_NO_XCD_INTERLEAVE) && ph->n_recs >= 2 * uint64_t(kXcds) &&
                     ph->n_recs <= UINT32_MAX - kXcds;
  }
  // Per-peer piece lists (piece order) and payloads, from which the device
  // recomputes the buffer offsets.
  p->payload.assign(n_pieces, 0);
  p->peer_begin.assign(size_t(n_peers) + 1, 0);
  for (int32_t k = 0; k < n_pieces; ++k) {
    const sr_piece& pc = pieces[k];
    if (pc.kind == SR_PIECE_ZERO) continue;
    p->payload[k] = pc.rows * pc.cols * uint64_t(dtype_size(p->src[pc.src].dtype));
    ++p->peer_begin[pc.peer + 1];
  }
  for (int32_t q = 0; q < n_peers; ++q) p->peer_begin[q + 1] += p->peer_begin[q];
  p->peer_list.assign(p->peer_begin[n_peers], 0);
  {
    std::vector<uint32_t> fill(p->peer_begin.begin(), p->peer_begin.end() - 1);
    for (int32_t k = 0; k < n_pieces; ++k)
      if (pieces[k].kind != SR_PIECE_ZERO) p->peer_list[fill[pieces[k].peer]++] = uint32_t(k);
  }
  gather_alignment(p);
  // Item tables are rebuilt from the descriptors; the per-item host copies
  // are no longer needed.
  for (Phase* ph : {&p->pack, &p->unpack, &p->gather}) std::vector<HostItem>().swap(ph->items);
  *out_plan = p;
  return SR_OK;
}

int sr_plan_peer_bytes(const sr_plan* plan, int32_t peer, uint64_t* out_bytes) {
  if (!plan || !out_bytes) return fail(SR_EINVAL, "null argument");
  if (peer < 0 || peer >= plan->n_peers) return fail(SR_EINVAL, "peer %d out of range", peer);
  *out_bytes = plan->peer_bytes[peer];
  return SR_OK;
}

int sr_plan_piece_offset(const sr_plan* plan, int32_t piece, uint64_t* out_offset) {
  if (!plan || !out_offset) return fail(SR_EINVAL, "null argument");
  if (piece < 0 || size_t(piece) >= plan->pieces.size())
    return fail(SR_EINVAL, "piece %d out of range", piece);
  *out_offset = plan->piece_offset[piece];
  return SR_OK;
}

int sr_plan_info_get(const sr_plan* plan, sr_plan_info* out) {
  if (!plan || !out) return fail(SR_EINVAL, "null argument");
  out->n_pieces = int64_t(plan->pieces.size());
  out->n_peers = plan->n_peers;
  out->n_src = int64_t(plan->src.size());
  out->n_dst = int64_t(plan->dst.size());
  out->pack_tiles = int64_t(plan->pack.n_tiles);
  out->unpack_tiles = int64_t(plan->unpack.n_tiles);
  out->pack_bytes_read = plan->pack.bytes_read;
  out->pack_bytes_written = plan->pack.bytes_written;
  out->unpack_bytes_read = plan->unpack.bytes_read;
  out->unpack_bytes_written = plan->unpack.bytes_written;
  out->gather_tiles = int64_t(plan->gather.n_tiles);
  out->gather_bytes_read = plan->gather.bytes_read;
  out->gather_bytes_written = plan->gather.bytes_written;
  uint64_t b = 0;
  for (uint64_t v : plan->peer_bytes) b += v;
  out->buffer_bytes = b;
  return SR_OK;
}

int sr_pack(sr_plan* plan, const void* const* src_ptrs, void* const* peer_bufs, hipStream_t stream) {
  if (!plan) return fail(SR_EINVAL, "plan is null");
  if (plan->opt.flags & SR_OPT_GATHER_ONLY) return fail(SR_EINVAL, "sr_pack: the plan was created gather-only");
  // Alignment each pointer must satisfy: its element size; 0 = not read.
  std::vector<uint32_t> sal(plan->src.size(), 0), bal(plan->n_peers, 0);
  for (const sr_piece& pc : plan->pieces) {
    if (pc.kind == SR_PIECE_ZERO) continue;
    sal[pc.src] = dtype_size(plan->src[pc.src].dtype);
    bal[pc.peer] = 16;
  }
  int rc = check_ptrs(src_ptrs, plan->src.size(), sal, "src_ptrs");
  if (rc != SR_OK) return rc;
  rc = check_ptrs(reinterpret_cast<const void* const*>(peer_bufs), plan->n_peers, bal, "peer_bufs");
  if (rc != SR_OK) return rc;
  return run_phase(plan, plan->pack, kPack,
                   pointer_table(src_ptrs, plan->src.size(), peer_bufs, size_t(plan->n_peers)), stream);
}

int sr_unpack(sr_plan* plan, const void* const* peer_bufs, void* const* dst_ptrs, hipStream_t stream) {
  if (!plan) return fail(SR_EINVAL, "plan is null");
  if (plan->opt.flags & SR_OPT_GATHER_ONLY) return fail(SR_EINVAL, "sr_unpack: the plan was created gather-only");
  std::vector<uint32_t> bal(plan->n_peers, 0), dal(plan->dst.size(), 0);
  for (const sr_piece& pc : plan->pieces) {
    if (pc.kind != SR_PIECE_ZERO) bal[pc.peer] = 16;
    if (pc.dst >= 0) dal[pc.dst] = dtype_size(plan->dst[pc.dst].dtype);
    if (pc.dst2 >= 0) dal[pc.dst2] = dtype_size(plan->dst[pc.dst2].dtype);
  }
  int rc = check_ptrs(peer_bufs, plan->n_peers, bal, "peer_bufs");
  if (rc != SR_OK) return rc;
  rc = check_ptrs(reinterpret_cast<const void* const*>(dst_ptrs), plan->dst.size(), dal, "dst_ptrs");
  if (rc != SR_OK) return rc;
  return run_phase(plan, plan->unpack, kUnpack,
                   pointer_table(peer_bufs, size_t(plan->n_peers), dst_ptrs, plan->dst.size()), stream);
}

int sr_gather(sr_plan* plan, const void* const* src_ptrs, void* const* dst_ptrs, hipStream_t stream) {
  if (!plan) return fail(SR_EINVAL, "plan is null");
  int rc = check_ptrs(src_ptrs, plan->src.size(), plan->gather_src_align, "src_ptrs");
  if (rc != SR_OK) return rc;
  rc = check_ptrs(reinterpret_cast<const void* const*>(dst_ptrs), plan->dst.size(), plan->gather_dst_align,
                  "dst_ptrs");
  if (rc != SR_OK) return rc;
  return run_phase(plan, plan->gather, kGather,
                   pointer_table(src_ptrs, plan->src.size(), dst_ptrs, plan->dst.size()), stream);
}

int sr_prepare(hipStream_t stream) {
  int dev = -1;
  SR_HIP_TRY(hipGetDevice(&dev));
  TableCache& cache = table_cache();
  hipStream_t setup = nullptr;
  int rc = cache.setup_stream(dev, &setup);
  if (rc != SR_OK) return rc;
  // one upload of half a block on each stream (a first copy of that size
  // sets up the runtime's copy path for the stream) and one launch (loads
  // the library's GPU code); the blocks then go back to the cache
  constexpr size_t kBytes = size_t(1) << 20;
  void* d = nullptr;
  unsigned char* h = nullptr;
  size_t dcap = 0, hcap = 0;
  if ((rc = cache.get(false, dev, kBytes, &d, &dcap)) != SR_OK) return rc;
  if ((rc = cache.get(true, dev, kBytes, reinterpret_cast<void**>(&h), &hcap)) != SR_OK) {
    cache.put(false, dev, d, dcap);
    return rc;
  }
  std::memset(h, 0, hcap);
  const size_t half = std::min(dcap, hcap) / 2;
  const hipStream_t streams[2] = {stream, setup};
  hipError_t err = hipSuccess;
  for (int i = 0; i < 2 && err == hipSuccess; ++i) {
    err = hipMemcpyAsync(static_cast<unsigned char*>(d) + i * half, h + i * half, half, hipMemcpyHostToDevice,
                         streams[i]);
    if (err == hipSuccess) {
      hipLaunchKernelGGL(sr_prepare_kernel, dim3(1), dim3(64), 0, streams[i]);
      err = hipGetLastError();
    }
  }
  for (hipStream_t st : streams) {
    const hipError_t e = hipStreamSynchronize(st);
    if (err == hipSuccess) err = e;
  }
  cache.put(false, dev, d, dcap);
  cache.put(true, dev, h, hcap);
  if (err != hipSuccess) return fail(SR_EHIP, "sr_prepare: %s", hipGetErrorString(err));
  // events for the first plans' phases
  hipEvent_t ev[8] = {};
  for (hipEvent_t& e : ev)
    if ((rc = cache.get_event(dev, &e)) != SR_OK) break;
  for (hipEvent_t e : ev) cache.put_event(dev, e);
  return rc;
}

int sr_gather_noalloc(const sr_plan* plan, const void* const* src_ptrs, void* const* dst_ptrs,
                      hipStream_t stream) {
  if (!plan) return fail(SR_EINVAL, "plan is null");
  const Phase& ph = plan->gather;
  // The size check comes first: it needs neither the pointers nor a device.
  const ScratchLayout L = scratch_layout(ph);
  if (L.end > size_t(SR_SCRATCH_BYTES))
    return fail(SR_ENOMEM,
                "sr_gather_noalloc: the plan's gather tables need %zu bytes (%zu items, %llu tiles) but "
                "the scratch holds %zu; create the plan with a larger tile_bytes or split the transfer",
                L.end, ph.rel.size(), (unsigned long long)ph.n_tiles, size_t(SR_SCRATCH_BYTES));
  int rc = check_ptrs(src_ptrs, plan->src.size(), plan->gather_src_align, "src_ptrs");
  if (rc != SR_OK) return rc;
  rc = check_ptrs(reinterpret_cast<const void* const*>(dst_ptrs), plan->dst.size(), plan->gather_dst_align,
                  "dst_ptrs");
  if (rc != SR_OK) return rc;
  if (ph.rel.empty()) return SR_OK;
  const std::vector<uint64_t> ptrs = pointer_table(src_ptrs, plan->src.size(), dst_ptrs, plan->dst.size());
  if ((rc = check_disjoint(ph, ptrs)) != SR_OK) return rc;
  // The tables go up from pageable host memory that is released when the
  // call returns: a graph captured from this call would replay copies out of
  // freed memory, so a capturing stream is refused before any device work
  // (the argument checks above need no device).
  {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    SR_HIP_TRY(hipStreamIsCapturing(stream, &cap));
    if (cap != hipStreamCaptureStatusNone)
      return fail(SR_EINVAL,
                  "sr_gather_noalloc: the stream is capturing a graph; this call uploads its tables from "
                  "pageable host memory at every call and cannot be captured");
  }

  int dev = -1;
  SR_HIP_TRY(hipGetDevice(&dev));
  unsigned char* s = nullptr;
  if ((rc = scratch_base(dev, &s)) != SR_OK) return rc;
  DevRel* d_rel = reinterpret_cast<DevRel*>(s + L.rel);
  uint64_t* d_ptrs = reinterpret_cast<uint64_t*>(s + L.ptrs);
  DevItem* d_items = reinterpret_cast<DevItem*>(s + L.items);
  uint64_t* d_base = reinterpret_cast<uint64_t*>(s + L.base);
  EmitChunk* d_chunks = reinterpret_cast<EmitChunk*>(s + L.chunks);
  DevTile* d_tiles = reinterpret_cast<DevTile*>(s + L.tiles);
  const uint32_t n = uint32_t(ph.rel.size());
  const uint32_t n_chunks = uint32_t(ph.emit_chunks.size());

  // Descriptors, tile prefix, chunks and pointers go up in one copy, laid out
  // as in the scratch, from pageable host memory, which HIP copies
  // synchronously: the copy waits for the work queued on `stream` before it
  // (a previous call may still read the scratch) and the host buffer may be
  // released on return.  The GPU idles meanwhile: with one copy per table,
  // 30 us between a call's kernels and the next call's (GPT-125M TP2 -> TP4:
  // 286 us a call), with one copy 18 us (280 us), about 4 us for each copy
  // saved.  Every table is then written whole -- the uploaded ones by the
  // copy, each tile record and each item by the emit -- so nothing needs
  // clearing.
  const size_t up = L.ptrs + ptrs.size() * sizeof(uint64_t);
  std::unique_ptr<unsigned char[]> host(new (std::nothrow) unsigned char[up]);
  if (!host) return fail(SR_ENOMEM, "out of host memory");
  std::memcpy(host.get() + L.rel, ph.rel.data(), n * sizeof(DevRel));
  std::memcpy(host.get() + L.base, ph.tile_base.data(), (size_t(n) + 1) * sizeof(uint64_t));
  std::memcpy(host.get() + L.chunks, ph.emit_chunks.data(), n_chunks * sizeof(EmitChunk));
  std::memcpy(host.get() + L.ptrs, ptrs.data(), ptrs.size() * sizeof(uint64_t));
  SR_HIP_TRY(hipMemcpyAsync(s, host.get(), up, hipMemcpyHostToDevice, stream));
  // gather items read no buffer offsets (no side is a peer buffer)
  hipLaunchKernelGGL(sr_tile_emit_kernel, dim3(std::min<uint32_t>(n_chunks, 65535u)), dim3(kSetupBlock), 0,
                     stream, d_rel, d_base, d_chunks, n_chunks, d_tiles, d_ptrs,
                     static_cast<const uint64_t*>(nullptr), d_items);
  SR_HIP_TRY(hipGetLastError());
  return launch_copy(plan->opt, ph, kGather, d_items, d_tiles, true, stream);
}

void sr_plan_destroy(sr_plan* plan) {
  if (!plan) return;
  free_phase(plan->pack, plan->device);
  free_phase(plan->unpack, plan->device);
  free_phase(plan->gather, plan->device);
  TableCache& cache = table_cache();
  if (plan->ev_offsets) (void)hipEventSynchronize(plan->ev_offsets);
  cache.put(false, plan->device, plan->d_offmem, plan->d_offcap);
  cache.put(true, plan->device, plan->h_offmem, plan->h_offcap);
  cache.put_event(plan->device, plan->ev_offsets);
  delete plan;
}

}  // extern "C"
