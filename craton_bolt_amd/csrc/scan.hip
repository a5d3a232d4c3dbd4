// scan.hip — filter + stream compaction and mask prefix scan.
//
// Replaces launch_predicate_kernel (src/exec/compact.rs:183), the
// predicate / prefix-scan / gather kernels (src/jit/scan_kernel.rs:265,
// src/jit/prefix_scan.rs:175,430,834,1227) and compact_columns_on_gpu
// (src/exec/gpu_compact.rs:1005).  The reference writes a u8 mask, scans it
// per block, scans the block sums on the host (or multipass above 16.8M
// rows), then gathers each column in another launch.  Here a first kernel
// evaluates the predicate into one bit per row and a survivor count per chunk
// of tiles, and a second one sums the counts before its chunk, ranks the
// survivors from the bits and writes every column: each input byte is read
// once and each output byte written once, plus two bits per row.  A
// single-pass form (ticket and decoupled look-back per 4096-row tile) was
// bound by the serial chain between tiles: 21 ns a tile, 154 us of 30M rows
// with nothing kept.
#include <algorithm>

#include "ops_common.h"

namespace bolt {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;  // rows per thread per tile
constexpr int kScanWaves = kScanBlock / 64;
constexpr int kTileRows = kScanBlock * kScanItems;
// Rows per lane in flight: a tile is walked in groups of stripes, so the kernels
// stay small in registers (16 rows at once took 180 VGPRs, two waves a SIMD).
constexpr int kKeepRows = 8;    // of the predicate's columns
constexpr int kMoveRows = 8;    // of the columns that are compacted
static_assert(kScanItems * kScanWaves == 64, "a tile's 64 keep words are scanned by one wave, one per lane");
// A chunk is the tiles one workgroup walks.  Every workgroup of the second
// kernel sums the counts of the chunks before its own (32 KB at most, from
// L2), which saves a scan launch; 30M / 100M rows took 266 / 871 us with 2048
// chunks, 252 / 807 with 4096, 250 / 753 with 8192, 250 / 831 with 32768.
constexpr int kMaxChunks = 8192;
constexpr int kMaxCompactCols = 16;

struct GatherCol {
  const uint8_t* src;
  uint8_t* dst;
  const uint8_t* src_valid;
  uint32_t* dst_valid;  // zeroed bitmap words
  int32_t width;
  int32_t pad;
};
struct GatherList {
  GatherCol c[kMaxCompactCols];
  int32_t n;
  int64_t cap;  // rows the outputs hold: survivors beyond it are counted, not written
};

// Tile row of item j of this lane; rows past the tile's end re-read its last.
__device__ __forceinline__ uint32_t tile_row(int j, uint32_t rows) {
  const uint32_t r = threadIdx.x + (uint32_t)j * kScanBlock;
  return r < rows ? r : rows - 1;
}

// Keep flags (bit j = item j0 + j) of kKeepRows rows of a lane under one
// predicate term.  The dtype and operator are the same for every lane, so they
// are switched on once, outside the row loop, and the loads of all rows are
// issued before the first comparison (evaluating row by row waited on every
// load in turn).  Addresses are the tile's (uniform) plus a 32-bit offset.
template <typename T, typename C>
__device__ __forceinline__ uint32_t term_flags(const void* data, int64_t base, int j0, uint32_t rows, int op, C lit) {
  const T* __restrict__ d = static_cast<const T*>(data) + base;
  T v[kKeepRows];
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) v[j] = d[tile_row(j0 + j, rows)];
  uint32_t lt = 0, eq = 0, gt = 0;  // all three clear: an unordered float comparison
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) {
    const C x = (C)v[j];
    lt |= (uint32_t)(x < lit) << j;
    eq |= (uint32_t)(x == lit) << j;
    gt |= (uint32_t)(x > lit) << j;
  }
  switch (op) {
    case BOLT_CMP_LT: return lt;
    case BOLT_CMP_LE: return lt | eq;
    case BOLT_CMP_GT: return gt;
    case BOLT_CMP_GE: return gt | eq;
    case BOLT_CMP_EQ: return eq;
    case BOLT_CMP_NE: return ~eq;  // C's !=: true for NaN, as eval_term's
  }
  return 0;
}

__device__ __forceinline__ uint32_t term_flags_dec(const DevTerm& t, int64_t base, int j0, uint32_t rows) {
  const ulonglong2* __restrict__ d = static_cast<const ulonglong2*>(t.data) + base;
  ulonglong2 v[kKeepRows];
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) v[j] = d[tile_row(j0 + j, rows)];
  uint32_t keep = 0;
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) {
    const int64_t hi = (int64_t)v[j].y;
    const int c = hi < t.lit_hi ? -1 : hi > t.lit_hi ? 1
                : (v[j].x < (uint64_t)t.lit_i64 ? -1 : v[j].x > (uint64_t)t.lit_i64 ? 1 : 0);
    keep |= (uint32_t)cmp_apply(t.op, c) << j;
  }
  return keep;
}

// Validity flags of the same rows.
__device__ __forceinline__ uint32_t valid_flags(const uint8_t* validity, int64_t base, int j0, uint32_t rows) {
  const uint8_t* __restrict__ d = validity + base / 8;  // a tile starts on a byte
  uint8_t v[kKeepRows];
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) v[j] = d[tile_row(j0 + j, rows) >> 3];
  uint32_t f = 0;
#pragma unroll
  for (int j = 0; j < kKeepRows; j++) f |= (uint32_t)((v[j] >> (threadIdx.x & 7)) & 1) << j;  // 256 j: same bit
  return f;
}

__device__ __forceinline__ uint32_t filter_flags(const DevFilter& f, int64_t base, int j0, uint32_t rows) {
  uint32_t keep = ~0u;
  for (int i = 0; i < f.n; i++) {
    const DevTerm& t = f.t[i];
    if (t.validity) {
      const uint32_t v = valid_flags(t.validity, base, j0, rows);
      keep &= t.op == BOLT_CMP_IS_NULL ? ~v : v;
    } else if (t.op == BOLT_CMP_IS_NULL) {
      keep = 0;
    }
    if (t.op == BOLT_CMP_IS_NULL || t.op == BOLT_CMP_IS_NOT_NULL) continue;
    switch (t.dtype) {
      case BOLT_F64: keep &= term_flags<double, double>(t.data, base, j0, rows, t.op, t.lit_f64); break;
      case BOLT_F32: keep &= term_flags<float, double>(t.data, base, j0, rows, t.op, t.lit_f64); break;
      case BOLT_DEC128: keep &= term_flags_dec(t, base, j0, rows); break;
      case BOLT_I64: keep &= term_flags<int64_t, int64_t>(t.data, base, j0, rows, t.op, t.lit_i64); break;
      case BOLT_BOOL: keep &= term_flags<uint8_t, int64_t>(t.data, base, j0, rows, t.op, t.lit_i64); break;
      default: keep &= term_flags<int32_t, int64_t>(t.data, base, j0, rows, t.op, t.lit_i64); break;
    }
  }
  return keep;
}

// Kept rows of one column, items j0 .. j0 + kMoveRows - 1 of the tile (flags
// `write`), to their output rows.  Lanes without a row read the tile's first
// row (one cached line), so the loads are all in flight before the first store.
typedef uint32_t Quad __attribute__((ext_vector_type(4)));  // a 16-byte value kept in registers

template <typename T>
__device__ __forceinline__ void move_rows(const GatherCol& g, int j0, uint32_t write, int64_t base,
                                          const uint32_t (&rel)[kMoveRows], int64_t prefix) {
  const T* __restrict__ src = reinterpret_cast<const T*>(g.src) + base;
  T* __restrict__ dst = reinterpret_cast<T*>(g.dst) + prefix;
  T v[kMoveRows];
#pragma unroll
  for (int j = 0; j < kMoveRows; j++)
    v[j] = src[(write >> j) & 1u ? threadIdx.x + (uint32_t)(j0 + j) * kScanBlock : 0u];
#pragma unroll
  for (int j = 0; j < kMoveRows; j++)
    if ((write >> j) & 1u) dst[rel[j]] = v[j];
}

// The bits of `x` at the set bits of `m`, moved to the low end in order (the
// parallel-suffix compress of Hacker's Delight, section 7-4).
__device__ __forceinline__ uint64_t compress_bits(uint64_t x, uint64_t m) {
  x &= m;
  uint64_t mk = ~m << 1;  // bits with an odd number of zeros of m to their right are moved first
#pragma unroll
  for (int i = 0; i < 6; i++) {
    uint64_t mp = mk ^ (mk << 1);
    mp ^= mp << 2;
    mp ^= mp << 4;
    mp ^= mp << 8;
    mp ^= mp << 16;
    mp ^= mp << 32;
    const uint64_t mv = mp & m;
    m = (m ^ mv) | (mv >> (1 << i));
    const uint64_t t = x & mv;
    x = (x ^ t) | (t >> (1 << i));
    mk &= ~mp;
  }
  return x;
}

// The survivors' validity bits of one column and tile, written by one wave.
// Lane l holds keep word l of the tile (`own` survivors, the first of them the
// tile's survivor `excl`): it compresses the validity bits of the same 64 rows
// and places them in an LDS bitmap of the tile.  Only the first and last
// output words, shared with the neighbouring tiles, need a global atomic.
__device__ __forceinline__ void write_bitmap(const GatherCol& g, uint64_t keep, uint32_t excl, uint32_t own,
                                             uint32_t total, int64_t tile, int64_t n, int64_t prefix, int64_t cap,
                                             uint32_t* lds) {
  const int lane = threadIdx.x & 63;
  const int64_t byte = tile * (kTileRows / 8) + lane * 8, end = (n + 7) / 8;
  uint64_t v = 0;
  if (byte + 8 <= end) {
    __builtin_memcpy(&v, g.src_valid + byte, 8);
  } else {
    for (int k = 0; byte + k < end; k++) v |= (uint64_t)g.src_valid[byte + k] << (8 * k);
  }
  for (int i = lane; i < kTileRows / 32 + 2; i += 64) lds[i] = 0;
  uint64_t m = compress_bits(v, keep);
  const int64_t room = cap - prefix - excl;  // bits past the capacity are not written
  if (room < (int64_t)own) m &= room > 0 ? (1ull << room) - 1 : 0ull;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const uint32_t skew = (uint32_t)(prefix & 31);  // bit 0 of lds is output row prefix - skew
  const uint32_t at = skew + excl;
  const int sh = at & 31;
  const uint32_t w0 = (uint32_t)(m << sh), w1 = (uint32_t)(m >> (32 - sh)), w2 = sh ? (uint32_t)(m >> (64 - sh)) : 0u;
  if (w0) atomicOr(&lds[at >> 5], w0);
  if (w1) atomicOr(&lds[(at >> 5) + 1], w1);
  if (w2) atomicOr(&lds[(at >> 5) + 2], w2);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  uint32_t* __restrict__ out = g.dst_valid + (prefix - skew) / 32;
  const uint32_t nbits = skew + total;
  for (uint32_t i = lane; i * 32 < nbits; i += 64) {
    const uint32_t w = lds[i];
    const bool whole = (i > 0 || skew == 0) && (i + 1) * 32 <= nbits;
    if (w == 0) continue;  // the bitmap was cleared
    if (whole) out[i] = w;
    else atomicOr(&out[i], w);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// First kernel: keep words and chunk counts.  Word j * kScanWaves + w of a
// tile holds the flags of its 64 rows from (j * kScanWaves + w) * 64.
__global__ __launch_bounds__(kScanBlock) void keep_kernel(DevFilter f, const uint8_t* __restrict__ mask, int64_t n,
                                                          int64_t n_tiles, int64_t per,
                                                          uint64_t* __restrict__ bits, uint32_t* __restrict__ count) {
  __shared__ uint32_t sh_cnt[kScanWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t t0 = (int64_t)blockIdx.x * per;
  const int64_t t1 = t0 + per < n_tiles ? t0 + per : n_tiles;
  uint32_t kept = 0;
  for (int64_t tile = t0; tile < t1; tile++) {
    const int64_t base = tile * kTileRows;
    const uint32_t rows = (uint32_t)(n - base < kTileRows ? n - base : kTileRows);
    uint64_t mine = 0;
#pragma unroll 1
    for (int j0 = 0; j0 < kScanItems; j0 += kKeepRows) {
      uint32_t keep = filter_flags(f, base, j0, rows);
      if (mask) {
        uint8_t m[kKeepRows];
#pragma unroll
        for (int j = 0; j < kKeepRows; j++) m[j] = (mask + base)[tile_row(j0 + j, rows)];
#pragma unroll
        for (int j = 0; j < kKeepRows; j++)
          if (m[j] == 0) keep &= ~(1u << j);
      }
#pragma unroll
      for (int j = 0; j < kKeepRows; j++) {
        const uint64_t b = __ballot(((keep >> j) & 1u) && threadIdx.x + (uint32_t)(j0 + j) * kScanBlock < rows);
        if (lane == j0 + j) mine = b;
      }
    }
    if (lane < kScanItems) bits[tile * 64 + lane * kScanWaves + wave] = mine;
    kept += (uint32_t)__popcll(mine);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) kept += __shfl_xor(kept, m);
  if (lane == 0) sh_cnt[wave] = kept;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t c = 0;
    for (int w = 0; w < kScanWaves; w++) c += sh_cnt[w];
    count[blockIdx.x] = c;  // at most 2^32 rows / kMaxChunks per chunk
  }
}

// Second kernel.  MODE 0: write the survivors of `cols`; MODE 1: write the
// exclusive prefix of the keep flags for every row into `offsets`.
//
// Bound by HBM: the columns where rows survive, the survivors written once.
// A wave needs no other wave of its workgroup: it reads the tile's 64 keep
// words, one per lane, and scans their counts with shuffles.  A column's
// bitmap is one wave's work (write_bitmap), the columns' in turn.  30M rows
// of 8 + 8 + 4 bytes and one bitmap, 30% kept, whole call: 529 us when each
// row went through run-time dispatch, with a wait per load and an atomic per
// bit, 289 us as a single pass with batched loads, 250 us in two kernels
// (785 MB: 3.1 TB/s; a plain copy reaches 4.7 TB/s).
template <int MODE>
__global__ __launch_bounds__(kScanBlock) void compact_kernel(const uint64_t* __restrict__ bits,
                                                             const uint32_t* __restrict__ count, int64_t n,
                                                             int64_t n_tiles, int64_t per, GatherList cols,
                                                             uint32_t* __restrict__ offsets,
                                                             unsigned long long* __restrict__ total_out) {
  __shared__ uint64_t sh_before[kScanWaves];
  __shared__ uint32_t sh_bits[kScanWaves][kTileRows / 32 + 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t prefix;  // output row of the tile's first survivor
  {
    uint64_t c = 0;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kScanBlock) c += count[i];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) c += __shfl_xor(c, m);
    if (lane == 0) sh_before[wave] = c;
    __syncthreads();
    c = 0;
    for (int w = 0; w < kScanWaves; w++) c += sh_before[w];
    prefix = (int64_t)c;
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total_out = c + count[blockIdx.x];
  }
  const int64_t t0 = (int64_t)blockIdx.x * per;
  const int64_t t1 = t0 + per < n_tiles ? t0 + per : n_tiles;
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint64_t next = bits[t0 * 64 + lane];
  for (int64_t tile = t0; tile < t1; tile++) {
    const int64_t base = tile * kTileRows;
    const uint64_t word = next;
    next = bits[(tile + 1 < t1 ? tile + 1 : tile) * 64 + lane];
    uint32_t incl = (uint32_t)__popcll(word);
    const uint32_t own = incl;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t t = __shfl_up(incl, d);
      if (lane >= d) incl += t;
    }
    const uint32_t total = __shfl(incl, 63);
    const uint32_t excl = incl - own;
    if (MODE == 1 || total) {
#pragma unroll 1
      for (int j0 = 0; j0 < kScanItems; j0 += kMoveRows) {
        uint32_t write = 0;      // survivors the outputs have room for
        uint32_t rel[kMoveRows]; // their output rows, from `prefix`
#pragma unroll
        for (int j = 0; j < kMoveRows; j++) {
          const int at = (j0 + j) * kScanWaves + wave;
          const uint64_t b = __shfl(word, at);
          rel[j] = __shfl(excl, at) + (uint32_t)__popcll(b & below);
          write |= (uint32_t)(((b >> lane) & 1u) && prefix + rel[j] < cols.cap) << j;
        }
        if constexpr (MODE == 1) {
#pragma unroll
          for (int j = 0; j < kMoveRows; j++) {
            const int64_t row = base + threadIdx.x + (j0 + j) * kScanBlock;
            if (row < n) offsets[row] = (uint32_t)(prefix + rel[j]);
          }
        } else {
          for (int c = 0; c < cols.n; c++) {
            const GatherCol& g = cols.c[c];
            switch (g.width) {
              case 1: move_rows<uint8_t>(g, j0, write, base, rel, prefix); break;
              case 4: move_rows<uint32_t>(g, j0, write, base, rel, prefix); break;
              case 8: move_rows<uint64_t>(g, j0, write, base, rel, prefix); break;
              case 16: move_rows<Quad>(g, j0, write, base, rel, prefix); break;
            }
          }
        }
      }
      if constexpr (MODE == 0) {
        for (int c = wave; c < cols.n; c += kScanWaves)
          if (cols.c[c].dst_valid)
            write_bitmap(cols.c[c], word, excl, own, total, tile, n, prefix, cols.cap, sh_bits[wave]);
      }
    }
    prefix += total;
  }
}

// Scratch of one call and the first kernel's launch.
struct ScanScratch {
  DevBuf<uint64_t> bits;    // keep words of every tile, then the total
  DevBuf<uint32_t> count;   // survivors per chunk
  int64_t n_tiles = 0, per = 0;
  unsigned grid = 0;
  unsigned long long* total() { return reinterpret_cast<unsigned long long*>(bits.ptr + n_tiles * 64); }
};

static int scan_keep(ScanScratch& sc, const DevFilter& f, const uint8_t* mask, int64_t n, hipStream_t s) {
  sc.n_tiles = (n + kTileRows - 1) / kTileRows;
  sc.per = (sc.n_tiles + kMaxChunks - 1) / kMaxChunks;
  sc.grid = (unsigned)((sc.n_tiles + sc.per - 1) / sc.per);
  BOLT_TRY(sc.bits.alloc((size_t)sc.n_tiles * 64 + 1, s));
  BOLT_TRY(sc.count.alloc(sc.grid, s));
  keep_kernel<<<sc.grid, kScanBlock, 0, s>>>(f, mask, n, sc.n_tiles, sc.per, sc.bits.ptr, sc.count.ptr);
  BOLT_HIP(hipGetLastError());
  return BOLT_OK;
}

// Gather: dst[i] = src[rows[i]].  Bound by the row ids and the output streamed
// past the random reads of src.  A workgroup covers kTakeItems stripes of 256
// consecutive rows at a time: all row ids are loaded before the first is used
// and all gathers before the first store, with clamped indexes instead of
// branches, so a lane keeps kTakeItems random reads in flight.  The validity
// bitmap is rebuilt a wave at a time (64 bits, lanes 0..7 write one byte
// each), so it needs no clearing.  Row ids out of range and NULL row ids are
// noted in a register and reported with one atomic per wave that saw one (an
// atomic per such row, all on one word, took 3.55 ms for 2M NULL row ids
// among 20M int32 rows; 0.10 ms now).
constexpr int kTakeItems = 4;
template <typename T>
__global__ __launch_bounds__(256) void take_kernel(const T* __restrict__ src, const uint8_t* __restrict__ sval,
                                                   int64_t src_len, const uint32_t* __restrict__ rows, int64_t n,
                                                   T* __restrict__ dst, uint8_t* __restrict__ dval,
                                                   uint32_t* __restrict__ err) {
  constexpr int64_t kTile = 256 * kTakeItems;
  const int lane = threadIdx.x & 63;
  const int64_t nbytes = (n + 7) / 8;
  uint32_t seen = 0;
  for (int64_t base = (int64_t)blockIdx.x * kTile + threadIdx.x; base - threadIdx.x < n;
       base += (int64_t)gridDim.x * kTile) {
    uint32_t r[kTakeItems];
    bool ok[kTakeItems];
    T v[kTakeItems];
#pragma unroll
    for (int j = 0; j < kTakeItems; j++) {
      const int64_t i = base + j * 256;
      r[j] = __builtin_nontemporal_load(rows + (i < n ? i : n - 1));
    }
#pragma unroll
    for (int j = 0; j < kTakeItems; j++) {
      const bool in = base + j * 256 < n;
      const bool null_row = r[j] == 0xFFFFFFFFu;  // the NULL index of an outer join
      ok[j] = in && !null_row && (int64_t)r[j] < src_len;
      if (in && !ok[j]) seen |= null_row ? (dval ? 0u : 2u) : 1u;
      if (!ok[j]) r[j] = 0;
    }
    if (src_len > 0) {
#pragma unroll
      for (int j = 0; j < kTakeItems; j++) v[j] = src[r[j]];
    }
#pragma unroll
    for (int j = 0; j < kTakeItems; j++) {
      const int64_t i = base + j * 256;
      if (i < n) dst[i] = ok[j] ? v[j] : T{};
    }
    if (dval) {
#pragma unroll
      for (int j = 0; j < kTakeItems; j++) {
        const uint64_t b = __ballot(ok[j] && bit_valid(sval, r[j]));
        const int64_t byte = (base + j * 256 - lane) / 8 + lane;  // the wave's first row is a multiple of 64
        if (lane < 8 && byte < nbytes) dval[byte] = (uint8_t)(b >> (8 * lane));
      }
    }
  }
  const uint32_t w = (__ballot(seen & 1u) ? 1u : 0u) | (__ballot(seen & 2u) ? 2u : 0u);
  if (w && lane == 0) atomicOr(err, w);
}

template <typename T>
static void launch_take(const bolt_column_t* src, const uint32_t* rows, int64_t n, const bolt_column_t* dst,
                        uint32_t* err, hipStream_t s) {
  take_kernel<T><<<grid_for(n, 256, kTakeItems, 256 * 8), 256, 0, s>>>(
      static_cast<const T*>(src->data), src->validity, src->length, rows, n,
      static_cast<T*>(const_cast<void*>(dst->data)), const_cast<uint8_t*>(dst->validity), err);
}

}  // namespace bolt

using namespace bolt;

extern "C" int bolt_filter_compact(bolt_stream_t stream, const bolt_column_t* cols, int32_t n_cols,
                                   const bolt_filter_t* filter, const uint8_t* mask, bolt_column_t* out,
                                   int64_t* n_out) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  *n_out = 0;
  if (n_cols < 1 || n_cols > kMaxCompactCols || cols == nullptr || out == nullptr)
    return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: 1..%d columns required, got %d", kMaxCompactCols, n_cols);
  int64_t n = cols[0].length;
  GatherList gl;
  memset(&gl, 0, sizeof gl);
  gl.n = n_cols;
  gl.cap = out[0].length;
  for (int i = 0; i < n_cols; i++) {
    if (cols[i].length != n)
      return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: column %d has %lld rows, column 0 has %lld", i,
                       (long long)cols[i].length, (long long)n);
    int w = dtype_size(cols[i].dtype);
    if (w == 0) return set_error(BOLT_ERR_TYPE, "bolt_filter_compact: column %d has unknown dtype", i);
    if (out[i].dtype != cols[i].dtype)
      return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: output column %d dtype differs from input", i);
    if (out[i].length < 0)
      return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: output column %d has a negative capacity", i);
    gl.cap = std::min<int64_t>(gl.cap, out[i].length);
    if (cols[i].validity && !out[i].validity)
      return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: input column %d has NULLs, output has no bitmap", i);
    gl.c[i].src = static_cast<const uint8_t*>(cols[i].data);
    gl.c[i].dst = static_cast<uint8_t*>(out[i].data);
    gl.c[i].src_valid = cols[i].validity;
    gl.c[i].dst_valid = cols[i].validity ? reinterpret_cast<uint32_t*>(const_cast<uint8_t*>(out[i].validity)) : nullptr;
    gl.c[i].width = w;
    if (gl.c[i].dst_valid && (reinterpret_cast<uintptr_t>(gl.c[i].dst_valid) & 3))
      return set_error(BOLT_ERR_PLAN, "bolt_filter_compact: output bitmap %d must be 4-byte aligned", i);
  }
  DevFilter f;
  BOLT_TRY(make_dev_filter(filter, cols, n_cols, n, &f));
  if (n == 0) return BOLT_OK;
  for (int i = 0; i < n_cols; i++)
    if (gl.c[i].dst_valid) BOLT_TRY(fill_u32(gl.c[i].dst_valid, 0, (size_t)(std::min(gl.cap, n) + 31) / 32, s));
  ScanScratch sc;
  BOLT_TRY(scan_keep(sc, f, mask, n, s));
  compact_kernel<0><<<sc.grid, kScanBlock, 0, s>>>(sc.bits.ptr, sc.count.ptr, n, sc.n_tiles, sc.per, gl, nullptr,
                                                   sc.total());
  BOLT_HIP(hipGetLastError());
  unsigned long long total = 0;
  BOLT_TRY(read_back(s, {{&total, sc.total(), 8}}));
  *n_out = (int64_t)total;
  if (*n_out > gl.cap)
    return set_error(BOLT_DECLINE, "bolt_filter_compact: %lld rows survive, the outputs hold %lld",
                     (long long)*n_out, (long long)gl.cap);
  return BOLT_OK;
}

extern "C" int bolt_prefix_scan_mask(bolt_stream_t stream, const uint8_t* mask, int64_t n, uint32_t* offsets,
                                     int64_t* total_out) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  *total_out = 0;
  if (n < 0 || n > 0xFFFFFFFFll) return set_error(BOLT_ERR_PLAN, "bolt_prefix_scan_mask: n out of range");
  if (n == 0) return BOLT_OK;
  if (mask == nullptr) return set_error(BOLT_ERR_PLAN, "bolt_prefix_scan_mask: mask is NULL");
  DevFilter f;
  memset(&f, 0, sizeof f);
  GatherList gl;
  memset(&gl, 0, sizeof gl);
  ScanScratch sc;
  BOLT_TRY(scan_keep(sc, f, mask, n, s));
  compact_kernel<1><<<sc.grid, kScanBlock, 0, s>>>(sc.bits.ptr, sc.count.ptr, n, sc.n_tiles, sc.per, gl, offsets,
                                                   sc.total());
  BOLT_HIP(hipGetLastError());
  unsigned long long total = 0;
  BOLT_TRY(read_back(s, {{&total, sc.total(), 8}}));
  *total_out = (int64_t)total;
  return BOLT_OK;
}

extern "C" int bolt_take(bolt_stream_t stream, const bolt_column_t* src, const uint32_t* rows, int64_t n,
                         bolt_column_t* dst) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  if (!src || !dst) return set_error(BOLT_ERR_PLAN, "bolt_take: NULL column");
  if (n < 0) return set_error(BOLT_ERR_PLAN, "bolt_take: negative length");
  const int width = dtype_size(src->dtype);
  if (width == 0) return set_error(BOLT_ERR_TYPE, "bolt_take: unknown dtype %d", src->dtype);
  if (src->validity && !dst->validity)
    return set_error(BOLT_ERR_PLAN, "bolt_take: the source has a validity bitmap, the destination none");
  dst->dtype = src->dtype;
  dst->scale = src->scale;
  dst->length = n;
  if (n == 0) return BOLT_OK;
  if (!rows || !dst->data) return set_error(BOLT_ERR_PLAN, "bolt_take: NULL rows or destination");
  DevBuf<uint32_t> err;
  BOLT_TRY(err.alloc(1, s));
  BOLT_TRY(fill_u32(err.ptr, 0, 1, s));
  switch (width) {
    case 1: launch_take<uint8_t>(src, rows, n, dst, err.ptr, s); break;
    case 4: launch_take<uint32_t>(src, rows, n, dst, err.ptr, s); break;
    case 8: launch_take<uint64_t>(src, rows, n, dst, err.ptr, s); break;
    case 16: launch_take<uint4>(src, rows, n, dst, err.ptr, s); break;
  }
  BOLT_HIP(hipGetLastError());
  uint32_t e = 0;
  BOLT_TRY(read_back(s, {{&e, err.ptr, 4}}));
  if (e & 1u) return set_error(BOLT_ERR_PLAN, "bolt_take: a row id is out of range (source has %lld rows)",
                               (long long)src->length);
  if (e & 2u) return set_error(BOLT_ERR_PLAN, "bolt_take: a NULL row id needs a destination validity bitmap");
  return BOLT_OK;
}
