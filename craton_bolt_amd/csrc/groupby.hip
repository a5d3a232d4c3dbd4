// groupby.hip — hash GROUP BY.
//
// Replaces execute_groupby (src/exec/groupby.rs:295) with its cascade of
// Tier-1 LDS kernels (src/jit/shmem_*_kernel.rs, groupby_shmem_*_exec.rs),
// Tier-2 partitioned kernels (src/jit/partition_*.rs, groupby_tier2_*.rs) and
// the classic global-atomic path (src/jit/hash_kernels.rs:246,764,
// src/jit/float_atomics.rs:139), which launch one kernel per aggregate and
// round-trip to the host between passes.  Here every aggregate of the query
// is updated by the same pass:
//
//   copy    Only where a sample of the keys finds more groups than an LDS table
//           holds and at most what 256 of them do: the rows are copied grouped
//           by key hash, and pass A gives each part a table (no spills).
//   pass A  LDS tier.  Each workgroup keeps an open-addressing table of up to
//           a few thousand groups in LDS (keys + one 64-bit word per
//           accumulator field) and updates it with LDS atomics.  Rows whose
//           key finds no LDS slot within a short probe are spilled (row ids
//           appended with one atomic per wave).  At the end the workgroup
//           appends its groups as partial records.  A HyperLogLog sketch of
//           every partial key and spilled key estimates the group count.
//   pass B  HBM tier.  A global open-addressing table sized from the sketch
//           (retried 4x larger if it fills) absorbs the partial records and
//           the spilled rows with global atomics.
//   pass C  Extraction: occupied slots are compacted with decoupled look-back
//           into the output columns, finalising each aggregate on the way.
//
// Accumulators are exact where the reference's are: integer SUM keeps a
// 128-bit total per group through a carry-propagating pair of 64-bit
// atomics (overflow of i64 is reported at finalize, like checked_group_sum,
// src/exec/groupby.rs:1775); Decimal128 SUM keeps 192 bits; MIN / MAX of
// every type use native unsigned 64-bit atomic min / max on an
// order-preserving image (floats in the NaN-largest order of
// src/jit/float_atomics.rs:27-62), so no CAS loop is needed.  Float SUM uses
// hardware f64 atomic adds (order-dependent, like the reference's atomics).
//
// Keys (src/exec/groupby_common.rs:352): one Int32 / Int64 / Float32 /
// Float64 / Date32 column, or two 32-bit columns packed (a << 32) | b; float
// keys canonicalise -0.0 and NaN (groupby_common.rs:302).  A single-column
// key with NULLs forms one NULL group (groupby.rs:528-606); two-column keys
// drop rows with a NULL key, as the reference does.  There is no sentinel
// restriction: a key equal to the empty marker and the NULL group live in two
// dedicated slots after the table.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>

#include "groupby_dev.h"
#include "jit.h"
#include "scan_common.h"

namespace bolt {

int radix_sort_u64_pairs(hipStream_t s, const uint64_t* keys_in, const uint32_t* vals_in, int64_t n,
                         uint64_t* keys_out, uint32_t* vals_out, int key_bits, uint64_t in_xor = 0,
                         uint64_t out_xor = 0);

// ---- pass A: LDS tier ------------------------------------------------------------

__global__ __launch_bounds__(kGbBlock) void gb_lds_kernel(KeySpec ks, DevFilter f, GPlan P, int64_t n, int S,
                                                         PartOut out) {
  extern __shared__ unsigned long long sm[];
  const int SS = S + 2;  // + NULL group + empty-marker key
  unsigned long long* skeys = sm;
  unsigned long long* swords = sm + SS;
  uint32_t* shll = reinterpret_cast<uint32_t*>(swords + (size_t)P.words * SS);
  uint32_t* sused = shll + kHllRegs;  // [0..1] specials used, [2] spill count, [3] occupied slots
  for (int i = threadIdx.x; i < SS; i += kGbBlock) skeys[i] = kEmpty;
  for (int w = 0; w < P.words; w++) {
    unsigned long long id = word_identity(P, w);
    for (int i = threadIdx.x; i < SS; i += kGbBlock) swords[(size_t)w * SS + i] = id;
  }
  for (int i = threadIdx.x; i < kHllRegs; i += kGbBlock) shll[i] = 0;
  if (threadIdx.x < 4) sused[threadIdx.x] = 0;
  __syncthreads();

  const int64_t stride = (int64_t)gridDim.x * kGbBlock;
  const int64_t end = ((n + kGbBlock - 1) / kGbBlock) * kGbBlock;  // wave-uniform trip count
  for (int64_t row = (int64_t)blockIdx.x * kGbBlock + threadIdx.x; row < end; row += stride) {
    bool spill = false;
    uint64_t key = 0;
    if (row < n && eval_filter(f, row)) {
      int kr = row_key(ks, row, &key);
      int slot = -1;
      if (kr == 2) {
        slot = S;
        sused[0] = 1;
      } else if (kr == 1) {
        if (key == kEmpty) {
          slot = S + 1;
          sused[1] = 1;
        } else {
          slot = gb_lds_slot(skeys, S, key, &sused[3]);
          spill = slot < 0;
        }
      }
      if (slot >= 0) update_slot(P, swords, SS, (uint32_t)slot, row);
    }
    gb_spill(spill, row, key, sused, shll, out);
  }
  gb_lds_flush(skeys, swords, S, P.words, shll, sused, out);
}

// ---- key partition: when the groups are too many for one LDS table -------------------
//
// Between what one workgroup's LDS table holds and what 256 of them hold, the LDS
// tier alone spills most rows to global atomics on the table's words. There the
// input is first copied, partitioned by the key's hash, and each of 256 workgroups
// runs the LDS tier on one partition: no row spills, and every group is complete in
// one workgroup.  A sample of the keys proposes it: more groups than one table
// holds, and no key frequent enough to leave its partition's workgroup behind the
// others (the plain path aggregates such keys in every workgroup).  From 4096 keys
// a million groups look like 0.6 to 2 million, and a few frequent keys hide a long
// tail, so the first pass over the keys counts the groups (HyperLogLog, within
// 2.3%) and stops the others on the device where they would fill the tables beyond
// kGbPartLoad.  10M rows of two int32 keys and two float sums against the LDS tier
// and global atomics alone: 10,000 groups 1.40 -> 0.56 ms, 100,000 1.60 -> 0.88,
// 980,000 1.76 -> 1.09; 100M rows, 50,000 groups 8.5 -> 3.2 ms.  10M rows of 1.1M
// groups, which the count sends back: 1.69 ms without the attempt, 1.77 with it.
// Below 2^21 rows the copy and the sample's round trip cost what they save.

constexpr int kGbSample = 4096;
constexpr int kGbSampleSlots = 2 * kGbSample;
constexpr int64_t kGbPartMinRows = (int64_t)1 << 21;
// Share of the tables' slots that the counted groups may take.  Three standard
// errors of the count more and the fullest partition's excess are below 0.7
// full, where every key finds a slot within kPartProbes.
constexpr double kGbPartLoad = 0.6;
// How full the plain path's LDS tables are where the partition begins to pay.  The
// rows that they spill there are few, against a copy of all rows: two float sums
// by an int32 key, plain / partitioned in us, 10M rows 0.8 full 501 / 423, 1.0
// full 709 / 424; 50M rows 0.8 full 624 / 1308, 0.9 836 / 1311, 1.0 1783 / 1331,
// 1.1 2070 / 1321 (by two int32 keys 667 / 1615, 717 / 1585, 1556 / 1583, 2037 /
// 1596).
constexpr double gb_part_full(int64_t n) { return n <= (int64_t)1 << 24 ? 0.75 : 1.0; }

// One workgroup: distinct keys among kGbSample stratified rows that pass the
// filter.  out = {rows with a regular key, distinct keys, most frequent key's
// rows}.
__global__ __launch_bounds__(1024) void gb_sample_kernel(KeySpec ks, DevFilter f, int64_t n,
                                                         uint32_t* __restrict__ out) {
  __shared__ unsigned long long slot[kGbSampleSlots];
  __shared__ uint32_t cnt[kGbSampleSlots];
  __shared__ uint32_t res[3];
  for (int i = threadIdx.x; i < kGbSampleSlots; i += 1024) {
    slot[i] = kEmpty;
    cnt[i] = 0;
  }
  if (threadIdx.x < 3) res[threadIdx.x] = 0;
  __syncthreads();
  uint64_t key[kGbSample / 1024];
  int kind[kGbSample / 1024];
#pragma unroll
  for (int u = 0; u < kGbSample / 1024; u++) {
    const int j = u * 1024 + threadIdx.x;
    const int64_t lo = (int64_t)j * n / kGbSample, hi = (int64_t)(j + 1) * n / kGbSample;
    const int64_t row = lo + (int64_t)(((uint64_t)((uint32_t)j * 0x9E3779B1u) * (uint64_t)(hi - lo)) >> 32);
    key[u] = 0;
    kind[u] = eval_filter(f, row) ? row_key(ks, row, &key[u]) : 0;
  }
#pragma unroll
  for (int u = 0; u < kGbSample / 1024; u++) {
    if (kind[u] != 1 || key[u] == kEmpty) continue;
    uint32_t s = (uint32_t)(mix64(key[u]) >> 32) & (kGbSampleSlots - 1);
    for (;;) {  // at most half of the slots are ever taken
      const unsigned long long prev = atomicCAS(&slot[s], kEmpty, (unsigned long long)key[u]);
      if (prev == kEmpty || prev == key[u]) break;
      s = (s + 1) & (kGbSampleSlots - 1);
    }
    atomicAdd(&cnt[s], 1u);
  }
  __syncthreads();
  uint32_t rows = 0, keys = 0, most = 0;
  for (int i = threadIdx.x; i < kGbSampleSlots; i += 1024) {
    const uint32_t c = cnt[i];
    rows += c;
    keys += c ? 1u : 0u;
    most = c > most ? c : most;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    rows += __shfl_xor(rows, m);
    keys += __shfl_xor(keys, m);
    const uint32_t o = __shfl_xor(most, m);
    most = o > most ? o : most;
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&res[0], rows);
    atomicAdd(&res[1], keys);
    atomicMax(&res[2], most);
  }
  __syncthreads();
  if (threadIdx.x < 3) out[threadIdx.x] = res[threadIdx.x];
}

// counts[c][p] -> first output row of chunk c's rows of partition p (rows of a
// partition in chunk order), and ranges[p] = the partition's first row.  One
// workgroup; thread (q, p) sums a quarter q of the chunks.  `hll` holds the keys'
// registers: where the sum of 2^-register, in units of 2^-40, is below `least`
// there are more groups than the tables take, every range is left empty (the
// kernels behind then do nothing) and ranges[256 + 1] is 1.
constexpr int kPartHllUnit = 40;
__global__ __launch_bounds__(1024) void gb_part_offsets_kernel(uint32_t* __restrict__ counts, int chunks,
                                                               const uint32_t* __restrict__ hll, uint64_t least,
                                                               uint32_t* __restrict__ ranges) {
  constexpr int P = 1 << kGbPartBits;
  static_assert(P == 256, "one thread per partition and quarter");
  __shared__ uint32_t part[4][P];
  __shared__ uint32_t start[P];
  __shared__ uint32_t wtot[4];
  __shared__ uint64_t hsum[16];
  const int p = threadIdx.x & (P - 1), q = threadIdx.x >> 8, lane = threadIdx.x & 63;
  uint64_t h = 0;
  for (int i = threadIdx.x; i < kHllRegs; i += 1024) {
    const uint32_t r = hll[i];
    h += r <= kPartHllUnit ? 1ull << (kPartHllUnit - r) : 0ull;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) h += __shfl_xor(h, m);
  if (lane == 0) hsum[threadIdx.x >> 6] = h;
  __syncthreads();
  h = 0;
  for (int w = 0; w < 16; w++) h += hsum[w];
  if (h < least) {  // block-uniform
    if (threadIdx.x <= P + 1) ranges[threadIdx.x] = threadIdx.x == P + 1 ? 1u : 0u;
    return;
  }
  const int per = (chunks + 3) / 4;
  const int c0 = q * per, c1 = c0 + per < chunks ? c0 + per : chunks;
  uint32_t sum = 0;
#pragma unroll 8
  for (int c = c0; c < c1; c++) sum += counts[(int64_t)c * P + p];
  part[q][p] = sum;
  __syncthreads();
  uint32_t tot = 0, inc = 0;
  if (q == 0) {
    for (int k = 0; k < 4; k++) tot += part[k][p];
    inc = tot;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t v = __shfl_up(inc, d);
      if (lane >= d) inc += v;
    }
    if (lane == 63) wtot[p >> 6] = inc;
  }
  __syncthreads();
  if (q == 0) {
    for (int w = 0; w < (p >> 6); w++) inc += wtot[w];
    start[p] = inc - tot;
    ranges[p] = inc - tot;
    if (p == P - 1) {
      ranges[P] = inc;
      ranges[P + 1] = 0;
    }
  }
  __syncthreads();
  uint32_t at = start[p];
  for (int k = 0; k < q; k++) at += part[k][p];
#pragma unroll 8
  for (int c = c0; c < c1; c++) {
    const uint32_t v = counts[(int64_t)c * P + p];
    counts[(int64_t)c * P + p] = at;
    at += v;
  }
}

// Extraction straight from the partial records, when every group has exactly
// one: t.keys / t.words are the records (words `stride` apart).
__global__ __launch_bounds__(256) void gb_extract_dense_kernel(GTable t, GPlan P, KeySpec ks, OutSpec o, int64_t n,
                                                               size_t stride) {
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const uint64_t key = t.keys[i];
    o.packed[i] = key;
    if (ks.n_keys == 1) {
      write_key(o.key[0], i, key);
    } else {
      write_key(o.key[0], i, key >> 32);
      write_key(o.key[1], i, key & 0xFFFFFFFFull);
    }
    for (int a = 0; a < P.n; a++) finalize_to(t, P.a[a], o.agg[a], stride, (uint64_t)i, (uint64_t)i);
  }
}

// ---- pass B: global table ------------------------------------------------------------


__global__ void gb_init_kernel(GTable t, GPlan P) {
  const size_t total = t.cap + 2;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    if (i < t.cap) t.keys[i] = kEmpty;
    for (int w = 0; w < P.words; w++) t.words[(size_t)w * total + i] = word_identity(P, w);
  }
  if (blockIdx.x == 0 && threadIdx.x < 2) t.used_special[threadIdx.x] = 0;
}


__global__ __launch_bounds__(256) void gb_merge_parts_kernel(GTable t, GPlan P, const unsigned long long* pkeys,
                                                            const uint8_t* ptag, const unsigned long long* pwords,
                                                            int64_t pcap, int64_t np) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < np; i += stride) {
    int64_t s = gslot(t, ptag[i], pkeys[i]);
    if (s < 0) continue;
    merge_slot(P, t.words, t.cap + 2, (uint32_t)s, pwords + i, (size_t)pcap);
  }
}

// Partial records merged in two levels when the groups are few: each
// workgroup folds its share of the records into an LDS table (LDS atomics),
// then merges that table into the global one, so a group receives one
// global update per merging workgroup instead of one per LDS-tier workgroup
// (the latter all hit the same few words).  Records that find no LDS slot go
// to the global table directly.
__global__ __launch_bounds__(kGbBlock) void gb_merge_lds_kernel(GTable t, GPlan P, const unsigned long long* pkeys,
                                                               const uint8_t* ptag, const unsigned long long* pwords,
                                                               int64_t pcap, int64_t np, int S) {
  extern __shared__ unsigned long long sm[];
  const int SS = S + 2;
  unsigned long long* skeys = sm;
  unsigned long long* swords = sm + SS;
  uint32_t* sused = reinterpret_cast<uint32_t*>(swords + (size_t)P.words * SS);  // [0..1] specials, [2] occupied
  for (int i = threadIdx.x; i < SS; i += kGbBlock) skeys[i] = kEmpty;
  for (int w = 0; w < P.words; w++) {
    const unsigned long long id = word_identity(P, w);
    for (int i = threadIdx.x; i < SS; i += kGbBlock) swords[(size_t)w * SS + i] = id;
  }
  if (threadIdx.x < 3) sused[threadIdx.x] = 0;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * kGbBlock;
  for (int64_t r = (int64_t)blockIdx.x * kGbBlock + threadIdx.x; r < np; r += stride) {
    const uint8_t tag = ptag[r];
    const unsigned long long key = pkeys[r];
    int slot;
    if (tag == 1) { slot = S; sused[0] = 1; }
    else if (tag == 2) { slot = S + 1; sused[1] = 1; }
    else slot = gb_lds_slot(skeys, S, key, &sused[2]);
    if (slot >= 0) {
      merge_slot(P, swords, SS, (uint32_t)slot, pwords + r, (size_t)pcap);
    } else {
      const int64_t g = gslot(t, tag, key);
      if (g >= 0) merge_slot(P, t.words, t.cap + 2, (uint32_t)g, pwords + r, (size_t)pcap);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < SS; i += kGbBlock) {
    int64_t g = -1;
    if (i < S) {
      if (skeys[i] != kEmpty) g = gslot(t, 0, skeys[i]);
    } else if (sused[i - S]) {
      g = gslot(t, i - S + 1, 0);
    }
    if (g >= 0) merge_slot(P, t.words, t.cap + 2, (uint32_t)g, swords + i, (size_t)SS);
  }
}

// Rows processed straight against the global table: the spilled rows
// (rows != nullptr) or every row of the input (rows == nullptr).
__global__ __launch_bounds__(256) void gb_rows_kernel(GTable t, GPlan P, KeySpec ks, DevFilter f,
                                                     const uint32_t* rows, int64_t nrows) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nrows; i += stride) {
    int64_t row = rows ? (int64_t)rows[i] : i;
    if (!rows && !eval_filter(f, row)) continue;
    uint64_t key = 0;
    int kr = row_key(ks, row, &key);
    if (kr == 0) continue;
    int64_t s = gslot(t, kr == 2 ? 1 : 0, key);
    if (s < 0) continue;
    update_slot(P, t.words, t.cap + 2, (uint32_t)s, row);
  }
}

// The spilled rows, segment by segment: blocks (b, k) for k < K share
// workgroup b's segment.
__global__ __launch_bounds__(256) void gb_rows_seg_kernel(GTable t, GPlan P, KeySpec ks, const uint32_t* spill,
                                                         int64_t per, const uint32_t* seg_count, int K) {
  const int b = blockIdx.x / K, k = blockIdx.x % K;
  const uint32_t cnt = seg_count[b];
  for (uint32_t i = (uint32_t)k * blockDim.x + threadIdx.x; i < cnt; i += (uint32_t)K * blockDim.x) {
    const int64_t row = (int64_t)spill[(int64_t)b * per + i];
    uint64_t key = 0;
    const int kr = row_key(ks, row, &key);
    if (kr == 0) continue;
    const int64_t sl = gslot(t, kr == 2 ? 1 : 0, key);
    if (sl < 0) continue;
    update_slot(P, t.words, t.cap + 2, (uint32_t)sl, row);
  }
}

// Second pass for VAR / STDDEV: M2 = sum over the group of (x - mean)^2, with
// the mean taken from the finished first pass (two-pass variance).
__global__ __launch_bounds__(256) void gb_m2_kernel(GTable t, GPlan P, KeySpec ks, DevFilter f, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const size_t total = t.cap + 2;
  for (int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; row < n; row += stride) {
    if (!eval_filter(f, row)) continue;
    uint64_t key = 0;
    int kr = row_key(ks, row, &key);
    if (kr == 0) continue;
    int64_t s;
    if (kr == 2) s = (int64_t)t.cap;
    else if (key == kEmpty) s = (int64_t)t.cap + 1;
    else {
      uint32_t q = global_find(t.keys, t.cap - 1, key);
      if (q == 0xFFFFFFFFu) continue;
      s = q;
    }
    for (int a = 0; a < P.n; a++) {
      const GAgg& g = P.a[a];
      if (g.kind != K_VAR || !bit_valid(g.validity, row)) continue;
      double v = g.dtype == BOLT_F64 ? static_cast<const double*>(g.data)[row]
               : g.dtype == BOLT_F32 ? (double)static_cast<const float*>(g.data)[row]
               : g.dtype == BOLT_I64 ? (double)static_cast<const int64_t*>(g.data)[row]
                                     : (double)static_cast<const int32_t*>(g.data)[row];
      double sum = as_f64(t.words[(size_t)g.w * total + s]);
      double cnt = (double)t.words[(size_t)g.nw * total + s];
      double d = v - sum / cnt;
      unsafeAtomicAdd(reinterpret_cast<double*>(&t.words[(size_t)(g.w + 1) * total + s]), d * d);
    }
  }
}

// ---- pass C: extraction ---------------------------------------------------------------


constexpr int kExBlock = 256;
constexpr int kExItems = 16;

// ITEMS slots per thread: 16 for large tables, 1 for small ones (more tiles,
// so a table of a few thousand slots is not left to one or two workgroups).
template <int ITEMS>
__global__ __launch_bounds__(kExBlock) void gb_extract_kernel(GTable t, GPlan P, KeySpec ks, OutSpec o,
                                                             uint64_t* __restrict__ status,
                                                             uint32_t* __restrict__ ticket,
                                                             unsigned long long* __restrict__ total_out) {
  __shared__ uint32_t sh_tile;
  __shared__ uint32_t sh_cnt[ITEMS * 4];
  __shared__ uint64_t sh_prefix;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) sh_tile = atomicAdd(ticket, 1u);
  __syncthreads();
  const int64_t tile = sh_tile;
  const uint64_t total = t.cap + 2;
  const uint64_t base = (uint64_t)tile * kExBlock * ITEMS;
  uint32_t keep = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    uint64_t s = base + (uint64_t)j * kExBlock + threadIdx.x;
    bool k = false;
    if (s < t.cap) k = t.keys[s] != kEmpty;
    else if (s < total) k = t.used_special[s - t.cap] != 0;
    keep |= (uint32_t)k << j;
    uint64_t b = __ballot(k);
    if (lane == 0) sh_cnt[j * 4 + wave] = (uint32_t)__popcll(b);
  }
  __syncthreads();
  if (wave == 0) {
    uint32_t c = lane < ITEMS * 4 ? sh_cnt[lane] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      uint32_t v = __shfl_up(incl, d);
      if (lane >= d) incl += v;
    }
    uint32_t tile_total = __shfl(incl, 63);
    if (lane < ITEMS * 4) sh_cnt[lane] = incl - c;
    uint64_t excl = lookback_wave(status, tile, tile_total, &t.err[1]);
    if (lane == 0) {
      sh_prefix = excl;
      if (tile == (int64_t)gridDim.x - 1) *total_out = excl + tile_total;
    }
  }
  __syncthreads();
  const uint64_t prefix = sh_prefix;
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int j = 0; j < ITEMS; j++) {
    bool k = (keep >> j) & 1u;
    uint64_t b = __ballot(k);
    if (!k) continue;
    uint64_t s = base + (uint64_t)j * kExBlock + threadIdx.x;
    uint64_t pos = prefix + sh_cnt[j * 4 + wave] + (uint64_t)__popcll(b & below);
    bool null_group = s == t.cap;
    uint64_t packed = s < t.cap ? t.keys[s] : (null_group ? 0x7FFFFFFFFFFFFFFFull : kEmpty);
    o.packed[pos] = packed;
    o.slot_of[pos] = (uint32_t)s;
    if (ks.n_keys == 1) {
      write_key(o.key[0], pos, null_group ? 0 : packed);
      if (o.key[0].valid && !null_group) set_valid(o.key[0].valid, pos);
    } else {
      write_key(o.key[0], pos, packed >> 32);
      write_key(o.key[1], pos, packed & 0xFFFFFFFFull);
    }
    for (int a = 0; a < P.n; a++) finalize_to(t, P.a[a], o.agg[a], total, s, pos);
  }
}

// err[0] = 1 when a valid Decimal128 key does not fit i64 (its high word is
// not the sign extension of its low word).
__global__ void dec_key_fit_kernel(const uint64_t* __restrict__ d, const uint8_t* __restrict__ valid, int64_t n,
                                   uint32_t* __restrict__ err) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    if (bit_valid(valid, i) && d[2 * i + 1] != (uint64_t)((int64_t)d[2 * i] >> 63)) *err = 1u;
}

// The reference synthesises the NULL group of a single nullable key column
// under the packed key i64::MAX; when a genuine key equal to i64::MAX exists
// it runs its valid-flag executor instead, which drops the NULL-key rows
// (src/exec/groupby.rs:553-583).  res[0] = output row of the NULL group
// (preset -1), res[1] = 1 when a genuine i64::MAX key is among the groups.
__global__ void gb_null_clash_kernel(const unsigned long long* __restrict__ packed, const uint32_t* __restrict__ slot_of,
                                     int64_t n, uint64_t cap, int64_t* __restrict__ res) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if (slot_of[i] == (uint32_t)cap) res[0] = i;
    else if (packed[i] == 0x7FFFFFFFFFFFFFFFull) res[1] = 1;
  }
}

struct MoveCols {
  uint8_t* d[kMaxAggs + 2];
  uint32_t* v[kMaxAggs + 2];
  int32_t w[kMaxAggs + 2];
  int32_t n;
};

// Output row `src` (the last) moves to row `dst`, in every column, its
// validity bit and the packed key / slot arrays the ordering reads.
__global__ void gb_move_row_kernel(MoveCols mc, unsigned long long* __restrict__ packed, uint32_t* __restrict__ slot_of,
                                   int64_t dst, int64_t src) {
  const int c = threadIdx.x;
  if (c == 0) {
    packed[dst] = packed[src];
    slot_of[dst] = slot_of[src];
  }
  if (c >= mc.n) return;
  for (int b = 0; b < mc.w[c]; b++) mc.d[c][dst * mc.w[c] + b] = mc.d[c][src * mc.w[c] + b];
  if (uint32_t* v = mc.v[c]) {
    const uint32_t bit = 1u << (dst & 31);
    if ((v[src >> 5] >> (src & 31)) & 1u) atomicOr(&v[dst >> 5], bit);
    else atomicAnd(&v[dst >> 5], ~bit);
  }
}

// The calling thread's last bolt_groupby plan (bolt_groupby_last_plan).
struct GbLastPlan {
  int32_t tier;  // 0 LDS tier only, 1 global table, 2 partitioned tier
  int64_t spilled, partials;
  int32_t partitions;
  int32_t est_bucket, words;  // the fan-out tuning key
};
static thread_local GbLastPlan t_last_plan{0, 0, 0, 0, 0, 0};

// ---- the partitioned tier's fan-out ---------------------------------------------
// bolt_groupby_autotune_partitions times the partition counts around the
// default (gb_part_bits) and keeps the fastest per (log2 of the estimated
// group count, accumulator words) for the rest of the process;
// BOLT_GB_PART_BITS_DELTA overrides.  While it times a candidate,
// t_force_delta holds it.
std::mutex g_part_mu;
std::map<std::pair<int, int>, int> g_part_delta;
static thread_local int t_force_delta = 0;
static thread_local bool t_forcing = false;

int est_bucket(double est) { return est < 1 ? 0 : (int)std::floor(std::log2(est)); }

int part_bits_delta(double est, int words) {
  if (t_forcing) return t_force_delta;
  if (const char* e = getenv("BOLT_GB_PART_BITS_DELTA")) return std::max(-12, std::min(12, atoi(e)));
  std::lock_guard<std::mutex> lk(g_part_mu);
  const auto it = g_part_delta.find({est_bucket(est), words});
  return it == g_part_delta.end() ? 0 : it->second;
}

// Columns of a result put in key order.  A count that only the device knows
// is read there (n_dev), so the host need not wait for it between the
// extraction and the ordering.
struct OrderCols {
  const uint8_t* src[kMaxAggs + 2];
  uint8_t* dst[kMaxAggs + 2];
  const uint32_t* vsrc[kMaxAggs + 2];
  uint32_t* vdst[kMaxAggs + 2];  // zeroed bitmap words
  int32_t width[kMaxAggs + 2];
};

// out[i] = in[perm[i]] for column blockIdx.y: all columns in one launch.
__global__ __launch_bounds__(256) void gather_cols_kernel(OrderCols oc, const uint32_t* __restrict__ perm, int64_t n,
                                                          const unsigned long long* __restrict__ n_dev) {
  if (n_dev) n = (int64_t)*n_dev;
  const int c = blockIdx.y;
  const uint8_t* src = oc.src[c];
  uint8_t* dst = oc.dst[c];
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    const int64_t p = perm[i];
    switch (oc.width[c]) {
      case 4: reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(src)[p]; break;
      case 8: reinterpret_cast<uint64_t*>(dst)[i] = reinterpret_cast<const uint64_t*>(src)[p]; break;
      case 16: reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[p]; break;
    }
    if (oc.vsrc[c] && ((oc.vsrc[c][p >> 5] >> (p & 31)) & 1u)) atomicOr(&oc.vdst[c][i >> 5], 1u << (i & 31));
  }
}

// i64 order of the packed key as an unsigned radix key
__global__ void flip_sign_kernel(const unsigned long long* __restrict__ in, uint64_t* __restrict__ out,
                                 uint32_t* __restrict__ idx, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    out[i] = in[i] ^ 0x8000000000000000ull;
    idx[i] = (uint32_t)i;
  }
}

// Ascending order of a few signed 64-bit keys (ties by position): the rank
// of a key is the number of keys that precede it.  A workgroup ranks 64 keys;
// its 16 waves count over interleaved shares of all keys (staged through LDS,
// read as broadcasts) and add their counts.  Keys before the workgroup's own
// count when <=, those after when <, so only the 64 in between compare
// positions.  One launch and no host round trip; O(n^2) work, bound by two
// vector operations a pair, so only up to kRankSortMax keys (10,000 keys:
// 28 us; the splitter sort's launches and read-back take about 95).
constexpr int kRankChunk = 4096;
constexpr int64_t kRankSortMax = 16384;
__global__ __launch_bounds__(1024) void rank_sort_kernel(const unsigned long long* __restrict__ keys, int64_t n,
                                                         const unsigned long long* __restrict__ n_dev,
                                                         uint32_t* __restrict__ perm) {
  __shared__ long long sk[kRankChunk];
  __shared__ uint32_t part[16][64];
  if (n_dev) n = (int64_t)*n_dev;
  const int64_t i0 = (int64_t)blockIdx.x * 64;
  if (i0 >= n) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = i0 + lane;
  const long long ki = (long long)keys[i < n ? i : n - 1];
  uint32_t r = 0;
  for (int64_t base = 0; base < n; base += kRankChunk) {
    const int m = (int)(n - base < kRankChunk ? n - base : kRankChunk);
    __syncthreads();
    for (int j = threadIdx.x; j < m; j += 1024) sk[j] = (long long)keys[base + j];
    __syncthreads();
    const int64_t rel = i0 - base;  // the workgroup's first key in this chunk
    const int own = rel < 0 ? 0 : (rel > m ? m : (int)rel);
    const int after = rel < 0 ? 0 : (rel + 64 > m ? m : (int)rel + 64);
#pragma unroll 8
    for (int j = wave; j < own; j += 16) r += sk[j] <= ki ? 1u : 0u;
    for (int j = own + wave; j < after; j += 16) {
      const long long a = sk[j];
      r += (a < ki || (a == ki && j - (int)rel < lane)) ? 1u : 0u;
    }
#pragma unroll 8
    for (int j = after + wave; j < m; j += 16) r += sk[j] < ki ? 1u : 0u;
  }
  part[wave][lane] = r;
  __syncthreads();
  if (wave == 0 && i < n) {
    uint32_t at = 0;
    for (int w = 0; w < 16; w++) at += part[w][lane];
    perm[at] = (uint32_t)i;
  }
}

}  // namespace bolt

using namespace bolt;

// ---- result tables ------------------------------------------------------------------------

struct bolt_table {
  std::vector<bolt_column_t> cols;
  std::vector<void*> owned;
  int64_t n_rows = 0;
  hipStream_t stream = nullptr;
};

extern "C" int bolt_table_num_rows(const bolt_table_t* t, int64_t* n) {
  if (!t) return set_error(BOLT_ERR_PLAN, "table is NULL");
  *n = t->n_rows;
  return BOLT_OK;
}
extern "C" int bolt_table_num_columns(const bolt_table_t* t, int32_t* n) {
  if (!t) return set_error(BOLT_ERR_PLAN, "table is NULL");
  *n = (int32_t)t->cols.size();
  return BOLT_OK;
}
extern "C" int bolt_table_column(const bolt_table_t* t, int32_t i, bolt_column_t* col) {
  if (!t || i < 0 || i >= (int32_t)t->cols.size()) return set_error(BOLT_ERR_PLAN, "column index out of range");
  *col = t->cols[i];
  return BOLT_OK;
}
extern "C" void bolt_table_release(bolt_table_t* t) {
  if (!t) return;
  for (void* p : t->owned) dev_free(p, t->stream);
  delete t;
}

static int table_alloc_col(bolt_table_t* t, int32_t dtype, int64_t cap, bool with_valid, hipStream_t s,
                           bolt_column_t* out) {
  void* d = nullptr;
  BOLT_TRY(dev_alloc(&d, (size_t)(cap > 0 ? cap : 1) * dtype_size(dtype), s));
  t->owned.push_back(d);
  void* v = nullptr;
  if (with_valid) {
    size_t words = (size_t)(cap + 31) / 32 + 1;
    BOLT_TRY(dev_alloc(&v, words * 4, s));
    t->owned.push_back(v);
    BOLT_TRY(fill_u32(v, 0, words, s));
  }
  out->data = d;
  out->validity = static_cast<const uint8_t*>(v);
  out->length = 0;
  out->dtype = dtype;
  out->scale = 0;
  return BOLT_OK;
}

// ---- plan construction ---------------------------------------------------------------------

int bolt::make_gplan(const bolt_agg_t* aggs, int32_t n_aggs, const bolt_column_t* inputs, int32_t n_inputs,
                      int64_t n, GPlan* P, int32_t* out_dtype) {
  memset(P, 0, sizeof *P);
  if (n_aggs < 0 || n_aggs > kMaxAggs) return set_error(BOLT_ERR_PLAN, "%d aggregates (max %d)", n_aggs, kMaxAggs);
  int w = 0;
  for (int i = 0; i < n_aggs; i++) {
    GAgg& g = P->a[i];
    g.op = aggs[i].op;
    g.nw = -1;
    if (g.op < BOLT_AGG_SUM || g.op > BOLT_AGG_STDDEV_SAMP) return set_error(BOLT_ERR_PLAN, "aggregate %d: unknown op", i);
    if (g.op == BOLT_AGG_COUNT_STAR) {
      g.kind = K_COUNT;
      g.dtype = BOLT_I64;
      g.w = w++;
      out_dtype[i] = BOLT_I64;
      continue;
    }
    if (aggs[i].col < 0 || aggs[i].col >= n_inputs)
      return set_error(BOLT_ERR_PLAN, "aggregate %d: input column %d out of range (%d inputs)", i, aggs[i].col, n_inputs);
    const bolt_column_t& c = inputs[aggs[i].col];
    if (c.length != n)
      return set_error(BOLT_ERR_PLAN, "aggregate %d: input has %lld rows, keys have %lld", i, (long long)c.length,
                       (long long)n);
    g.data = c.data;
    g.validity = c.validity;
    g.dtype = c.dtype;
    bool nullable = c.validity != nullptr;
    int dt = c.dtype;
    if (g.op == BOLT_AGG_COUNT) {
      g.kind = K_COUNT;
      g.w = w++;
      out_dtype[i] = BOLT_I64;
      continue;
    }
    if (dt == BOLT_BOOL) return set_error(BOLT_ERR_TYPE, "aggregate %d: Bool inputs are not supported", i);
    if (dt == BOLT_TIMESTAMP)
      return set_error(BOLT_ERR_TYPE, "aggregate %d: a Timestamp enters through an expression program (EXTRACT, "
                       "DATE_TRUNC, comparisons)", i);
    switch (g.op) {
      case BOLT_AGG_SUM:
        if (dt == BOLT_DATE32) return set_error(BOLT_ERR_TYPE, "SUM over a temporal type is undefined in SQL (Date32)");
        if (dt == BOLT_DEC128) { g.kind = K_DSUM; g.w = w; w += 3; out_dtype[i] = BOLT_DEC128; }
        else if (dtype_is_float(dt)) { g.kind = K_FSUM; g.w = w++; out_dtype[i] = dt; }
        else { g.kind = K_ISUM; g.w = w; w += 2; out_dtype[i] = BOLT_I64; }
        if (nullable) g.nw = w++;
        break;
      case BOLT_AGG_MIN:
      case BOLT_AGG_MAX:
        if (dt == BOLT_DEC128) return set_error(BOLT_ERR_UNSUPPORTED, "GROUP BY MIN/MAX over Decimal128");
        g.kind = K_MINMAX;
        g.w = w++;
        out_dtype[i] = dt;
        if (nullable) g.nw = w++;
        break;
      case BOLT_AGG_AVG:
        if (dt == BOLT_DATE32 || dt == BOLT_DEC128) return set_error(BOLT_ERR_TYPE, "AVG over %s is not supported", dtype_name(dt));
        g.kind = K_AVG;
        g.w = w++;
        g.nw = w++;
        out_dtype[i] = BOLT_F64;
        break;
      default:
        if (dt == BOLT_DATE32 || dt == BOLT_DEC128) return set_error(BOLT_ERR_TYPE, "VAR/STDDEV over %s is not supported", dtype_name(dt));
        g.kind = K_VAR;
        g.w = w;
        w += 2;
        g.nw = w++;
        out_dtype[i] = BOLT_F64;
        break;
    }
  }
  P->n = n_aggs;
  P->words = w;
  return BOLT_OK;
}

double bolt::hll_estimate(const uint32_t* regs) {
  const double m = kHllRegs;
  double sum = 0;
  int zeros = 0;
  for (int i = 0; i < kHllRegs; i++) {
    sum += std::ldexp(1.0, -(int)regs[i]);
    zeros += regs[i] == 0;
  }
  double alpha = 0.7213 / (1.0 + 1.079 / m);
  double e = alpha * m * m / sum;
  if (e <= 2.5 * m && zeros > 0) e = m * std::log(m / zeros);
  return e;
}

// Groups that a sample of m keys with d distinct ones stands for, if they are
// about equally frequent: the G with G (1 - exp(-m / G)) = d.
double bolt::sample_groups(double m, double d) {
  if (d >= m) return 1e18;
  double lo = d, hi = 1e12;
  for (int i = 0; i < 100; i++) {
    const double g = std::sqrt(lo * hi);
    if (g * -std::expm1(-m / g) < d) lo = g;
    else hi = g;
  }
  return lo;
}

uint64_t bolt::next_pow2(uint64_t x) {
  uint64_t p = 1;
  while (p < x) p <<= 1;
  return p;
}

// The generated LDS-tier kernel's shape for this query (filter, keys, plan).
static int gb_jit_spec(const KeySpec& ks, const GPlan& P, const DevFilter& f, GbJitSpec* sp, JitLits* lits,
                       JitCols* cols) {
  *sp = GbJitSpec();
  memset(lits, 0, sizeof *lits);
  memset(cols, 0, sizeof *cols);
  sp->n_keys = ks.n_keys;
  sp->t0 = ks.t0;
  sp->t1 = ks.t1;
  sp->kv0 = ks.v0 != nullptr;
  sp->kv1 = ks.n_keys == 2 && ks.v1 != nullptr;
  sp->words = P.words;
  sp->ident.assign(P.words, 0ull);
  for (int a = 0; a < P.n; a++)
    if (P.a[a].kind == K_MINMAX) sp->ident[P.a[a].w] = P.a[a].op == BOLT_AGG_MIN ? ~0ull : 0ull;
  for (int t = 0; t < f.n; t++) {
    const int c = jit_row_agg_col(f.t[t].data, f.t[t].validity, f.t[t].dtype, &sp->cols, cols);
    if (c < 0) return set_error(BOLT_ERR_UNSUPPORTED, "jit: too many columns");
    sp->terms.push_back({c, f.t[t].op});
    lits->i[t] = f.t[t].lit_i64;
    lits->f[t] = f.t[t].lit_f64;
    lits->hi[t] = f.t[t].lit_hi;
  }
  for (int a = 0; a < P.n; a++) {
    const GAgg& g = P.a[a];
    GbJitSpec::Agg ja{g.op, g.kind, g.dtype, -1, g.w, g.nw};
    if (g.op != BOLT_AGG_COUNT_STAR) {
      ja.col = jit_row_agg_col(g.data, g.validity, g.dtype, &sp->cols, cols);
      if (ja.col < 0) return set_error(BOLT_ERR_UNSUPPORTED, "jit: too many columns");
    }
    sp->aggs.push_back(ja);
  }
  // rows in flight per lane: as many as the registers hold at 1024 threads
  // (32-bit words loaded per row: keys and every column)
  int words = ks.n_keys;
  for (const JitSpec::Col& c : sp->cols) words += c.dtype == BOLT_DEC128 ? 4 : (dtype_size(c.dtype) + 3) / 4;
  sp->unroll = words <= 6 ? 8 : words <= 12 ? 4 : 2;
  if (const char* u = getenv("BOLT_GB_UNROLL")) {
    const int v = atoi(u);
    if (v >= 1 && v <= 8) sp->unroll = v;
  }
  return BOLT_OK;
}

// The key-partitioned copy of an input and where its partitions start.
struct GbPartCopy {
  DevBuf<uint32_t> counts, ranges, hll;
  std::vector<DevBuf<uint8_t>> bufs;
  KeySpec ks;          // the copied key (NULLs one byte per row)
  GbJitSpec spec;      // the LDS tier's kernel over the copies
  JitCols cols;
};

// Groups that the partitions' tables of part_S slots take.
static double part_groups_most(int part_S) { return kGbPartLoad * part_S * (1 << kGbPartBits); }

// Whether the input goes through the key partition (synchronises).
static int gb_part_wanted(hipStream_t s, const KeySpec& ks, const DevFilter& f, int64_t n, int S, int part_S,
                          bool* yes) {
  *yes = false;
  if (const char* e = getenv("BOLT_GB_KEY_PARTITION")) {  // testing: 0 never, 1 always
    *yes = e[0] == '1';
    return BOLT_OK;
  }
  if (n < kGbPartMinRows) return BOLT_OK;
  DevBuf<uint32_t> out;
  uint32_t h[3];
  BOLT_TRY(out.alloc(4, s));
  gb_sample_kernel<<<1, 1024, 0, s>>>(ks, f, n, out.ptr);
  BOLT_HIP(hipGetLastError());
  BOLT_TRY(read_back(s, {{h, out.ptr, 12}}));
  // few sampled rows pass the filter: the plain path; a key above 0.4% of the
  // rows (its share of 1/256) would make one workgroup the last; above 1.2 times
  // the limit an attempt, which costs 110 us where the count ends it, rarely holds
  const double est = sample_groups(h[0], h[1]);
  *yes = h[0] >= kGbSample / 4 && est > gb_part_full(n) * S && est <= 1.2 * part_groups_most(part_S) &&
         h[2] <= 8 + h[0] / 256;
  return BOLT_OK;
}

// Copies the rows that pass the filter, partitioned by key hash (nothing, with
// ranges[257] set, where the groups are too many).
static int gb_part_copy(hipStream_t s, const KeySpec& ks, const GbJitSpec& gs, JitLits& lits, JitCols& cols, int64_t n,
                        int part_S, GbPartCopy* out, bool* ok) {
  *ok = false;
  std::vector<int> copied;
  for (const GbJitSpec::Agg& a : gs.aggs)
    if (a.col >= 0 && std::find(copied.begin(), copied.end(), a.col) == copied.end()) copied.push_back(a.col);
  hipFunction_t fn = nullptr;
  if (jit_get_keyed(gb_partition_jit_key(gs, copied), [&] { return jit_gb_partition_source(gs, copied); }, &fn) != BOLT_OK) {
    clear_error();
    return BOLT_OK;
  }
  const int64_t tiles = (n + kGbPartTile - 1) / kGbPartTile;
  const int64_t per_tiles = (tiles + 511) / 512;
  const int chunks = (int)((tiles + per_tiles - 1) / per_tiles);
  long long per = per_tiles * kGbPartTile, nn = n;
  const int np = 1 << kGbPartBits;
  BOLT_TRY(out->counts.alloc((size_t)chunks * np, s));
  BOLT_TRY(out->ranges.alloc(np + 2, s));
  BOLT_TRY(out->hll.alloc(kHllRegs, s));
  BOLT_TRY(fill_u32(out->hll.ptr, 0, kHllRegs, s));
  GbCopies dst;
  memset(&dst, 0, sizeof dst);
  auto buf = [&](size_t bytes, void** p) -> int {
    out->bufs.emplace_back();
    BOLT_TRY(out->bufs.back().alloc(bytes, s));
    *p = out->bufs.back().ptr;
    return BOLT_OK;
  };
  void* p = nullptr;
  // the LDS tier over the copies: the same aggregates, no filter, and only
  // the columns that the aggregates read
  GbJitSpec& sp = out->spec;
  sp = gs;
  sp.terms.clear();
  sp.cols.clear();
  memset(&out->cols, 0, sizeof out->cols);
  memset(&out->ks, 0, sizeof out->ks);
  out->ks = ks;
  out->ks.v0 = out->ks.v1 = nullptr;
  const bool kv = ks.n_keys == 1 && ks.v0 != nullptr;
  sp.kv0 = kv;
  sp.kv1 = false;
  if (sp.t0 == BOLT_DEC128) sp.t0 = BOLT_I64;
  BOLT_TRY(buf((size_t)n * dtype_size(sp.t0), &p));
  out->ks.d0 = dst.k0 = p;
  if (ks.n_keys == 2) {
    BOLT_TRY(buf((size_t)n * 4, &p));
    out->ks.d1 = dst.k1 = p;
  }
  if (kv) {
    BOLT_TRY(buf((size_t)n, &p));
    dst.kv = static_cast<unsigned char*>(p);
    out->ks.v0 = dst.kv;
  }
  bool any_valid = kv;
  std::vector<int> at(gs.cols.size(), -1);
  for (int c : copied) {
    const JitSpec::Col& jc = gs.cols[c];
    BOLT_TRY(buf((size_t)n * dtype_size(jc.dtype), &p));
    dst.d[c] = p;
    if (jc.has_valid) {
      BOLT_TRY(buf((size_t)n, &p));
      dst.v[c] = static_cast<unsigned char*>(p);
      any_valid = true;
    }
    at[c] = (int)sp.cols.size();
    out->cols.d[at[c]] = dst.d[c];
    out->cols.v[at[c]] = dst.v[c];
    sp.cols.push_back(jc);
  }
  for (GbJitSpec::Agg& a : sp.aggs)
    if (a.col >= 0) a.col = at[a.col];
  sp.vbytes = any_valid;
  unsigned int* counts = out->counts.ptr;
  unsigned int* hll = out->hll.ptr;
  const unsigned int* rows_kept = out->ranges.ptr + np;
  // the registers' sum at which hll_estimate gives the limit (its plain form,
  // the one that holds at limits of tens of thousands and more)
  const double m = kHllRegs, most = part_groups_most(part_S);
  const uint64_t least = (uint64_t)std::ldexp(0.7213 / (1.0 + 1.079 / m) * m * m / most, kPartHllUnit);
  for (int mode = 0; mode < 2; mode++) {
    void* args[] = {&nn, &per, &mode, (void*)&ks.d0, (void*)&ks.v0, (void*)&ks.d1, (void*)&ks.v1, &lits, &cols,
                    (void*)&counts, &dst, (void*)&hll, (void*)&rows_kept};
    BOLT_HIP(hipModuleLaunchKernel(fn, (unsigned)chunks, 1, 1, 1024, 1, 1, 0, s, args, nullptr));
    if (mode == 0) gb_part_offsets_kernel<<<1, 1024, 0, s>>>(counts, chunks, hll, least, out->ranges.ptr);
  }
  BOLT_HIP(hipGetLastError());
  *ok = true;
  return BOLT_OK;
}

static int lds_max_bytes() {
  static int cached = -1;
  if (cached < 0) {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) {
      (void)hipGetLastError();
      v = 65536;
    }
    cached = v;
  }
  return cached;
}

// Slots of an LDS table of W words in `budget` bytes, beside the sketch.
static int lds_slots(int budget, int W, int most) {
  return std::min(most, (int)((budget - (kHllRegs + 4) * 4) / (8 * (1 + W))) - 2);
}

static int lds_budget_bytes() {
  static int cached = -1;
  if (cached < 0) {
    const int v = lds_max_bytes();
    int kb = 96;  // one 1024-thread workgroup per CU either way; BOLT_GB_LDS_KB overrides
    if (const char* e = getenv("BOLT_GB_LDS_KB")) {
      const int x = atoi(e);
      if (x >= 16 && x <= 160) kb = x;
    }
    cached = std::min(v, kb * 1024);
  }
  return cached;
}

// Puts a result's columns in ascending packed-key order (src/exec/groupby.rs:800):
// `n` groups, or at most n with the count at n_dev.  `cols` become the ordered
// columns, owned by the table as well.
static int order_groups(hipStream_t s, bolt_table* tbl, std::vector<bolt_column_t>& cols,
                        const unsigned long long* packed, int64_t n, const unsigned long long* n_dev) {
  if (n < 1) return BOLT_OK;
  DevBuf<uint64_t> kin, kout;
  DevBuf<uint32_t> vin, perm;
  BOLT_TRY(perm.alloc((size_t)n, s));
  if (n <= kRankSortMax + 2) {
    rank_sort_kernel<<<(unsigned)((n + 63) / 64), 1024, 0, s>>>(packed, n, n_dev, perm.ptr);
  } else {
    BOLT_TRY(kin.alloc((size_t)n, s));
    BOLT_TRY(kout.alloc((size_t)n, s));
    BOLT_TRY(vin.alloc((size_t)n, s));
    flip_sign_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(packed, kin.ptr, vin.ptr, n);
    BOLT_TRY(radix_sort_u64_pairs(s, kin.ptr, vin.ptr, n, kout.ptr, perm.ptr, 64));
  }
  OrderCols oc;
  memset(&oc, 0, sizeof oc);
  for (size_t c = 0; c < cols.size(); c++) {
    bolt_column_t out;
    BOLT_TRY(table_alloc_col(tbl, cols[c].dtype, n, cols[c].validity != nullptr, s, &out));
    oc.src[c] = static_cast<const uint8_t*>(cols[c].data);
    oc.dst[c] = static_cast<uint8_t*>(out.data);
    oc.vsrc[c] = reinterpret_cast<const uint32_t*>(cols[c].validity);
    oc.vdst[c] = reinterpret_cast<uint32_t*>(const_cast<uint8_t*>(out.validity));
    oc.width[c] = dtype_size(cols[c].dtype);
    cols[c] = out;
  }
  gather_cols_kernel<<<dim3(grid_for(n, 256, 4), (unsigned)cols.size()), 256, 0, s>>>(oc, perm.ptr, n, n_dev);
  BOLT_HIP(hipGetLastError());
  return BOLT_OK;
}

// `parted` (may be null: no key partition) is set once the call has gone for the
// key partition; kGbPlain: it does not hold the input, run again without.
constexpr int kGbPlain = 1 << 20;  // no status of the API
static int groupby_run(bolt_stream_t stream, const bolt_column_t* keys, int32_t n_keys, const bolt_column_t* inputs,
                       int32_t n_inputs, const bolt_agg_t* aggs, int32_t n_aggs, const bolt_filter_t* filter,
                       uint32_t flags, bool* parted, bolt_table_t** out) {
  BOLT_CHECK_DEVICE();
  clear_error();
  *out = nullptr;
  hipStream_t s = (hipStream_t)stream;
  if (n_keys < 1 || n_keys > 2 || keys == nullptr)
    return set_error(BOLT_ERR_PLAN, "bolt_groupby: 1 or 2 key columns required, got %d", n_keys);
  const int64_t n = keys[0].length;
  if (n > 0xFFFFFFFFll) return set_error(BOLT_ERR_PLAN, "bolt_groupby: %lld rows exceeds the u32 row-id limit", (long long)n);
  KeySpec ks;
  memset(&ks, 0, sizeof ks);
  ks.n_keys = n_keys;
  for (int k = 0; k < n_keys; k++) {
    int dt = keys[k].dtype;
    // src/exec/groupby_common.rs:117 key_bit_width accepts Int32 / Int64 /
    // floats; Date32 packs like Int32, and a single Decimal128 key whose
    // values fit i64 packs like Int64 (wider values decline)
    if (!(dt == BOLT_I32 || dt == BOLT_I64 || dt == BOLT_F32 || dt == BOLT_F64 || dt == BOLT_DATE32 ||
          (dt == BOLT_DEC128 && n_keys == 1)))
      return set_error(BOLT_ERR_TYPE, "GROUP BY key dtype %s not supported", dtype_name(dt));
    if (keys[k].length != n) return set_error(BOLT_ERR_PLAN, "bolt_groupby: key columns differ in length");
    if (n_keys == 2 && dtype_size(dt) != 4)
      return set_error(BOLT_ERR_UNSUPPORTED,
                       "multi-column GROUP BY with > 64 bits of key width not yet supported");
  }
  ks.d0 = keys[0].data;
  ks.v0 = keys[0].validity;
  ks.t0 = keys[0].dtype;
  if (n_keys == 2) {
    ks.d1 = keys[1].data;
    ks.v1 = keys[1].validity;
    ks.t1 = keys[1].dtype;
  }
  ks.null_group = (n_keys == 1 && keys[0].validity != nullptr) ? 1 : 0;
  GPlan P;
  int32_t out_dt[kMaxAggs];
  BOLT_TRY(make_gplan(aggs, n_aggs, inputs, n_inputs, n, &P, out_dt));
  DevFilter f;
  BOLT_TRY(make_dev_filter(filter, inputs, n_inputs, n, &f));
  if (keys[0].dtype == BOLT_DEC128 && n > 0) {
    DevBuf<uint32_t> err;
    uint32_t h = 0;
    BOLT_TRY(err.alloc(1, s));
    BOLT_TRY(fill_u32(err.ptr, 0, 1, s));
    dec_key_fit_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(static_cast<const uint64_t*>(keys[0].data),
                                                          keys[0].validity, n, err.ptr);
    BOLT_HIP(hipGetLastError());
    BOLT_TRY(read_back(s, {{&h, err.ptr, 4}}));
    if (h)
      return set_error(BOLT_DECLINE, "GROUP BY on a Decimal128 key with values beyond 64 bits (the host path takes it)");
  }

  // ---- pass A ----
  const int W = P.words;
  int S = lds_slots(lds_budget_bytes(), W, 4096);
  // a partition's table: as large as LDS allows, since every group of the
  // input is in one of them
  const int part_S = lds_slots(lds_max_bytes() - 1024, W, 8192);
  const bool use_lds = !(flags & BOLT_GROUPBY_FORCE_GLOBAL) && S >= 256 && n > 0;
  int64_t n_parts = 0, n_spill = 0;
  double est = 0;
  bool key_parts = false;  // the input was partitioned by key
  DevBuf<unsigned long long> pkeys, pwords;
  DevBuf<uint8_t> ptag;
  DevBuf<uint32_t> spill, hll, spill_seg;
  DevBuf<unsigned long long> spill_key;
  unsigned grid = 0;
  int64_t spill_per = 0;
  if (use_lds) {
    // the per-query generated kernel when hipRTC is available, else the
    // precompiled one; rows_per_iter is what one workgroup iteration covers
    hipFunction_t gfn = nullptr;
    GbJitSpec gs;
    JitLits glits;
    JitCols gcols;
    const bool jit = jit_enabled() && gb_jit_spec(ks, P, f, &gs, &glits, &gcols) == BOLT_OK;
    // more groups than one LDS table holds: the key partition first
    GbPartCopy pc;
    const KeySpec* pks = &ks;
    JitCols* pcols = &gcols;
    const uint32_t* ranges = nullptr;
    if (jit && parted) {
      bool yes = false;
      BOLT_TRY(gb_part_wanted(s, ks, f, n, S, part_S, &yes));
      *parted = yes;
      if (yes) BOLT_TRY(gb_part_copy(s, ks, gs, glits, gcols, n, part_S, &pc, &yes));
      if (yes && jit_get_keyed(gb_jit_key(pc.spec), [&] { return jit_gb_lds_source(pc.spec); }, &gfn) == BOLT_OK) {
        gs = pc.spec;
        pks = &pc.ks;
        pcols = &pc.cols;
        ranges = pc.ranges.ptr;
      } else {
        pc.bufs.clear();
      }
    }
    key_parts = ranges != nullptr;
    if (jit && !key_parts && jit_get_keyed(gb_jit_key(gs), [&] { return jit_gb_lds_source(gs); }, &gfn) != BOLT_OK)
      gfn = nullptr;
    clear_error();
    if (key_parts) S = part_S;
    const size_t lds = (size_t)(S + 2) * 8 * (1 + W) + (kHllRegs + 4) * 4;
    const int64_t rows_per_iter = (int64_t)kGbBlock * (gfn ? gs.unroll : 1);
    if (!gfn)
      BOLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gb_lds_kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    grid = key_parts ? 1u << kGbPartBits : grid_for(n, kGbBlock, 16, 256);
    const int64_t pcap = (int64_t)grid * (S + 2);
    // a workgroup handles at most ceil(n / (grid * rows_per_iter)) iterations
    spill_per = (n + (int64_t)grid * rows_per_iter - 1) / ((int64_t)grid * rows_per_iter) * rows_per_iter;
    BOLT_TRY(pkeys.alloc((size_t)pcap, s));
    BOLT_TRY(ptag.alloc((size_t)pcap, s));
    BOLT_TRY(pwords.alloc((size_t)pcap * (W > 0 ? W : 1), s));
    if (!key_parts) {  // partitions do not spill; if one does after all, the plain path runs instead
      BOLT_TRY(spill.alloc((size_t)grid * spill_per, s));
      BOLT_TRY(spill_seg.alloc(grid, s));
    }
    // inputs large enough for the partitioned tier: the spilled rows' keys are
    // captured beside the row ids (8 bytes more per spilled row, from a
    // register), so that tier's histogram and first scatter read them in
    // order instead of gathering them by row id
    if (n > ((int64_t)1 << 25) && !key_parts) BOLT_TRY(spill_key.alloc((size_t)grid * spill_per, s));
    // sketch registers and the two counters in one buffer: one read-back
    BOLT_TRY(hll.alloc(kHllRegs + 4, s));
    BOLT_TRY(fill_u32(hll.ptr, 0, kHllRegs + 4, s));
    unsigned long long* counters = reinterpret_cast<unsigned long long*>(hll.ptr + kHllRegs);
    PartOut po{pkeys.ptr, ptag.ptr, pwords.ptr, pcap, counters, spill.ptr, counters + 1, spill_seg.ptr,
               spill_per, hll.ptr, spill_key.ptr};
    prof_begin(s);
    if (gfn) {
      long long nn = n;
      int SSz = S;
      void* args[] = {&nn, &SSz, (void*)&pks->d0, (void*)&pks->v0, (void*)&pks->d1, (void*)&pks->v1, &glits, pcols, &po,
                      (void*)&ranges};
      BOLT_HIP(hipModuleLaunchKernel(gfn, grid, 1, 1, kGbBlock, 1, 1, (unsigned)lds, s, args, nullptr));
    } else {
      gb_lds_kernel<<<grid, kGbBlock, lds, s>>>(ks, f, P, n, S, po);
    }
    prof_end(s);
    BOLT_HIP(hipGetLastError());
    std::vector<uint32_t> regs(kHllRegs + 4);
    uint32_t declined = 0;
    if (key_parts)
      BOLT_TRY(read_back(s, {{regs.data(), hll.ptr, (kHllRegs + 4) * 4}, {&declined, ranges + (1 << kGbPartBits) + 1, 4}}));
    else
      BOLT_TRY(read_back(s, {{regs.data(), hll.ptr, (kHllRegs + 4) * 4}}));
    unsigned long long hc[2];
    memcpy(hc, regs.data() + kHllRegs, 16);
    n_parts = (int64_t)hc[0];
    n_spill = (int64_t)hc[1];
    est = hll_estimate(regs.data());
    if (key_parts && (declined || n_spill > 0)) return kGbPlain;  // more groups than the tables take
  } else {
    n_spill = n;  // every row goes to the global table
    est = (double)n;
  }

  // ---- pass B (global table) and pass C (extraction) ----
  // One host round trip for both: a table that overflowed is detected with
  // the extraction's results and the two passes rerun 4x larger.
  const int64_t upper = n_parts + n_spill;  // exact bound on the group count
  uint64_t want = (uint64_t)std::min<double>((double)upper, est * 1.25 + 64.0);
  uint64_t cap = next_pow2(std::max<uint64_t>(1024, 2 * want));
  if (const char* e = getenv("BOLT_GB_INITIAL_CAP")) {  // testing: force the overflow-and-rerun path
    const long long c = atoll(e);
    if (c >= 1024) cap = next_pow2((uint64_t)c);
  }
  bool has_var = false;
  for (int a = 0; a < P.n; a++) has_var |= P.a[a].kind == K_VAR;
  // many spilled rows over many groups: the radix-partitioned tier instead of
  // global atomics per spilled row (its records are built once, whatever the
  // table size).  Its passes cost a fixed ~2 ms more than the atomics save
  // below a few tens of millions of spilled rows (h2o q2 / q3 / q5 at 10M
  // rows: 5.0 / 3.8 / 5.6 ms partitioned, 3.0 / 3.0 / 4.4 ms with the global
  // table; 256M Zipf rows: 10.4 ms partitioned, 14.7 ms global), so it takes
  // over from 2^25 spilled rows.
  const bool partitioned = use_lds && n > 0 &&
                           ((flags & BOLT_GROUPBY_FORCE_PARTITIONED) ||
                            (n_spill > (int64_t)(1 << 25) && est > 0.75 * (double)S));
  // the partitioned tier writes each group once, with one claim, so its
  // table is sized for at most half load (1.6x the padded estimate) rather than
  // 2x: half the slots to initialise and for the extraction to scan
  if (partitioned && !getenv("BOLT_GB_INITIAL_CAP"))
    cap = next_pow2(std::max<uint64_t>(1024, (uint64_t)((double)want * 1.6)));
  GbPartitions parts;
  if (partitioned)
    BOLT_TRY(gb_part_build(s, ks, P, pkeys.ptr, ptag.ptr, pwords.ptr, (int64_t)pkeys.count, n_parts, spill.ptr,
                           spill_key.ptr, spill_per, spill_seg.ptr, (int)grid, n_spill, est, S,
                           part_bits_delta(est, W), &parts));
  t_last_plan = GbLastPlan{!use_lds ? 1 : (partitioned ? 2 : (n_spill > 0 ? 1 : 0)), n_spill, n_parts,
                           partitioned ? parts.np : 0, est_bucket(est), W};
  GTable t;
  DevBuf<unsigned long long> tkeys, twords;
  DevBuf<uint32_t> tmisc;
  BOLT_TRY(tmisc.alloc(8, s));
  bolt_table* tbl = nullptr;
  std::vector<bolt_column_t> cols(n_keys + n_aggs);
  DevBuf<unsigned long long> packed;
  DevBuf<uint32_t> slot_of;
  int64_t n_groups = 0;
  int st = BOLT_OK;
  const bool sorted = (flags & BOLT_GROUPBY_SORTED) != 0;
  const bool clash = ks.null_group && (keys[0].dtype == BOLT_I64 || keys[0].dtype == BOLT_DEC128);
  bool ordered = false;
  // every group in exactly one partial record: no table, the records are the groups
  const bool dense = key_parts && !ks.null_group && !has_var;
  for (int attempt = 0;; attempt++) {
    BOLT_TRY(fill_u32(tmisc.ptr, 0, 8, s));
    t.used_special = tmisc.ptr;
    t.err = tmisc.ptr + 4;
    if (dense) {
      t.keys = pkeys.ptr;
      t.words = pwords.ptr;
      t.cap = (uint64_t)n_parts;
    } else {
      BOLT_TRY(tkeys.alloc(cap, s));
      BOLT_TRY(twords.alloc((cap + 2) * (W > 0 ? W : 1), s));
      t.keys = tkeys.ptr;
      t.words = twords.ptr;
      t.cap = cap;
      gb_init_kernel<<<grid_for((int64_t)cap + 2, 256, 1), 256, 0, s>>>(t, P);
    }
    if (dense) {
    } else if (partitioned) {
      BOLT_TRY(gb_part_reduce(s, t, P, parts, S));
    } else if (n_parts > 0) {
      if (est < 0.75 * (double)S && n_parts > 4096) {
        // few groups: two-level merge through LDS tables of the same size
        const unsigned mgrid = (unsigned)std::min<int64_t>(64, (n_parts + 4095) / 4096);
        const size_t mlds = (size_t)(S + 2) * 8 * (1 + W) + 16;
        BOLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gb_merge_lds_kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)mlds));
        gb_merge_lds_kernel<<<mgrid, kGbBlock, mlds, s>>>(t, P, pkeys.ptr, ptag.ptr, pwords.ptr,
                                                          (int64_t)pkeys.count, n_parts, S);
      } else {  // also the key partition's records, one per group and workgroup
        gb_merge_parts_kernel<<<grid_for(n_parts, 256, 4), 256, 0, s>>>(t, P, pkeys.ptr, ptag.ptr, pwords.ptr,
                                                                        (int64_t)pkeys.count, n_parts);
      }
    }
    if (n_spill > 0 && !partitioned) {
      if (use_lds) {
        const int K = 16;  // blocks per spill segment
        gb_rows_seg_kernel<<<grid * K, 256, 0, s>>>(t, P, ks, spill.ptr, spill_per, spill_seg.ptr, K);
      } else {
        if (attempt == 0) prof_begin(s);
        gb_rows_kernel<<<grid_for(n_spill, 256, 4), 256, 0, s>>>(t, P, ks, f, nullptr, n_spill);
        if (attempt == 0) prof_end(s);
      }
    }
    if (has_var && n > 0) gb_m2_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(t, P, ks, f, n);
    BOLT_HIP(hipGetLastError());

    const uint64_t total = t.cap + 2;
    const int64_t out_cap = (int64_t)std::min<uint64_t>(total, (uint64_t)std::max<int64_t>(upper, 0) + 2);
    tbl = new bolt_table();
    tbl->stream = s;
    OutSpec o;
    memset(&o, 0, sizeof o);
    ordered = false;
    for (int k = 0; k < n_keys && st == BOLT_OK; k++) {
      st = table_alloc_col(tbl, keys[k].dtype, out_cap, k == 0 && ks.null_group, s, &cols[k]);
      cols[k].scale = keys[k].scale;
      o.key[k] = OutCol{static_cast<uint8_t*>(cols[k].data), (uint32_t*)cols[k].validity, keys[k].dtype, 0};
    }
    for (int a = 0; a < n_aggs && st == BOLT_OK; a++) {
      const GAgg& g = P.a[a];
      bool can_null = (g.nw >= 0 && g.kind != K_COUNT) ||
                      g.op == BOLT_AGG_VAR_SAMP || g.op == BOLT_AGG_STDDEV_SAMP;
      st = table_alloc_col(tbl, out_dt[a], out_cap, can_null, s, &cols[n_keys + a]);
      o.agg[a] = OutCol{static_cast<uint8_t*>(cols[n_keys + a].data), (uint32_t*)cols[n_keys + a].validity, out_dt[a], 0};
    }
    if (st == BOLT_OK) st = packed.alloc((size_t)out_cap, s);
    if (st == BOLT_OK) st = slot_of.alloc((size_t)out_cap, s);
    if (st != BOLT_OK) {
      bolt_table_release(tbl);
      return st;
    }
    o.packed = packed.ptr;
    o.slot_of = slot_of.ptr;
    if (dense && n_parts > 0)
      gb_extract_dense_kernel<<<grid_for(n_parts, 256, 1), 256, 0, s>>>(t, P, ks, o, n_parts, (size_t)pkeys.count);
    const bool small = total <= (1u << 20);
    const int64_t per_tile = (int64_t)kExBlock * (small ? 1 : kExItems);
    const int64_t tiles = (int64_t)((total + per_tile - 1) / per_tile);
    // look-back status words and the ticket / total in one buffer, one fill
    DevBuf<uint64_t> status;
    if ((st = status.alloc((size_t)tiles + 2, s)) != BOLT_OK ||
        (st = fill_u32(status.ptr, 0, ((size_t)tiles + 2) * 2, s)) != BOLT_OK) {
      bolt_table_release(tbl);
      return st;
    }
    uint32_t* emisc = reinterpret_cast<uint32_t*>(status.ptr + tiles);
    if (dense) {
    } else if (small)
      gb_extract_kernel<1><<<(unsigned)tiles, kExBlock, 0, s>>>(t, P, ks, o, status.ptr, emisc,
                                                               reinterpret_cast<unsigned long long*>(emisc + 2));
    else
      gb_extract_kernel<kExItems><<<(unsigned)tiles, kExBlock, 0, s>>>(
          t, P, ks, o, status.ptr, emisc, reinterpret_cast<unsigned long long*>(emisc + 2));
    // A table small enough for the rank sort is put in order before the host
    // learns the group count: one wait for both.
    if (sorted && !clash && total <= (uint64_t)kRankSortMax) {
      if ((st = order_groups(s, tbl, cols, packed.ptr, dense ? n_parts : (int64_t)total,
                             dense ? nullptr : reinterpret_cast<const unsigned long long*>(emisc + 2))) != BOLT_OK) {
        bolt_table_release(tbl);
        return st;
      }
      ordered = true;
    }
    hipError_t le = hipGetLastError();
    uint32_t eh[4] = {0, 0, 0, 0}, terr[4] = {0, 0, 0, 0};
    st = le == hipSuccess ? read_back(s, {{eh, emisc, 16}, {terr, t.err, 16}})
                          : set_error(BOLT_ERR_DEVICE, "GROUP BY extraction failed: %s", hipGetErrorString(le));
    if (st != BOLT_OK) {
      bolt_table_release(tbl);
      return st;
    }
    if (terr[0]) {  // the global table overflowed: discard this result and rerun larger
      bolt_table_release(tbl);
      tbl = nullptr;
      if (attempt >= 3 || cap >= (1ull << 33))
        return set_error(BOLT_ERR_MEMORY, "GROUP BY hash table overflow at %llu slots", (unsigned long long)cap);
      cap *= 4;
      continue;
    }
    n_groups = dense ? n_parts : (int64_t)(((uint64_t)eh[3] << 32) | eh[2]);
    if (terr[1]) {
      bolt_table_release(tbl);
      return set_error(BOLT_ERR_OTHER, "GROUP BY extraction look-back timed out");
    }
    if (terr[2] & 1u) {
      bolt_table_release(tbl);
      return set_error(BOLT_ERR_TYPE, "SUM(integer) overflow: accumulator exceeds i64 range");
    }
    if (terr[2] & 2u) {
      bolt_table_release(tbl);
      return set_error(BOLT_ERR_TYPE, "SUM(Decimal128) precision overflow: accumulator exceeds i128 range");
    }
    break;
  }

  if (clash && n_groups >= 2) {
    DevBuf<int64_t> clash;
    int64_t hc[2] = {-1, 0};
    st = clash.alloc(2, s);
    if (st == BOLT_OK) st = fill_u32(clash.ptr, 0xFFFFFFFFu, 2, s);
    if (st == BOLT_OK) st = fill_u32(reinterpret_cast<uint32_t*>(clash.ptr + 1), 0, 2, s);
    if (st == BOLT_OK) {
      gb_null_clash_kernel<<<grid_for(n_groups, 256, 4), 256, 0, s>>>(packed.ptr, slot_of.ptr, n_groups, cap,
                                                                     clash.ptr);
      if (hipGetLastError() != hipSuccess || hipMemcpyAsync(hc, clash.ptr, 16, hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess)
        st = set_error(BOLT_ERR_DEVICE, "GROUP BY NULL-group check failed");
    }
    if (st == BOLT_OK && hc[0] >= 0 && hc[1]) {
      MoveCols mc;
      memset(&mc, 0, sizeof mc);
      mc.n = (int32_t)cols.size();
      for (int c = 0; c < mc.n; c++) {
        mc.d[c] = static_cast<uint8_t*>(const_cast<void*>(cols[c].data));
        mc.v[c] = reinterpret_cast<uint32_t*>(const_cast<uint8_t*>(cols[c].validity));
        mc.w[c] = dtype_size(cols[c].dtype);
      }
      if (hc[0] != n_groups - 1)
        gb_move_row_kernel<<<1, 64, 0, s>>>(mc, packed.ptr, slot_of.ptr, hc[0], n_groups - 1);
      if (hipGetLastError() != hipSuccess) st = set_error(BOLT_ERR_DEVICE, "GROUP BY NULL-group removal failed");
      n_groups--;
    }
    if (st != BOLT_OK) {
      bolt_table_release(tbl);
      return st;
    }
  }

  // ---- ordering by packed key (src/exec/groupby.rs:800) ----
  if (sorted && n_groups > 1 && !ordered) {
    st = order_groups(s, tbl, cols, packed.ptr, n_groups, nullptr);
    if (st == BOLT_OK && hipStreamSynchronize(s) != hipSuccess) st = set_error(BOLT_ERR_DEVICE, "GROUP BY sort failed");
    if (st != BOLT_OK) {
      bolt_table_release(tbl);
      return st;
    }
  }
  for (auto& c : cols) c.length = n_groups;
  tbl->cols = cols;
  tbl->n_rows = n_groups;
  *out = tbl;
  return BOLT_OK;
}

extern "C" int bolt_groupby(bolt_stream_t stream, const bolt_column_t* keys, int32_t n_keys,
                            const bolt_column_t* inputs, int32_t n_inputs, const bolt_agg_t* aggs, int32_t n_aggs,
                            const bolt_filter_t* filter, uint32_t flags, bolt_table_t** out) {
  bool parted = false;
  int st = groupby_run(stream, keys, n_keys, inputs, n_inputs, aggs, n_aggs, filter, flags,
                       (flags & BOLT_GROUPBY_FORCE_PARTITIONED) ? nullptr : &parted, out);
  // the attempt's buffers are free again: what fits without the key partition
  // fits, wherever in the attempt the room ended
  if (st == kGbPlain || (parted && st == BOLT_ERR_MEMORY))
    st = groupby_run(stream, keys, n_keys, inputs, n_inputs, aggs, n_aggs, filter, flags, nullptr, out);
  return st;
}

extern "C" int bolt_groupby_last_plan(int32_t* tier, int64_t* spilled_rows, int64_t* partial_records,
                                      int32_t* partitions) {
  if (tier) *tier = bolt::t_last_plan.tier;
  if (spilled_rows) *spilled_rows = bolt::t_last_plan.spilled;
  if (partial_records) *partial_records = bolt::t_last_plan.partials;
  if (partitions) *partitions = bolt::t_last_plan.partitions;
  return BOLT_OK;
}

extern "C" int bolt_groupby_autotune_partitions(bolt_stream_t stream, const bolt_column_t* keys, int32_t n_keys,
                                                const bolt_column_t* inputs, int32_t n_inputs, const bolt_agg_t* aggs,
                                                int32_t n_aggs, int32_t reps, int32_t* best_partitions,
                                                float* best_ms) {
  using namespace bolt;
  if (reps < 1) reps = 1;
  double best = 1e300;
  int best_delta = 0, best_np = 0, key_bucket = 0, key_words = 0;
  int seen_np[5] = {-1, -1, -1, -1, -1};
  int st = BOLT_OK;
  for (int d = -2; d <= 2 && st == BOLT_OK; d++) {
    t_forcing = true;
    t_force_delta = d;
    double total = 0;
    for (int r = 0; r <= reps && st == BOLT_OK; r++) {  // one untimed call first (pool, code objects)
      bolt_table_t* t = nullptr;
      const auto t0 = std::chrono::steady_clock::now();
      st = bolt_groupby(stream, keys, n_keys, inputs, n_inputs, aggs, n_aggs, nullptr,
                        BOLT_GROUPBY_FORCE_PARTITIONED, &t);
      const auto t1 = std::chrono::steady_clock::now();
      if (t) bolt_table_release(t);
      if (r > 0) total += std::chrono::duration<double, std::milli>(t1 - t0).count();
    }
    t_forcing = false;
    if (st != BOLT_OK) break;
    const int np = t_last_plan.partitions;
    bool dup = false;  // a delta that clamps to a partition count already timed
    for (int k = 0; k < 5; k++) dup |= seen_np[k] == np;
    seen_np[d + 2] = np;
    key_bucket = t_last_plan.est_bucket;
    key_words = t_last_plan.words;
    if (!dup && total / reps < best) {
      best = total / reps;
      best_delta = d;
      best_np = np;
    }
  }
  t_forcing = false;
  if (st != BOLT_OK) return st;
  {
    std::lock_guard<std::mutex> lk(g_part_mu);
    g_part_delta[{key_bucket, key_words}] = best_delta;
  }
  if (best_partitions) *best_partitions = best_np;
  if (best_ms) *best_ms = (float)best;
  return BOLT_OK;
}
