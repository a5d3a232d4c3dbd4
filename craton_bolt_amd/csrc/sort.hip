// sort.hip — stable LSD radix sort of (64-bit key, u32 value) pairs, and
// the multi-column ORDER BY permutation built on it.
//
// Replaces run_radix_pipeline_i64 (src/exec/gpu_sort.rs:1493) and the
// histogram / scatter kernels (src/jit/sort_kernel_radix.rs:489,885), which
// use 4-bit digits (16 passes for int64) with a device-to-host histogram
// copy, a host scan and a host-to-device offset copy between passes.  Here:
//   * one up-front pass histograms all eight 8-bit digits at once (LDS
//     histograms, one global atomic per bin per block);
//   * each digit is then one "onesweep" pass (Adinets & Merrill, 2022): a
//     4096-key tile ranks its keys with wave64 ballot matching (8 ballots
//     per key give each key its set of same-digit peers), looks back across
//     earlier tiles per digit for its global offsets (decoupled look-back,
//     one digit per thread), reorders the tile by digit in LDS and writes
//     runs of equal digits with coalesced stores;
//   * passes whose digit is constant over the whole input are skipped; keys in
//     which few digits vary take a pass per digit (sort_by_bytes);
//   * others, up to 2^23 rows, and up to 2^25 where the top digits are uneven,
//     get buckets from a sample of the keys instead (sort_split.h);
//   * for larger inputs with three or more varying digits the sort is hybrid
//     (MSD-grouped, LSD-finished): only the two most significant varying
//     digits get global onesweep passes; they leave up to 65536 contiguous
//     buckets of ~n/65536 keys, which one workgroup each sorts by the
//     remaining bytes entirely in LDS and writes back once (Stehle &
//     Jacobsen's hybrid radix sort, 2017).  Three HBM round trips replace
//     eight for 64-bit keys.  Skewed inputs whose largest bucket exceeds the
//     LDS capacity fall back to plain LSD.
// Key transforms follow src/exec/gpu_sort.rs:1070-1180: signed integers flip
// the sign bit, floats use the IEEE-monotonic flip after canonicalising NaN
// (sorted last) and -0.0 (== +0.0), DESC is the bitwise NOT; for int64
// pairs the transform is an xor applied as the first pass loads and undone
// as the last one stores.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "bolt_internal.h"

namespace bolt {

constexpr int kRadixBits = 8;
constexpr int kBins = 1 << kRadixBits;
constexpr int kSortBlock = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortBlock * kSortItems;  // 4096 keys
constexpr int kSortWaves = kSortBlock / 64;
constexpr int kMaxPasses = 9;  // up to 72 key bits

constexpr uint32_t kSFlagAgg = 1u << 30;
constexpr uint32_t kSFlagInc = 2u << 30;
constexpr uint32_t kSValue = (1u << 30) - 1;

// ---- histogram of the digits -----------------------------------------------------

// Digits p < passes whose bit is set in `digits`.  Bound by its LDS atomics, one a
// key and digit.
__global__ __launch_bounds__(kSortBlock) void radix_hist_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                int passes, uint32_t digits,
                                                                uint32_t* __restrict__ hist, uint64_t in_xor) {
  __shared__ uint32_t h[kMaxPasses][kBins];
  for (int i = threadIdx.x; i < passes * kBins; i += kSortBlock) (&h[0][0])[i] = 0;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * kSortBlock;
  for (int64_t i = (int64_t)blockIdx.x * kSortBlock + threadIdx.x; i < n; i += stride) {
    uint64_t k = __builtin_nontemporal_load(keys + i) ^ in_xor;
    for (int p = 0; p < passes; p++)
      if ((digits >> p) & 1u) atomicAdd(&h[p][(k >> (p * kRadixBits)) & (kBins - 1)], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < passes * kBins; i += kSortBlock) {
    uint32_t v = (&h[0][0])[i];
    if (v) atomicAdd(&hist[i], v);
  }
}

// exclusive scan of each pass's 256 bins (one block per pass)
__global__ __launch_bounds__(kBins) void radix_scan_kernel(const uint32_t* __restrict__ hist,
                                                           uint32_t* __restrict__ offs) {
  __shared__ uint32_t s[kBins];
  const int p = blockIdx.x, t = threadIdx.x;
  s[t] = hist[p * kBins + t];
  __syncthreads();
  for (int d = 1; d < kBins; d <<= 1) {
    uint32_t v = t >= d ? s[t - d] : 0;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  offs[p * kBins + t] = s[t] - hist[p * kBins + t];
}

// ---- one onesweep pass ------------------------------------------------------------

// Where a pass finds a row's digit: 8 bits of the key, the low `shift` bits of
// its 16-bit code (the code's other bits are then carried along, for the next
// pass), or an 8-bit digit carried by the pass before.
enum { kDigitKey = 0, kDigitCode = 1, kDigitByte = 2 };

template <int SRC>
__global__ __launch_bounds__(kSortBlock) void radix_pass_kernel(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint64_t* __restrict__ kout,
    uint32_t* __restrict__ vout, int64_t n, int shift, const uint32_t* __restrict__ digit_base,
    uint32_t* __restrict__ status, uint32_t* __restrict__ ticket, uint32_t* __restrict__ err, uint64_t in_xor,
    uint64_t out_xor, const void* __restrict__ din, uint8_t* __restrict__ dout) {
  __shared__ uint64_t sk[kSortTile];
  __shared__ uint32_t sv[kSortTile];
  __shared__ uint32_t wh[kSortWaves][kBins];  // per-wave digit counts, then per-wave prefixes
  __shared__ uint32_t lex[kBins];             // tile-local exclusive digit offsets
  __shared__ uint32_t gb[kBins];              // global base of each digit's run in this tile
  __shared__ uint32_t wtot[kSortWaves];
  __shared__ uint32_t sh_tile;
  __shared__ uint16_t sd[SRC == kDigitKey ? 1 : kSortTile];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) sh_tile = atomicAdd(ticket, 1u);
  for (int i = threadIdx.x; i < kSortWaves * kBins; i += kSortBlock) (&wh[0][0])[i] = 0;
  __syncthreads();
  const int64_t tile = sh_tile;
  const int64_t tbase = tile * kSortTile;
  // wave w owns tile keys [w*64*ITEMS, (w+1)*64*ITEMS), item j covers 64
  // consecutive keys: input order = (wave, item, lane)
  uint64_t key[kSortItems];
  uint32_t val[kSortItems];
  uint16_t rank[kSortItems];
  uint16_t code[SRC == kDigitKey ? 1 : kSortItems];
  const uint32_t dmask = SRC == kDigitCode ? (1u << shift) - 1 : kBins - 1;
  auto digit = [&](int j) -> uint32_t {
    if constexpr (SRC == kDigitKey) return (uint32_t)(key[j] >> shift) & (kBins - 1);
    else return code[j] & dmask;
  };
  // branch-free loads (clamped index) so all 2 x ITEMS loads are in flight at
  // once; out-of-range lanes become ~0 (last digit) and are never stored
#pragma unroll
  for (int j = 0; j < kSortItems; j++) {
    const int64_t i = tbase + (int64_t)wave * 64 * kSortItems + j * 64 + lane;
    const int64_t ic = i < n ? i : n - 1;
    key[j] = __builtin_nontemporal_load(kin + ic);
    val[j] = __builtin_nontemporal_load(vin + ic);
    if constexpr (SRC == kDigitCode) code[j] = static_cast<const uint16_t*>(din)[ic];
    if constexpr (SRC == kDigitByte) code[j] = static_cast<const uint8_t*>(din)[ic];
  }
#pragma unroll
  for (int j = 0; j < kSortItems; j++) {
    const int64_t i = tbase + (int64_t)wave * 64 * kSortItems + j * 64 + lane;
    key[j] = i < n ? key[j] ^ in_xor : ~0ull;
    if constexpr (SRC != kDigitKey) code[j] = i < n ? code[j] : (uint16_t)0xFFFF;
  }
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int j = 0; j < kSortItems; j++) {
    const uint32_t d = digit(j);
    uint64_t peers = ~0ull;
#pragma unroll
    for (int b = 0; b < kRadixBits; b++) {
      uint64_t m = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? m : ~m;
    }
    const int leader = __builtin_ctzll(peers);
    uint32_t old = 0;
    if (lane == leader) {
      old = wh[wave][d];
      wh[wave][d] = old + (uint32_t)__popcll(peers);
    }
    old = __shfl(old, leader);
    rank[j] = (uint16_t)(old + (uint32_t)__popcll(peers & lt));
  }
  __syncthreads();
  // thread t owns digit t: wave prefixes and the tile's count, published at
  // once so that later tiles' look-backs find it early
  const int t = threadIdx.x;
  uint32_t cnt = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; w++) {
    uint32_t c = wh[w][t];
    wh[w][t] = cnt;
    cnt += c;
  }
  // The status word holds its whole payload, so relaxed device-scope atomics
  // suffice (acquire / release at agent scope would invalidate / write back
  // the per-XCD L2).
  uint32_t* st = status + (size_t)tile * kBins + t;
  __hip_atomic_store(st, (tile == 0 ? kSFlagInc : kSFlagAgg) | cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // exclusive scan of the 256 digit counts (4 waves x 64 digits, shuffles)
  {
    uint32_t inc = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t v = __shfl_up(inc, d);
      if (lane >= d) inc += v;
    }
    if (lane == 63) wtot[wave] = inc;
    lex[t] = inc - cnt;
  }
  __syncthreads();
  {
    uint32_t add = 0;
    for (int k = 0; k < wave; k++) add += wtot[k];
    lex[t] += add;
  }
  // decoupled look-back for digit t, four predecessors per round trip
  uint32_t prefix = 0;
  if (tile > 0) {
    int64_t pt = tile - 1;
    uint32_t spins = 0;
    bool done = false;
    while (!done) {
      uint32_t v[4];
#pragma unroll
      for (int q = 0; q < 4; q++)
        v[q] = pt - q >= 0 ? __hip_atomic_load(status + (size_t)(pt - q) * kBins + t, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)
                           : kSFlagInc;  // before tile 0: an inclusive zero
      int q = 0;
      for (; q < 4; q++) {
        const uint32_t fl = v[q] & ~kSValue;
        if (fl == 0) break;  // not published yet: wait on this one
        prefix += v[q] & kSValue;
        if (fl == kSFlagInc) {
          done = true;
          break;
        }
      }
      if (done) break;
      pt -= q;
      if (q < 4) {
        if (++spins > (1u << 24)) {
          atomicOr(err, 1u);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __hip_atomic_store(st, kSFlagInc | (prefix + cnt), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  gb[t] = digit_base[t] + prefix;
  __syncthreads();
  // reorder the tile by digit in LDS (stable: rank follows input order)
#pragma unroll
  for (int j = 0; j < kSortItems; j++) {
    int64_t i = tbase + (int64_t)wave * 64 * kSortItems + j * 64 + lane;
    if (i < n) {
      const uint32_t d = digit(j);
      const uint32_t pos = lex[d] + wh[wave][d] + rank[j];
      sk[pos] = key[j];
      sv[pos] = val[j];
      if constexpr (SRC != kDigitKey) sd[pos] = code[j];
    }
  }
  __syncthreads();
  const int64_t valid = n - tbase < kSortTile ? n - tbase : kSortTile;
#pragma unroll
  for (int j = 0; j < kSortItems; j++) {
    const int i = j * kSortBlock + threadIdx.x;
    if (i < valid) {
      const uint64_t k = sk[i];
      const uint32_t d = SRC == kDigitKey ? (uint32_t)(k >> shift) & (kBins - 1) : sd[i] & dmask;
      const uint64_t dst = (uint64_t)gb[d] + (uint32_t)i - lex[d];
      kout[dst] = k ^ out_xor;
      vout[dst] = sv[i];
      if constexpr (SRC == kDigitCode)
        if (dout) dout[dst] = (uint8_t)(sd[i] >> shift);
    }
  }
}

__global__ void copy_pairs_kernel(const uint64_t* __restrict__ ki, const uint32_t* __restrict__ vi,
                                  uint64_t* __restrict__ ko, uint32_t* __restrict__ vo, int64_t n, uint64_t x) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    ko[i] = ki[i] ^ x;
    vo[i] = vi[i];
  }
}

// ---- hybrid tail: per-bucket LDS sort ------------------------------------------------
//
// After two stable global passes on the two most significant varying digits
// (p1 < p2), the keys form up to 65536 contiguous buckets, one per (digit p2,
// digit p1) pair, and every bit above byte p1 other than those two digits is
// constant.  One workgroup then sorts each bucket entirely in LDS by the
// remaining low bytes (stable LSD, skipping bytes that are constant within the
// bucket) and writes it once: three HBM round trips instead of one per digit.

constexpr int kLocBlock = 512;
constexpr int kLocItems = 11;
constexpr int kLocMax = kLocBlock * kLocItems;  // 5632 keys per bucket
constexpr int kLocWaves = kLocBlock / 64;
constexpr int kBuckets = 1 << 16;

__device__ __forceinline__ uint32_t bucket_of(uint64_t k, int s1, int s2) {
  return (uint32_t)((((k >> s2) & 255) << 8) | ((k >> s1) & 255));
}

// start[b] = first index whose bucket is >= b (b = 0 .. 65536); *max_size =
// the largest bucket.  keys ^ x are sorted by bucket.
__global__ void bucket_bounds_kernel(const uint64_t* __restrict__ keys, int64_t n, uint64_t x, int s1, int s2,
                                     uint32_t* __restrict__ start, uint32_t* __restrict__ max_size) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b > kBuckets) return;
  auto lower = [&](uint32_t target) -> int64_t {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (bucket_of(keys[mid] ^ x, s1, s2) < target) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  const int64_t s0 = b < kBuckets ? lower((uint32_t)b) : n;
  start[b] = (uint32_t)s0;
  if (b < kBuckets) {
    const int64_t e = b + 1 < kBuckets ? lower((uint32_t)(b + 1)) : n;
    atomicMax(max_size, (uint32_t)(e - s0));
  }
}

__global__ __launch_bounds__(kLocBlock) void local_sort_kernel(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint64_t* __restrict__ kout,
    uint32_t* __restrict__ vout, const uint32_t* __restrict__ start, int low_bits, uint32_t byte_mask,
    uint64_t out_xor, uint32_t* __restrict__ err) {
  __shared__ uint64_t sk[kLocMax];
  __shared__ uint32_t sv[kLocMax];
  __shared__ uint32_t wh[kLocWaves][kBins];
  __shared__ uint32_t lex[kBins];
  __shared__ uint32_t wtot[4];
  __shared__ uint32_t wtot8[kLocWaves];
  __shared__ uint32_t sh_max;
  __shared__ uint64_t red[2][kLocWaves];
  const uint32_t s0 = start[blockIdx.x];
  const int size = (int)(start[blockIdx.x + 1] - s0);
  if (size <= 0) return;
  if (size > kLocMax) {  // the host checks the largest bucket first; never write out of range
    if (threadIdx.x == 0) atomicOr(err, 2u);
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t low_mask = (1ull << low_bits) - 1;  // low_bits <= 48
  const uint64_t top = kin[s0] & ~low_mask;           // constant over the bucket
  // element order: (wave, item, lane); w = (low bits << 16) | element index
  uint64_t w[kLocItems];
  uint32_t vv[kLocItems];
  uint64_t a = ~0ull, o = 0;
  // branch-free (clamped) loads first, so they are all in flight together
#pragma unroll
  for (int j = 0; j < kLocItems; j++) {
    const int i = wave * 64 * kLocItems + j * 64 + lane;
    const int ic = i < size ? i : size - 1;
    w[j] = kin[s0 + ic];
    vv[j] = vin[s0 + ic];
  }
#pragma unroll
  for (int j = 0; j < kLocItems; j++) {
    const int i = wave * 64 * kLocItems + j * 64 + lane;
    const uint64_t low = w[j] & low_mask;
    const bool in = i < size;
    a &= in ? low : ~0ull;
    o |= in ? low : 0ull;
    w[j] = in ? ((low << 16) | (uint64_t)i) : ~0ull;  // out-of-range: after every element of the bucket
    if (in) sv[i] = vv[j];
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    a &= __shfl_xor(a, m);
    o |= __shfl_xor(o, m);
  }
  if (lane == 0) {
    red[0][wave] = a;
    red[1][wave] = o;
  }
  __syncthreads();
  uint64_t varying = 0;
  {
    uint64_t ra = ~0ull, ro = 0;
    for (int k = 0; k < kLocWaves; k++) {
      ra &= red[0][k];
      ro |= red[1][k];
    }
    varying = ra ^ ro;
  }
  const int t = threadIdx.x;
  // ---- fast path: one counting pass on the 11 bits below the bucket's top
  // varying bit (sub-buckets of ~size/2048 keys), then an insertion sort of
  // each sub-bucket by the whole packed word; its low 16 bits are the
  // element's position, so equal keys keep their input order (stable) even
  // though the atomic scatter is not.  Buckets with a sub-bucket above 64
  // keys (heavy duplicates) take the LSD passes below instead.
  if (varying != 0) {
    const int h = 63 - __clzll(varying);
    const int dsh = 16 + (h >= 10 ? h - 10 : 0);
    uint32_t* cnt = &wh[0][0];  // 2048 counters
    for (int i = t; i < kLocWaves * kBins; i += kLocBlock) cnt[i] = 0;
    if (t == 0) sh_max = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLocItems; j++)
      if (w[j] != ~0ull) atomicAdd(&cnt[(uint32_t)(w[j] >> dsh) & 2047u], 1u);
    __syncthreads();
    {
      const uint32_t c0 = cnt[4 * t], c1 = cnt[4 * t + 1], c2 = cnt[4 * t + 2], c3 = cnt[4 * t + 3];
      const uint32_t local = c0 + c1 + c2 + c3;
      uint32_t inc = local;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(inc, d);
        if (lane >= d) inc += v;
      }
      if (lane == 63) wtot8[wave] = inc;
      const uint32_t mx = max(max(c0, c1), max(c2, c3));
      if (mx) atomicMax(&sh_max, mx);
      __syncthreads();
      uint32_t carry = 0;
      for (int k = 0; k < wave; k++) carry += wtot8[k];
      const uint32_t ex = carry + inc - local;
      cnt[4 * t] = ex;
      cnt[4 * t + 1] = ex + c0;
      cnt[4 * t + 2] = ex + c0 + c1;
      cnt[4 * t + 3] = ex + c0 + c1 + c2;
    }
    __syncthreads();
    if (sh_max <= 64u) {  // block-uniform
#pragma unroll
      for (int j = 0; j < kLocItems; j++)
        if (w[j] != ~0ull) sk[atomicAdd(&cnt[(uint32_t)(w[j] >> dsh) & 2047u], 1u)] = w[j];
      __syncthreads();
      // cnt[d] is now the end of sub-bucket d (= the start of d + 1)
      for (int d = t; d < 2048; d += kLocBlock) {
        const int b = d ? (int)cnt[d - 1] : 0, e = (int)cnt[d];
        for (int x = b + 1; x < e; x++) {
          const uint64_t v = sk[x];
          int y = x - 1;
          while (y >= b && sk[y] > v) {
            sk[y + 1] = sk[y];
            y--;
          }
          sk[y + 1] = v;
        }
      }
      __syncthreads();
      for (int i = t; i < size; i += kLocBlock) {
        const uint64_t ww = sk[i];
        kout[s0 + i] = (top | (ww >> 16)) ^ out_xor;
        vout[s0 + i] = sv[(uint32_t)(ww & 0xFFFF)];
      }
      return;
    }
  }
  // ---- general path: stable LSD over the bytes that vary in this bucket
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int q = 0; q * 8 < low_bits; q++) {
    if (!((byte_mask >> q) & 1u) || ((varying >> (8 * q)) & 255) == 0) continue;  // block-uniform
    const int shift = 16 + 8 * q;
    for (int i = t; i < kLocWaves * kBins; i += kLocBlock) (&wh[0][0])[i] = 0;
    __syncthreads();
    // rank within the wave: peers by ballot matching; the per-wave digit
    // counters are bumped with returning LDS atomics issued for all items
    // back to back (LDS keeps a wave's operations in order, so ranks stay
    // stable) and read once afterwards
    uint32_t rank[kLocItems], oldv[kLocItems];
    int lead[kLocItems];
#pragma unroll
    for (int j = 0; j < kLocItems; j++) {
      const uint32_t d = (uint32_t)(w[j] >> shift) & (kBins - 1);
      uint64_t peers = ~0ull;
#pragma unroll
      for (int bit = 0; bit < kRadixBits; bit++) {
        const uint64_t m = __ballot((d >> bit) & 1u);
        peers &= ((d >> bit) & 1u) ? m : ~m;
      }
      lead[j] = __builtin_ctzll(peers);
      rank[j] = (uint32_t)__popcll(peers & lt);
      oldv[j] = 0;
      if (lane == lead[j]) oldv[j] = atomicAdd(&wh[wave][d], (uint32_t)__popcll(peers));
    }
#pragma unroll
    for (int j = 0; j < kLocItems; j++) rank[j] += __shfl(oldv[j], lead[j]);
    __syncthreads();
    // digit t: exclusive offsets per wave, then an exclusive scan over the
    // 256 digits (waves 0..3 scan 64 digits each with shuffles)
    if (t < kBins) {
      uint32_t cnt = 0;
#pragma unroll
      for (int k = 0; k < kLocWaves; k++) {
        const uint32_t c = wh[k][t];
        wh[k][t] = cnt;
        cnt += c;
      }
      uint32_t inc = cnt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(inc, d);
        if (lane >= d) inc += v;
      }
      if (lane == 63) wtot[wave] = inc;
      lex[t] = inc - cnt;
    }
    __syncthreads();
    if (t < kBins) {
      uint32_t add = 0;
      for (int k = 0; k < (t >> 6); k++) add += wtot[k];
      lex[t] += add;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLocItems; j++) {
      const uint32_t d = (uint32_t)(w[j] >> shift) & (kBins - 1);
      sk[lex[d] + wh[wave][d] + rank[j]] = w[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLocItems; j++) w[j] = sk[wave * 64 * kLocItems + j * 64 + lane];
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kLocItems; j++) {
    const int i = wave * 64 * kLocItems + j * 64 + lane;
    if (i < size) {
      kout[s0 + i] = (top | (w[j] >> 16)) ^ out_xor;
      vout[s0 + i] = sv[(uint32_t)(w[j] & 0xFFFF)];
    }
  }
}

}  // namespace bolt

#include "sort_split.h"

namespace bolt {

// Buckets of at most 384 rows on average (512 in one pass and above 3 << 23
// rows), most of which the first bucket kernel holds.
static int split_code_bits(int64_t n) {
  const bool one = n <= kSplitOnePass;
  int cbits = one ? 6 : 9;  // 6: the splitters of one sorted list, no merge
  while (((int64_t)(one ? 512 : 384) << cbits) < n && cbits < 16) cbits++;
  return cbits;
}
static int split_samples(int64_t n) {
  const int cbits = split_code_bits(n);
  return cbits == 6 ? kSampleList : cbits <= 12 ? 4096 : 16384;
}
// A sort's sample: S keys in sorted lists, then as one list.
struct SplitSample {
  DevBuf<uint64_t> keys;  // [2 S]
  const uint64_t* sorted = nullptr;
};
// Draws the sample; `vary` workgroups more look for varying bits.
static int split_sample(hipStream_t s, const uint64_t* keys, int64_t n, uint64_t in_xor, SplitSample& sample,
                        uint64_t* one_zero, int vary) {
  const int S = split_samples(n);
  BOLT_TRY(sample.keys.alloc((size_t)2 * S, s));
  split_sample_kernel<<<S / kSampleList + vary, kSampleList, 0, s>>>(keys, n, in_xor, S, sample.keys.ptr, one_zero);
  BOLT_HIP(hipGetLastError());
  return BOLT_OK;
}
// Draws it unless that is done, and merges its lists.
static int split_sorted_sample(hipStream_t s, const uint64_t* keys, int64_t n, uint64_t in_xor, SplitSample& sample) {
  if (sample.sorted) return BOLT_OK;
  if (!sample.keys.ptr) BOLT_TRY(split_sample(s, keys, n, in_xor, sample, nullptr, 0));
  const int S = split_samples(n);
  uint64_t* lists = sample.keys.ptr;
  if (S > 4096) split_merge_kernel<16><<<S / 64, 64, 0, s>>>(lists, lists + S);
  else if (S > kSampleList) split_merge_kernel<4><<<S / 64, 64, 0, s>>>(lists, lists + S);
  BOLT_HIP(hipGetLastError());
  sample.sorted = S > kSampleList ? lists + S : lists;
  return BOLT_OK;
}
// Rows that share a value, by the sample, if the values are about equally
// frequent.
static int split_rows_per_value(hipStream_t s, const uint64_t* keys, int64_t n, uint64_t in_xor, SplitSample& sample,
                                double* rows) {
  const int S = split_samples(n);
  DevBuf<uint32_t> out;
  uint32_t distinct = 0;
  BOLT_TRY(out.alloc(1, s));
  BOLT_TRY(split_sorted_sample(s, keys, n, in_xor, sample));
  split_distinct_kernel<<<1, 1024, 0, s>>>(sample.sorted, S, out.ptr);
  BOLT_HIP(hipGetLastError());
  BOLT_TRY(read_back(s, {{&distinct, out.ptr, 4}}));
  *rows = (double)n / sample_groups(S, distinct);
  return BOLT_OK;
}

// The splitter sort of 2 <= n <= kSplitMax pairs (`sample` may be drawn).  *done = false when a bucket
// of different keys exceeded the LDS sort (keys_out / vals_out then hold
// nothing of use; the inputs are untouched).
static int split_sort_u64_pairs(hipStream_t s, const uint64_t* keys_in, const uint32_t* vals_in, int64_t n,
                                uint64_t* keys_out, uint32_t* vals_out, uint64_t in_xor, uint64_t out_xor,
                                SplitSample& sample, bool* done) {
  *done = true;
  if (n <= kSplitWhole) {
    split_whole_kernel<<<1, 1024, 0, s>>>(keys_in, vals_in, keys_out, vals_out, (int)n, in_xor, out_xor);
    BOLT_HIP(hipGetLastError());
    return BOLT_OK;
  }
  const bool one = n <= kSplitOnePass;
  const int cbits = split_code_bits(n), C = 1 << cbits;
  const int b1 = one ? 8 : cbits / 2;
  const int S = split_samples(n);
  const int64_t tiles = (n + kSortTile - 1) / kSortTile;
  DevBuf<uint64_t> ktmp;
  DevBuf<uint32_t> vtmp, words, start;
  DevBuf<uint16_t> codes;
  DevBuf<uint8_t> digits;
  BOLT_TRY(split_sorted_sample(s, keys_in, n, in_xor, sample));
  BOLT_TRY(codes.alloc((size_t)n, s));
  // counts, scanned counts, tickets and error, then the look-back words of
  // each pass: one fill
  const size_t status_words = (size_t)tiles * kBins;
  const size_t head = 512 + 514 + 6;
  BOLT_TRY(words.alloc(head + status_words * (one ? 1 : 2), s));
  BOLT_TRY(fill_u32(words.ptr, 0, head + status_words * (one ? 1 : 2), s));
  uint32_t* hist = words.ptr;
  uint32_t* offs = words.ptr + 512;
  uint32_t* misc = offs + 514;
  uint32_t* status = words.ptr + head;
  const Splitters sp{sample.sorted, S, std::min(C, S), std::max(cbits - 14, 0)};
  const size_t lds = (size_t)(sp.G + 1) * 8;
  BOLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(split_code_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  split_code_kernel<<<grid_for(n, kCodeBlock, 4, sp.G > 8192 ? 256 : 512), kCodeBlock, lds, s>>>(
      keys_in, n, in_xor, sp, b1, codes.ptr, hist);
  split_scan_kernel<<<2, 256, 0, s>>>(hist, offs);
  const uint32_t* starts = offs;
  if (one) {
    radix_pass_kernel<kDigitCode><<<(unsigned)tiles, kSortBlock, 0, s>>>(keys_in, vals_in, keys_out, vals_out, n, b1,
                                                                        offs, status, misc, misc + 4, in_xor, out_xor,
                                                                        codes.ptr, nullptr);
  } else {
    BOLT_TRY(ktmp.alloc((size_t)n, s));
    BOLT_TRY(vtmp.alloc((size_t)n, s));
    BOLT_TRY(digits.alloc((size_t)n, s));
    BOLT_TRY(start.alloc((size_t)C + 1, s));
    radix_pass_kernel<kDigitCode><<<(unsigned)tiles, kSortBlock, 0, s>>>(keys_in, vals_in, ktmp.ptr, vtmp.ptr, n, b1,
                                                                        offs, status, misc, misc + 4, in_xor, 0,
                                                                        codes.ptr, digits.ptr);
    radix_pass_kernel<kDigitByte><<<(unsigned)tiles, kSortBlock, 0, s>>>(
        ktmp.ptr, vtmp.ptr, keys_out, vals_out, n, 0, offs + 257, status + status_words, misc + 1, misc + 4, 0,
        out_xor, digits.ptr, nullptr);
    split_bounds_kernel<<<C / 256 + 1, 256, 0, s>>>(keys_out, n, out_xor, sp, C, start.ptr);
    starts = start.ptr;
  }
  launch_bucket_sorts(keys_out, vals_out, starts, C, sp, out_xor, misc + 5, s);
  BOLT_HIP(hipGetLastError());
  uint32_t e[2] = {0, 0};
  BOLT_TRY(read_back(s, {{e, misc + 4, 8}}));
  if (e[0]) return set_error(BOLT_ERR_OTHER, "radix sort look-back timed out");
  *done = e[1] == 0;
  return BOLT_OK;
}

// The calling thread's last sort (bolt_sort_last_plan).
static thread_local bolt_sort_plan_t t_sort_plan = BOLT_SORT_COPY;
static thread_local int t_sort_passes = 0;
static void set_sort_plan(bolt_sort_plan_t plan, int passes) {
  t_sort_plan = plan;
  t_sort_passes = passes;
}

// Whether keys of np varying bytes are sorted by a onesweep pass per byte, n
// between kSplitOnePass and kSplitMax.  A pass costs 15 us at 150,000 rows, 30 at
// 1M, 60 at 5M and 120 at 20M, whatever the values; the splitter sort's cost
// hardly depends on the bytes, but grows with the rows that share a value.  By
// bytes / by splitters in us: 2,500 values (two bytes) 123 / 161 at 150,000 rows,
// 148 / 275 at 1M, 241 / 351 at 5M, 808 / 1393 at 20M; 2^17 values (three) 171 /
// 302 at 1M, 302 / 647 at 5M; 2^24 (three) 145 / 140 at 150,000, 166 / 195 at 1M;
// 2^32 (four) 157 / 144 at 150,000, 189 / 202 at 1M, 356 / 421 at 5M; 2^40 (five)
// 203 / 198 at 1M.  Above 2^23 rows a pass is cheaper still against the splitters
// (2^25 values, four bytes, 1059 / 1547 at 20M; a float, eight, 1520 / 1315).
static bool sort_by_bytes(int64_t n, int np) {
  if (n > kSplitFirst) return np <= 6;
  return np <= 2 || (np == 3 && n >= (1 << 18)) || (np == 4 && n >= (1 << 19));
}

// Sort (keys_in, vals_in) ascending by key ^ in_xor, stable, writing
// (key image ^ out_xor, value) to keys_out / vals_out.  The bits of the keys from
// key_bits up are the same in every key.  Inputs are not modified and must not
// alias the outputs.
int radix_sort_u64_pairs(hipStream_t s, const uint64_t* keys_in, const uint32_t* vals_in, int64_t n,
                         uint64_t* keys_out, uint32_t* vals_out, int key_bits, uint64_t in_xor, uint64_t out_xor) {
  if (n <= 0) return BOLT_OK;
  if (n >= (1ll << 30)) return set_error(BOLT_ERR_PLAN, "radix sort: %lld keys exceeds the 2^30 limit", (long long)n);
  const int passes = (key_bits + kRadixBits - 1) / kRadixBits;
  if (passes < 1 || passes > kMaxPasses) return set_error(BOLT_ERR_PLAN, "radix sort: bad key width %d", key_bits);
  const bool grouped = getenv("BOLT_SORT_LSD") == nullptr;
  SplitSample sample;
  auto split = [&](bool* done) -> int {
    BOLT_TRY(split_sort_u64_pairs(s, keys_in, vals_in, n, keys_out, vals_out, in_xor, out_xor, sample, done));
    if (*done) set_sort_plan(n <= kSplitWhole ? BOLT_SORT_WORKGROUP : BOLT_SORT_SAMPLE, 0);
    return BOLT_OK;
  };
  // Up to kSplitFirst rows the splitter sort, unless a pass over the keys beside
  // the sample (uniform keys 197 -> 206 us at 1M rows) finds few bytes that vary;
  // above, the histogram of all bytes decides (30M uniform keys: 1.08 ms by
  // digits, 1.84 ms by splitters).
  std::vector<int> todo;  // varying bytes
  bool known = false;
  if (n > kSplitOnePass && n <= kSplitFirst && grouped) {
    DevBuf<uint64_t> one_zero;
    uint64_t b[2 * kVaryGrid], one = 0, zero = 0;
    const int vary = (int)grid_for(n, kSampleList, kVaryRows, kVaryGrid);
    BOLT_TRY(one_zero.alloc(2 * kVaryGrid, s));
    BOLT_TRY(split_sample(s, keys_in, n, in_xor, sample, one_zero.ptr, vary));
    BOLT_TRY(read_back(s, {{b, one_zero.ptr, (size_t)vary * 16}}));
    for (int g = 0; g < vary; g++) {
      one |= b[2 * g];
      zero |= b[2 * g + 1];
    }
    for (int p = 0; p < passes; p++)
      if (((one & zero) >> (p * kRadixBits)) & (kBins - 1)) todo.push_back(p);
    known = true;
  }
  if (n <= kSplitFirst && grouped && !(known && sort_by_bytes(n, (int)todo.size()))) {
    bool done = false;
    BOLT_TRY(split(&done));
    if (done) return BOLT_OK;
    // a bucket too large for LDS: LSD passes from the input
  }
  auto copy_all = [&]() -> int {  // equal keys
    copy_pairs_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(keys_in, vals_in, keys_out, vals_out, n, in_xor ^ out_xor);
    BOLT_HIP(hipGetLastError());
    set_sort_plan(BOLT_SORT_COPY, 0);
    return BOLT_OK;
  };
  if (known && todo.empty()) return copy_all();
  DevBuf<uint32_t> hist, offs, misc;
  BOLT_TRY(hist.alloc((size_t)passes * kBins, s));
  BOLT_TRY(offs.alloc((size_t)passes * kBins, s));
  BOLT_TRY(misc.alloc(4, s));
  BOLT_TRY(fill_u32(hist.ptr, 0, (size_t)passes * kBins, s));
  uint32_t digits = known ? 0u : ~0u;
  for (int p : todo) digits |= 1u << p;
  radix_hist_kernel<<<grid_for(n, kSortBlock, 16, 2048), kSortBlock, 0, s>>>(keys_in, n, passes, digits, hist.ptr,
                                                                            in_xor);
  radix_scan_kernel<<<passes, kBins, 0, s>>>(hist.ptr, offs.ptr);
  BOLT_HIP(hipGetLastError());
  std::vector<uint32_t> h((size_t)passes * kBins);
  if (!known) {
    BOLT_TRY(read_back(s, {{h.data(), hist.ptr, h.size() * 4}}));
    for (int p = 0; p < passes; p++) {
      bool trivial = false;
      for (int b = 0; b < kBins; b++)
        if (h[(size_t)p * kBins + b] == (uint32_t)n) trivial = true;
      if (!trivial) todo.push_back(p);
    }
    if (todo.empty()) return copy_all();
  }
  const int64_t tiles = (n + kSortTile - 1) / kSortTile;
  DevBuf<uint64_t> ktmp;
  DevBuf<uint32_t> vtmp, status;
  BOLT_TRY(ktmp.alloc((size_t)n, s));
  BOLT_TRY(vtmp.alloc((size_t)n, s));
  BOLT_TRY(status.alloc((size_t)tiles * kBins, s));
  auto pass = [&](const uint64_t* ksrc, const uint32_t* vsrc, uint64_t* kdst, uint32_t* vdst, int p, uint64_t ix,
                  uint64_t ox) -> int {
    BOLT_TRY(fill_u32(status.ptr, 0, (size_t)tiles * kBins, s));
    BOLT_TRY(fill_u32(misc.ptr, 0, 4, s));
    radix_pass_kernel<kDigitKey><<<(unsigned)tiles, kSortBlock, 0, s>>>(
        ksrc, vsrc, kdst, vdst, n, p * kRadixBits, offs.ptr + (size_t)p * kBins, status.ptr, misc.ptr, misc.ptr + 1,
        ix, ox, nullptr, nullptr);
    BOLT_HIP(hipGetLastError());
    return BOLT_OK;
  };
  auto check_lookback = [&]() -> int {
    uint32_t e = 0;
    BOLT_TRY(read_back(s, {{&e, misc.ptr + 1, 4}}));
    if (e) return set_error(BOLT_ERR_OTHER, "radix sort look-back timed out");
    return BOLT_OK;
  };
  const int np = (int)todo.size();
  if (n > kSplitFirst && n <= 2 * kSplitMax && grouped) {
    // largest bucket of the top two varying digits if they were independent
    double most = (double)n;
    for (int q = np - 1; q >= 0 && q >= np - 2; q--)
      most *= (double)*std::max_element(h.begin() + (size_t)todo[q] * kBins, h.begin() + (size_t)(todo[q] + 1) * kBins) /
              (double)n;
    // three bytes up to kSplitMax: their passes (929 us for 20M rows, 1043 here)
    if (np >= (n <= kSplitMax ? 4 : 3) && most <= 0.8 * kSplitMid) {
      const int p1 = todo[np - 2], p2 = todo[np - 1];
      BOLT_TRY(pass(keys_in, vals_in, ktmp.ptr, vtmp.ptr, p1, in_xor, 0));
      BOLT_TRY(pass(ktmp.ptr, vtmp.ptr, keys_out, vals_out, p2, 0, out_xor));
      DevBuf<uint32_t> starts;
      BOLT_TRY(starts.alloc(kBuckets + 1, s));
      BOLT_TRY(fill_u32(misc.ptr + 2, 0, 2, s));
      bucket_bounds_kernel<<<(kBuckets + 1 + 255) / 256, 256, 0, s>>>(keys_out, n, out_xor, p1 * kRadixBits,
                                                                    p2 * kRadixBits, starts.ptr, misc.ptr + 2);
      BOLT_TRY(fill_u32(misc.ptr + 2, 0, 1, s));
      launch_bucket_sorts(keys_out, vals_out, starts.ptr, kBuckets, Splitters{nullptr, 0, 0, 0}, out_xor, misc.ptr + 2, s);
      BOLT_HIP(hipGetLastError());
      uint32_t e[2] = {0, 0};
      BOLT_TRY(read_back(s, {{e, misc.ptr + 1, 8}}));
      if (e[0]) return set_error(BOLT_ERR_OTHER, "radix sort look-back timed out");
      if (e[1] == 0) {
        set_sort_plan(BOLT_SORT_DIGITS, 2);
        return BOLT_OK;
      }
    }
    bool done = false;
    if (n <= kSplitMax && !sort_by_bytes(n, np)) {
      // Up to a bucket's rows on one value leave the buckets to LDS networks; from
      // there on values have buckets of their own.  20M floats in cents, by bytes
      // 1470 us: one row a value 1413 by splitters, 3 rows 1564, 12 2175, 100 2078,
      // 700 1609, 1000 1323; 33M, by bytes 2400: 1 2181, 3 2398, 100 3783, 1000 2638.
      double rows = 0;
      BOLT_TRY(split_rows_per_value(s, keys_in, n, in_xor, sample, &rows));
      if (rows < 2.5 || rows > 800.0) BOLT_TRY(split(&done));
    }
    if (done) return BOLT_OK;
  }
  // hybrid: two global passes on the top varying digits, then LDS bucket sorts
  if (np >= 3 && n > kSplitMax && getenv("BOLT_SORT_LSD") == nullptr) {
    const int p1 = todo[np - 2], p2 = todo[np - 1];
    BOLT_TRY(pass(keys_in, vals_in, keys_out, vals_out, p1, in_xor, 0));
    BOLT_TRY(pass(keys_out, vals_out, ktmp.ptr, vtmp.ptr, p2, 0, 0));
    DevBuf<uint32_t> starts;
    BOLT_TRY(starts.alloc(kBuckets + 1, s));
    BOLT_TRY(fill_u32(misc.ptr + 2, 0, 2, s));
    bucket_bounds_kernel<<<(kBuckets + 1 + 255) / 256, 256, 0, s>>>(ktmp.ptr, n, 0, p1 * kRadixBits, p2 * kRadixBits,
                                                                  starts.ptr, misc.ptr + 2);
    BOLT_HIP(hipGetLastError());
    uint32_t mx[2] = {0, 0};
    BOLT_TRY(read_back(s, {{mx, misc.ptr + 1, 8}}));
    if (mx[0]) return set_error(BOLT_ERR_OTHER, "radix sort look-back timed out");
    if (mx[1] <= (uint32_t)kLocMax) {
      uint32_t byte_mask = 0;
      for (int q = 0; q < np - 2; q++) byte_mask |= 1u << todo[q];
      BOLT_TRY(fill_u32(misc.ptr + 2, 0, 1, s));
      local_sort_kernel<<<kBuckets, kLocBlock, 0, s>>>(ktmp.ptr, vtmp.ptr, keys_out, vals_out, starts.ptr,
                                                       p1 * kRadixBits, byte_mask, out_xor, misc.ptr + 2);
      BOLT_HIP(hipGetLastError());
      uint32_t e2 = 0;
      BOLT_TRY(read_back(s, {{&e2, misc.ptr + 2, 4}}));
      if (e2) return set_error(BOLT_ERR_OTHER, "radix sort: bucket larger than the LDS sort");
      set_sort_plan(BOLT_SORT_DIGITS, 2);
      return BOLT_OK;
    }
    // a bucket too large for LDS (skewed keys): plain LSD from the input
  }
  // LSD: one pass per varying digit, ping-pong so the last pass writes the output
  set_sort_plan(BOLT_SORT_BYTES, np);
  const uint64_t* ksrc = keys_in;
  const uint32_t* vsrc = vals_in;
  for (int q = 0; q < np; q++) {
    const bool to_out = ((np - 1 - q) % 2) == 0;
    uint64_t* kdst = to_out ? keys_out : ktmp.ptr;
    uint32_t* vdst = to_out ? vals_out : vtmp.ptr;
    BOLT_TRY(pass(ksrc, vsrc, kdst, vdst, todo[q], q == 0 ? in_xor : 0, q == np - 1 ? out_xor : 0));
    ksrc = kdst;
    vsrc = vdst;
  }
  return check_lookback();
}

// ---- key transforms ------------------------------------------------------------------

// Ascending radix image of column value `row` (bits used: 32 or 64).
__device__ __forceinline__ uint64_t radix_image(const void* d, int dt, int64_t row) {
  switch (dt) {
    case BOLT_I32: case BOLT_DATE32: return (uint64_t)(static_cast<const uint32_t*>(d)[row] ^ 0x80000000u);
    case BOLT_I64: return static_cast<const uint64_t*>(d)[row] ^ 0x8000000000000000ull;
    case BOLT_F32: {
      uint32_t b = static_cast<const uint32_t*>(d)[row];
      if ((b & 0x7FFFFFFFu) > 0x7F800000u) b = 0x7FC00000u;  // canonical NaN
      else if ((b & 0x7FFFFFFFu) == 0) b = 0;
      uint32_t m = (uint32_t)((int32_t)b >> 31) | 0x80000000u;  // gpu_sort.rs:1150
      return (uint64_t)(b ^ m);
    }
    case BOLT_F64: {
      uint64_t b = static_cast<const uint64_t*>(d)[row];
      if ((b & 0x7FFFFFFFFFFFFFFFull) > 0x7FF0000000000000ull) b = 0x7FF8000000000000ull;
      else if ((b & 0x7FFFFFFFFFFFFFFFull) == 0) b = 0;
      uint64_t m = (uint64_t)((int64_t)b >> 63) | 0x8000000000000000ull;  // gpu_sort.rs:1169
      return b ^ m;
    }
    case BOLT_BOOL: return static_cast<const uint8_t*>(d)[row] ? 1 : 0;
    case BOLT_DEC128: return static_cast<const uint64_t*>(d)[2 * row];  // low word, unsigned (mode 2: high word)
  }
  return 0;
}

// key[i] = image of column value at perm[i]; mode 0 = value (DESC = NOT),
// mode 1 = null rank only (0 first / 1 last per nulls_first), mode 2 = the
// signed high word of a Decimal128 (its low word, unsigned, is mode 0).
__global__ void order_key_kernel(const void* __restrict__ d, const uint8_t* __restrict__ valid, int dt, int bits,
                                 int desc, int nulls_first, int mode, const uint32_t* __restrict__ perm,
                                 uint64_t* __restrict__ key, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const uint64_t mask = bits >= 64 ? ~0ull : ((1ull << bits) - 1);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    int64_t row = perm[i];
    if (mode == 1) {
      bool isnull = !bit_valid(valid, row);
      key[i] = isnull ? (nulls_first ? 0 : 1) : (nulls_first ? 1 : 0);
    } else {
      uint64_t k = 0;
      if (bit_valid(valid, row))
        k = mode == 2 ? static_cast<const uint64_t*>(d)[2 * row + 1] ^ 0x8000000000000000ull : radix_image(d, dt, row);
      key[i] = (desc ? ~k : k) & mask;
    }
  }
}

// ---- multi-column ORDER BY as one sort ---------------------------------------------
//
// Every ORDER BY key is one or two fields (its NULL rank, its value; a Decimal128
// value is its signed high word, then its low word), each an unsigned image that
// ascends along the order.  The fields' images, less their smallest value, are
// packed most significant first into one 64-bit key, so a single sort orders all
// columns: 0.74 ms for a nullable date and a float over 5M rows, where one sort
// per field, each reading its column through the permutation so far, took 1.60 ms.
// When the fields need more than 64 bits the last one that fits is cut.  Rows that
// agree on all 64 bits are then put in order run by run where the runs are short
// and few (tie_order_kernel).  Elsewhere the keys are replaced by their rank
// (rank_pack_kernel), which leaves room for the next bits, and sorted again: a
// sort per 64 bits or so, not per field.
constexpr int kMaxFields = 16;
enum { kFieldValue = 0, kFieldNull = 1, kFieldDecHigh = 2 };
struct OrderField {
  const void* d;
  const uint8_t* v;
  uint64_t min;      // smallest image of a valid row
  int32_t dt, kind, bits, desc, nulls_first;
  int32_t width;     // bits in the packed key
  int32_t drop;      // the image's bits below those
};
struct OrderFields {
  OrderField f[kMaxFields];
  int32_t n;
};

__device__ __forceinline__ uint64_t field_image(const OrderField& f, int64_t row) {
  const uint64_t k = f.kind == kFieldDecHigh ? static_cast<const uint64_t*>(f.d)[2 * row + 1] ^ 0x8000000000000000ull
                                             : radix_image(f.d, f.dt, row);
  return (f.desc ? ~k : k) & (f.bits >= 64 ? ~0ull : (1ull << f.bits) - 1);
}
__device__ __forceinline__ uint64_t null_rank(const OrderField& f, int64_t row) {
  return bit_valid(f.v, row) == (f.nulls_first != 0) ? 1 : 0;
}

// range[2 y], range[2 y + 1]: complement of the smallest image and the largest
// image of field y's valid rows (both start at 0 and grow).
__global__ __launch_bounds__(256) void field_range_kernel(OrderFields of, int64_t n,
                                                          unsigned long long* __restrict__ range) {
  const OrderField& f = of.f[blockIdx.y];
  if (f.kind == kFieldNull) return;
  uint64_t inv = 0, mx = 0;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < n; i0 += 4 * stride) {
    uint64_t k[4];
    bool ok[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int64_t i = i0 + u * stride < n ? i0 + u * stride : i0;
      ok[u] = bit_valid(f.v, i);
      k[u] = field_image(f, i);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (ok[u]) {
        inv = ~k[u] > inv ? ~k[u] : inv;
        mx = k[u] > mx ? k[u] : mx;
      }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const uint64_t a = __shfl_xor(inv, m), b = __shfl_xor(mx, m);
    inv = a > inv ? a : inv;
    mx = b > mx ? b : mx;
  }
  __shared__ uint64_t r[2][4];
  if ((threadIdx.x & 63) == 0) {
    r[0][threadIdx.x >> 6] = inv;
    r[1][threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    uint64_t x = r[threadIdx.x][0];
    for (int w = 1; w < 4; w++) x = r[threadIdx.x][w] > x ? r[threadIdx.x][w] : x;
    if (x) atomicMax(&range[2 * blockIdx.y + threadIdx.x], (unsigned long long)x);
  }
}

// The bits of field f (width > 0) that the packed key holds.
__device__ __forceinline__ uint64_t field_bits(const OrderField& f, int64_t row) {
  if (f.kind == kFieldNull) return null_rank(f, row);
  const uint64_t x = bit_valid(f.v, row) ? (field_image(f, row) - f.min) >> f.drop : 0ull;
  return f.width < 64 ? x & ((1ull << f.width) - 1) : x;
}

// key[i] = the packed fields of row i, rows[i] = i.
__global__ __launch_bounds__(256) void pack_fields_kernel(OrderFields of, int64_t n, uint64_t* __restrict__ key,
                                                          uint32_t* __restrict__ rows) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < n; i0 += 4 * stride) {
    uint64_t k[4] = {0, 0, 0, 0};
    for (int q = 0; q < of.n; q++) {
      const OrderField& f = of.f[q];
      if (f.width == 0) continue;  // constant, or beyond the packed bits
      uint64_t x[4];
#pragma unroll
      for (int u = 0; u < 4; u++) x[u] = field_bits(f, i0 + u * stride < n ? i0 + u * stride : i0);
#pragma unroll
      for (int u = 0; u < 4; u++) k[u] = f.width < 64 ? (k[u] << f.width) | x[u] : x[u];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int64_t i = i0 + u * stride;
      if (i < n) {
        key[i] = k[u];
        rows[i] = (uint32_t)i;
      }
    }
  }
}

// Sorted keys that packed rows share.  Workgroup g looks at rows [g * per,
// (g + 1) * per): heads[g] = the runs of equal keys that start there, work[g] =
// the sum of the squares of the lengths of those of two to kTieRun rows, which is
// what tie_order_kernel's insertion sorts cost; a longer run makes it kTieNever.
constexpr int kTieRun = 64;
constexpr int kTieGrid = 1024;
// Work a row up to which runs are put in order one by one: about three rows a
// value.  Two floats over 5M rows, by runs / by ranks in us: 1 row a value of the
// first 647 / 1117, 2 924 / 1188, 4 1322 / 1325, 8 2222 / 1519, 20 5211 / 1549 (a
// sort per field 1660); 500,000 rows: 2 360 / 461, 4 490 / 502, 8 723 / 523.
constexpr double kTieWork = 4.0;
constexpr unsigned long long kTieNever = 1ull << 50;  // kTieGrid of them fit 64 bits
__global__ __launch_bounds__(256) void tie_count_kernel(const uint64_t* __restrict__ key, int64_t n, int64_t per,
                                                        uint32_t* __restrict__ heads,
                                                        unsigned long long* __restrict__ work) {
  const int64_t lo = (int64_t)blockIdx.x * per, hi = lo + per < n ? lo + per : n;
  uint32_t h = 0;
  unsigned long long w = 0;
  constexpr int R = 4;  // rows of a lane in flight: one at a time is a chain of reads
  for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += 256 * R) {
    uint64_t k[R], before[R], after[R];
#pragma unroll
    for (int u = 0; u < R; u++) {
      const int64_t i = i0 + 256 * u < hi ? i0 + 256 * u : i0;
      k[u] = key[i];
      before[u] = key[i > 0 ? i - 1 : 0];
      after[u] = key[i + 1 < n ? i + 1 : i];
    }
#pragma unroll
    for (int u = 0; u < R; u++) {
      const int64_t i = i0 + 256 * u;
      if (i >= hi || (i > 0 && before[u] == k[u])) continue;
      h++;
      if (after[u] != k[u] || i + 1 == n) continue;
      int len = 2;
      while (len <= kTieRun && i + len < n && key[i + len] == k[u]) len++;
      if (len > kTieRun) w = kTieNever;
      else if (w < kTieNever) w += (unsigned long long)(len * len);
    }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    h += __shfl_xor(h, m);
    w += __shfl_xor(w, m);
  }
  __shared__ uint32_t sh[4];
  __shared__ unsigned long long sw[4];
  if ((threadIdx.x & 63) == 0) {
    sh[threadIdx.x >> 6] = h;
    sw[threadIdx.x >> 6] = w;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    heads[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    w = sw[0] + sw[1] + sw[2] + sw[3];
    work[blockIdx.x] = w < kTieNever ? w : kTieNever;
  }
}

// Rows that agree on the packed key, in row order: the first of each run sorts
// it by the fields that the key does not hold whole (an insertion sort, which
// keeps equal rows in row order).  Does nothing, and sets res[0], where
// tie_count_kernel found more than `limit` work; res[1] = the runs.
__device__ __forceinline__ int cmp_rows(const OrderFields& of, int first, uint32_t a, uint32_t b) {
  for (int q = first; q < of.n; q++) {
    const OrderField& f = of.f[q];
    uint64_t x, y;
    if (f.kind == kFieldNull) {
      x = null_rank(f, a);
      y = null_rank(f, b);
    } else {
      x = bit_valid(f.v, a) ? field_image(f, a) : f.min;
      y = bit_valid(f.v, b) ? field_image(f, b) : f.min;
    }
    if (x != y) return x < y ? -1 : 1;
  }
  return 0;
}
__global__ __launch_bounds__(256) void tie_order_kernel(OrderFields of, int first, const uint64_t* __restrict__ key,
                                                        int64_t n, uint32_t* __restrict__ rows,
                                                        const uint32_t* __restrict__ heads,
                                                        const unsigned long long* __restrict__ work, int chunks,
                                                        unsigned long long limit, uint32_t* __restrict__ res) {
  __shared__ uint32_t sh[4];
  __shared__ unsigned long long sw[4];
  uint32_t h = 0;
  unsigned long long w = 0;
  for (int c = threadIdx.x; c < chunks; c += 256) {
    h += heads[c];
    w += work[c];
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    h += __shfl_xor(h, m);
    w += __shfl_xor(w, m);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[threadIdx.x >> 6] = h;
    sw[threadIdx.x >> 6] = w;
  }
  __syncthreads();
  w = sw[0] + sw[1] + sw[2] + sw[3];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    res[0] = w > limit ? 1u : 0u;
    res[1] = sh[0] + sh[1] + sh[2] + sh[3];
  }
  if (w == 0 || w > limit) return;  // block-uniform
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i + 1 < n; i += stride) {
    const uint64_t k = key[i];
    if (key[i + 1] != k || (i > 0 && key[i - 1] == k)) continue;
    int len = 2;
    while (i + len < n && key[i + len] == k) len++;
    for (int x = 1; x < len; x++) {
      const uint32_t r = rows[i + x];
      int y = x - 1;
      while (y >= 0 && cmp_rows(of, first, rows[i + y], r) > 0) {
        rows[i + y + 1] = rows[i + y];
        y--;
      }
      rows[i + y + 1] = r;
    }
  }
}

// next[i] = the rank of key[i] among the distinct keys, then the fields' next
// bits of row rows[i].  Workgroups as tie_count_kernel's.
__global__ __launch_bounds__(256) void rank_pack_kernel(OrderFields of, const uint64_t* __restrict__ key, int64_t n,
                                                        int64_t per, const uint32_t* __restrict__ heads,
                                                        const uint32_t* __restrict__ rows,
                                                        uint64_t* __restrict__ next) {
  __shared__ uint32_t sh[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t before = 0;  // runs before this workgroup's rows
  for (int c = threadIdx.x; c < (int)blockIdx.x; c += 256) before += heads[c];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) before += __shfl_xor(before, m);
  if (lane == 0) sh[wave] = before;
  __syncthreads();
  before = sh[0] + sh[1] + sh[2] + sh[3];
  const int64_t lo = (int64_t)blockIdx.x * per, hi = lo + per < n ? lo + per : n;
  for (int64_t base = lo; base < hi; base += 256) {
    const int64_t i = base + threadIdx.x;
    const bool head = i < hi && (i == 0 || key[i] != key[i - 1]);
    const uint64_t b = __ballot(head);
    __syncthreads();  // sh is read
    if (lane == 0) sh[wave] = (uint32_t)__popcll(b);
    __syncthreads();
    uint32_t rank = before + (uint32_t)__popcll(b & (~0ull >> (63 - lane)));  // runs up to this row's
    for (int w = 0; w < wave; w++) rank += sh[w];
    before += sh[0] + sh[1] + sh[2] + sh[3];
    if (i >= hi) continue;
    uint64_t k = rank - 1;
    const int64_t row = rows[i];
    for (int q = 0; q < of.n; q++)
      if (of.f[q].width) k = of.f[q].width < 64 ? (k << of.f[q].width) | field_bits(of.f[q], row) : field_bits(of.f[q], row);
    next[i] = k;
  }
}

// ---- ORDER BY + LIMIT: radix select on the leading key ---------------------------------
//
// `coarse_of` maps the leading key of a row to a u64 that never decreases
// along the full sort order (NULL rank, direction and value in one word; a
// Decimal128 by its signed high word).  The K-th smallest image is T; every
// row among the first K of the order has an image <= T, so sorting only
// those rows by all keys (and by row id, for the stability of the full sort)
// gives the same first K rows as sorting everything.
struct TopKey {
  const void* d;
  const uint8_t* v;
  int dt, bits, desc, nulls_first;
};

// Raw bits of row i's key value: W = byte width (16 = Decimal128, whose
// signed high word is the part of the value the select looks at).
template <int W>
__device__ __forceinline__ uint64_t load_raw(const void* d, int64_t i) {
  if constexpr (W == 1) return static_cast<const uint8_t*>(d)[i];
  else if constexpr (W == 4) return static_cast<const uint32_t*>(d)[i];
  else if constexpr (W == 8) return static_cast<const uint64_t*>(d)[i];
  else return static_cast<const uint64_t*>(d)[2 * i + 1];
}

// The same past the caches, for a pass that reads the column once.
template <int W>
__device__ __forceinline__ uint64_t load_raw_once(const void* d, int64_t i) {
  if constexpr (W == 1) return __builtin_nontemporal_load(static_cast<const uint8_t*>(d) + i);
  else if constexpr (W == 4) return __builtin_nontemporal_load(static_cast<const uint32_t*>(d) + i);
  else if constexpr (W == 8) return __builtin_nontemporal_load(static_cast<const uint64_t*>(d) + i);
  else return __builtin_nontemporal_load(static_cast<const uint64_t*>(d) + 2 * i + 1);
}

// Ascending image of raw key bits (the transforms of radix_image).
__device__ __forceinline__ uint64_t raw_image(uint64_t b, int dt) {
  switch (dt) {
    case BOLT_I32: case BOLT_DATE32: return (uint64_t)((uint32_t)b ^ 0x80000000u);
    case BOLT_F32: {
      uint32_t x = (uint32_t)b;
      if ((x & 0x7FFFFFFFu) > 0x7F800000u) x = 0x7FC00000u;
      else if ((x & 0x7FFFFFFFu) == 0) x = 0;
      return (uint64_t)(x ^ ((uint32_t)((int32_t)x >> 31) | 0x80000000u));
    }
    case BOLT_F64: {
      if ((b & 0x7FFFFFFFFFFFFFFFull) > 0x7FF0000000000000ull) b = 0x7FF8000000000000ull;
      else if ((b & 0x7FFFFFFFFFFFFFFFull) == 0) b = 0;
      return b ^ ((uint64_t)((int64_t)b >> 63) | 0x8000000000000000ull);
    }
    case BOLT_BOOL: return b ? 1 : 0;
    default: return b ^ 0x8000000000000000ull;  // Int64; Decimal128 high word
  }
}

__device__ __forceinline__ uint64_t coarse_of(const TopKey& k, uint64_t raw, bool valid) {
  uint64_t x = 0;
  if (valid) {
    x = raw_image(raw, k.dt);
    if (k.desc) x = ~x & (k.bits >= 64 ? ~0ull : ((1ull << k.bits) - 1));
  }
  if (k.v == nullptr) return x;
  // every image stays below 2^bits, so the select can start at bit `bits`
  if (!valid) return k.nulls_first ? 0ull : (k.bits >= 64 ? ~0ull : (1ull << k.bits) - 1);
  return k.nulls_first ? (x >> 1) + 1 : x >> 1;
}

// Inputs whose leading key is read in about the time that the sample's kernels
// take keep the counting pass.
constexpr int64_t kTopSampleBytes = (int64_t)256 << 20;
constexpr int kSelBits = 14;
constexpr int kSelBins = 1 << kSelBits;  // 64 KB of LDS counters
constexpr int kSelBlock = 1024;
constexpr int kSelUnroll = 4;  // rows in flight per lane

// Per-workgroup histogram of digit (image >> shift) & (2^width - 1) over the
// rows whose image >> (shift + width) equals `prefix` (every row when
// shift + width = 64), written to part[block][bin] with plain stores (a
// global atomic per bin per workgroup would cost more than the row pass).
// With `spec` non-null (the first pass) the rows whose digit is at most
// spec_bound are also appended to spec (unordered, up to spec_cap): a guess
// at the candidates that saves the collect pass when the K-th row's digit
// turns out to be within the bound.
template <int W>
__global__ __launch_bounds__(kSelBlock) void topk_hist_kernel(TopKey k, int64_t n, int shift, int width,
                                                              uint64_t prefix, uint32_t* __restrict__ part,
                                                              uint64_t spec_bound, uint32_t* __restrict__ spec,
                                                              unsigned long long* __restrict__ spec_count,
                                                              int64_t spec_cap) {
  __shared__ uint32_t sh[kSelBins];
  __shared__ int spec_full;  // set once this workgroup has seen the guess buffer full
  const int nb = 1 << width;
  for (int b = threadIdx.x; b < nb; b += kSelBlock) sh[b] = 0;
  if (threadIdx.x == 0) spec_full = 0;
  __syncthreads();
  const int hi = shift + width;
  const uint64_t dmask = (uint64_t)nb - 1;
  const int64_t stride = (int64_t)gridDim.x * kSelBlock;
  for (int64_t i0 = (int64_t)blockIdx.x * kSelBlock + threadIdx.x; i0 < n; i0 += stride * kSelUnroll) {
    uint64_t x[kSelUnroll];
#pragma unroll
    for (int u = 0; u < kSelUnroll; u++) {
      const int64_t i = i0 + u * stride;
      x[u] = i < n ? load_raw<W>(k.d, i) : 0;
    }
#pragma unroll
    for (int u = 0; u < kSelUnroll; u++) {
      const int64_t i = i0 + u * stride;
      bool take = false;
      if (i < n) {
        const uint64_t c = coarse_of(k, x[u], bit_valid(k.v, i));
        if (hi >= 64 || (c >> hi) == prefix) atomicAdd(&sh[(c >> shift) & dmask], 1u);
        // a guess that has already overflowed is abandoned: the collect pass
        // runs instead, so further appends (one atomic per wave) are waste
        take = spec != nullptr && (c >> shift) <= spec_bound && !*(volatile int*)&spec_full;
      }
      const uint64_t m = __ballot(take);  // lanes still in the loop
      if (m) {
        const int lane = threadIdx.x & 63;
        const int leader = __builtin_ctzll(m);
        unsigned long long b = 0;
        if (lane == leader) {
          b = atomicAdd(spec_count, (unsigned long long)__popcll(m));
          if ((int64_t)b + __popcll(m) > spec_cap) *(volatile int*)&spec_full = 1;
        }
        b = __shfl(b, leader);
        if (take) {
          const int64_t pos = (int64_t)b + __popcll(m & ((1ull << lane) - 1));
          if (pos < spec_cap) spec[pos] = (uint32_t)i;
        }
      }
    }
  }
  __syncthreads();
  uint32_t* out = part + (int64_t)blockIdx.x * nb;
  for (int b = threadIdx.x; b < nb; b += kSelBlock) out[b] = sh[b];
}

// hist[b] += sum of part[w][b] over this launch row's share of workgroups
// (hist starts at zero; gridDim.y shares split the workgroups)
__global__ __launch_bounds__(256) void topk_hist_sum_kernel(const uint32_t* __restrict__ part, int blocks, int nb,
                                                            uint32_t* __restrict__ hist) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= nb) return;
  const int per = (blocks + (int)gridDim.y - 1) / (int)gridDim.y;
  const int w0 = (int)blockIdx.y * per;
  const int w1 = w0 + per < blocks ? w0 + per : blocks;
  uint32_t t = 0;
  for (int w = w0; w < w1; w++) t += part[(int64_t)w * nb + b];
  if (t) atomicAdd(&hist[b], t);
}

// A bound from a sample: large inputs are read once, comparing each row's image
// with a quantile of the sampled images a little above rank K, instead of
// counting digits of every row in LDS (2 GiB of int64 keys: 0.57 ms to count
// and guess, 0.35 to compare and collect; a plain read takes 0.33).  The
// sample's images in sorted lists, as split_sample_kernel's.
__global__ __launch_bounds__(kSampleList) void topk_sample_kernel(TopKey k, int64_t n, int S,
                                                                  uint64_t* __restrict__ lists) {
  __shared__ uint64_t key[kSampleList];
  const int j = blockIdx.x * kSampleList + threadIdx.x;
  const int64_t lo = (int64_t)j * n / S, hi = (int64_t)(j + 1) * n / S;
  const uint32_t h = (uint32_t)j * 0x9E3779B1u;
  const int64_t i = lo + (int64_t)(((uint64_t)h * (uint64_t)(hi - lo)) >> 32);
  uint64_t raw;
  switch (k.dt) {
    case BOLT_BOOL: raw = load_raw<1>(k.d, i); break;
    case BOLT_I32: case BOLT_F32: case BOLT_DATE32: raw = load_raw<4>(k.d, i); break;
    case BOLT_DEC128: raw = load_raw<16>(k.d, i); break;
    default: raw = load_raw<8>(k.d, i); break;
  }
  key[threadIdx.x] = coarse_of(k, raw, bit_valid(k.v, i));
  __syncthreads();
  lds_bitonic<kSampleList>(kSampleList, [&](int a, int b) {
    const uint64_t x = key[a], y = key[b];
    if (x > y) {
      key[a] = y;
      key[b] = x;
    }
  });
  lists[j] = key[threadIdx.x];
}

// plan[0] = the sample's rank-r image (1-based); plan[1] = samples at or below
// it (more than r where it is tied); one wave.
__global__ __launch_bounds__(64) void topk_bound_kernel(const uint64_t* __restrict__ sorted, int S, int r,
                                                        uint64_t* __restrict__ plan) {
  const uint64_t b = sorted[r - 1];
  int at = S;  // first sample above b
  for (int base = r; base < S; base += 64) {
    const int i = base + threadIdx.x;
    const uint64_t m = __ballot(i < S && sorted[i] > b);
    if (m) {
      at = base + __builtin_ctzll(m);
      break;
    }
  }
  if (threadIdx.x == 0) {
    plan[0] = b;
    plan[1] = (uint64_t)at;
  }
}

// Appends (unordered) the rows whose image >> shift <= bound.  With `plan`
// the bound is the sample's, the kernel leaves *count at all ones at once when
// the sample has more than max_ties rows at or below it, and the smallest image
// appended goes to *min_out.
template <int W, int DT = -1>
__global__ __launch_bounds__(256) void topk_collect_kernel(TopKey k, int64_t n, int shift, uint64_t bound,
                                                           uint32_t* __restrict__ out,
                                                           unsigned long long* __restrict__ count, int64_t cap,
                                                           const uint64_t* __restrict__ plan = nullptr,
                                                           uint64_t max_ties = 0,
                                                           unsigned long long* __restrict__ min_out = nullptr) {
  if constexpr (DT >= 0) k.dt = DT;  // the image's arithmetic without its switch: int64 396 -> 352 us, int32 380 -> 281
  if (plan) {
    bound = plan[0];
    if (plan[1] > max_ties) {
      if (blockIdx.x == 0 && threadIdx.x == 0) *count = ~0ull;
      return;
    }
  }
  // Rows are gathered per wave in LDS and appended with one atomic per
  // workgroup at the end (or per wave and kWaveBuf rows where many pass): an
  // atomic per wave and row group, all on one word, took 15 ns each, 1.28 ms
  // for 82,000 rows among 2^28.
  // 64 bytes in flight per lane; 4 rows: int64 431 us, int32 about 430 (2^28 rows)
  constexpr int kU = W >= 8 ? 8 : 16;
  constexpr int kWaveBuf = 128 * kU;
  __shared__ uint32_t buf[4][kWaveBuf];
  __shared__ uint32_t wcnt[4];
  __shared__ unsigned long long wbase[4];
  const int64_t stride = (int64_t)gridDim.x * 256;
  const int64_t end = (n + 255) / 256 * 256;  // block-uniform trip count for the ballot
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t have = 0;  // rows in buf[wave]
  uint64_t least = ~0ull;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < end; i0 += stride * kU) {
    uint64_t x[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int64_t i = i0 + u * stride;
      x[u] = load_raw_once<W>(k.d, i < n ? i : n - 1);
    }
    bool take[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int64_t i = i0 + u * stride;
      take[u] = false;
      if (i < n) {  // the validity bit, too, is read only for rows that exist
        const uint64_t c = shift >= 64 ? 0ull : coarse_of(k, x[u], bit_valid(k.v, i)) >> shift;
        take[u] = c <= bound;
        if (take[u] && c < least) least = c;
      }
    }
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const uint64_t m = __ballot(take[u]);
      if (m == 0) continue;
      if (take[u]) buf[wave][have + __popcll(m & ((1ull << lane) - 1))] = (uint32_t)(i0 + u * stride);
      have += (uint32_t)__popcll(m);
    }
    if (have > kWaveBuf - 64 * kU) {  // no room for another iteration's rows
      unsigned long long base = 0;
      if (lane == 0) base = atomicAdd(count, (unsigned long long)have);
      base = __shfl(base, 0);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (uint32_t j = lane; j < have; j += 64)
        if ((int64_t)(base + j) < cap) out[base + j] = buf[wave][j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      have = 0;
    }
  }
  if (min_out) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const uint64_t o = __shfl_xor(least, m);
      least = o < least ? o : least;
    }
    if (lane == 0) wbase[wave] = least;
  }
  if (lane == 0) wcnt[wave] = have;
  __syncthreads();
  if (threadIdx.x == 0) {
    if (min_out) {
      for (int w = 0; w < 4; w++) least = wbase[w] < least ? wbase[w] : least;
      if (least != ~0ull) atomicMin(min_out, (unsigned long long)least);
    }
    const uint32_t total = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    unsigned long long base = total ? atomicAdd(count, (unsigned long long)total) : 0ull;
    for (int w = 0; w < 4; w++) {
      wbase[w] = base;
      base += wcnt[w];
    }
  }
  __syncthreads();
  const unsigned long long base = wbase[wave];
  for (uint32_t j = lane; j < have; j += 64)
    if ((int64_t)(base + j) < cap) out[base + j] = buf[wave][j];
}

// ---- small final sets: narrowed over the candidates, sorted in one workgroup ----------
constexpr int kSmallSort = 4096;  // (image, row) pairs sorted in LDS by one workgroup

// hist[digit] over the candidates whose image >> (shift + width) == prefix.
// Counted in LDS first: candidates of neighbouring keys share their upper
// digits, and an atomic each on one word would take 15 ns each.
template <int W>
__global__ __launch_bounds__(kSelBlock) void topk_cand_hist_kernel(TopKey k, const uint32_t* __restrict__ cand,
                                                                   int64_t c, int shift, int width, uint64_t prefix,
                                                                   uint32_t* __restrict__ hist) {
  __shared__ uint32_t sh[kSelBins];
  const int nb = 1 << width;
  for (int b = threadIdx.x; b < nb; b += kSelBlock) sh[b] = 0;
  __syncthreads();
  const int hi = shift + width;
  for (int64_t j = (int64_t)blockIdx.x * kSelBlock + threadIdx.x; j < c; j += (int64_t)gridDim.x * kSelBlock) {
    const uint64_t x = coarse_of(k, load_raw<W>(k.d, cand[j]), true);
    if (hi >= 64 || (x >> hi) == prefix) atomicAdd(&sh[(x >> shift) & ((1ull << width) - 1)], 1u);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += kSelBlock)
    if (sh[b]) atomicAdd(&hist[b], sh[b]);
}

// Candidates tied on the whole image `img`: histogram of their row ids'
// bits [shift, shift + width) among those whose higher row-id bits are
// `rprefix` (the order among equal keys is by row id).
template <int W>
__global__ __launch_bounds__(256) void topk_tie_hist_kernel(TopKey k, const uint32_t* __restrict__ cand, int64_t c,
                                                            uint64_t img, int shift, int width, uint32_t rprefix,
                                                            uint32_t* __restrict__ hist) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= c) return;
  const uint32_t r = cand[j];
  if (coarse_of(k, load_raw<W>(k.d, r), true) != img) return;
  const int hi = shift + width;
  if (hi < 32 && (r >> hi) != rprefix) return;
  atomicAdd(&hist[(r >> shift) & ((1u << width) - 1)], 1u);
}

// appends the candidates whose image >> shift <= bound; with shift 0 and
// rmax < 0xFFFFFFFF, of the rows whose image equals `bound` only those with
// row id <= rmax
template <int W>
__global__ __launch_bounds__(256) void topk_cand_collect_kernel(TopKey k, const uint32_t* __restrict__ cand,
                                                                int64_t c, int shift, uint64_t bound,
                                                                uint32_t* __restrict__ out,
                                                                unsigned long long* __restrict__ count, int64_t cap,
                                                                uint32_t rmax = 0xFFFFFFFFu) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  bool take = false;
  uint32_t r = 0;
  if (j < c) {
    r = cand[j];
    const uint64_t x = shift >= 64 ? 0ull : coarse_of(k, load_raw<W>(k.d, r), true) >> shift;
    take = x < bound || (x == bound && r <= rmax);
  }
  const uint64_t m = __ballot(take);
  if (m == 0) return;
  const int leader = __builtin_ctzll(m);
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(count, (unsigned long long)__popcll(m));
  base = __shfl(base, leader);
  if (take) {
    const int64_t pos = (int64_t)base + __popcll(m & ((1ull << lane) - 1));
    if (pos < cap) out[pos] = r;
  }
}

// Sorts c <= kSmallSort rows by (image, row id) with a bitonic network in
// LDS (padded to a power of two with pairs that sort last) and writes rows
// [first, first + m) of the order.
template <int W>
__global__ __launch_bounds__(1024) void topk_small_sort_kernel(TopKey k, const uint32_t* __restrict__ rows, int c,
                                                               int npow, int first, int m,
                                                               uint32_t* __restrict__ out) {
  __shared__ uint64_t key[kSmallSort];
  __shared__ uint32_t row[kSmallSort];
  for (int i = threadIdx.x; i < npow; i += 1024) {
    if (i < c) {
      const uint32_t r = rows[i];
      key[i] = coarse_of(k, load_raw<W>(k.d, r), true);
      row[i] = r;
    } else {
      key[i] = ~0ull;
      row[i] = 0xFFFFFFFFu;
    }
  }
  __syncthreads();
  for (int size = 2; size <= npow; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < npow; i += 1024) {
        const int j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          const bool gt = key[i] > key[j] || (key[i] == key[j] && row[i] > row[j]);
          if (gt == up) {
            const uint64_t tk = key[i];
            key[i] = key[j];
            key[j] = tk;
            const uint32_t tr = row[i];
            row[i] = row[j];
            row[j] = tr;
          }
        }
      }
      __syncthreads();
    }
  for (int j = threadIdx.x; j < m; j += 1024) out[j] = row[first + j];
}

// out[j] = rows[perm[first + j]]
__global__ void topk_emit_kernel(const uint32_t* __restrict__ rows, const uint32_t* __restrict__ perm, int64_t first,
                                 int64_t m, uint32_t* __restrict__ out) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < m) out[j] = rows[perm[first + j]];
}

__global__ void iota_kernel(uint32_t* __restrict__ out, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = (uint32_t)i;
}

}  // namespace bolt

using namespace bolt;

extern "C" int bolt_sort_pairs_i64(bolt_stream_t stream, const int64_t* keys_in, const uint32_t* vals_in, int64_t n,
                                   int32_t descending, int64_t* keys_out, uint32_t* vals_out) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  if (n < 0) return set_error(BOLT_ERR_PLAN, "bolt_sort_pairs_i64: negative length");
  if (n == 0) return BOLT_OK;
  // radix image: sign bit flipped (src/exec/gpu_sort.rs:1091), all bits
  // inverted for DESC; applied on load by the first pass and undone on the
  // final store, so no separate transform kernels run
  const uint64_t x = descending ? 0x7FFFFFFFFFFFFFFFull : 0x8000000000000000ull;
  const uint64_t* kin = reinterpret_cast<const uint64_t*>(keys_in);
  const uint32_t* vin = vals_in;
  DevBuf<uint64_t> kcopy;
  DevBuf<uint32_t> vcopy;
  if ((const void*)keys_in == (const void*)keys_out || (const void*)vals_in == (const void*)vals_out) {
    BOLT_TRY(kcopy.alloc((size_t)n, s));
    BOLT_TRY(vcopy.alloc((size_t)n, s));
    BOLT_HIP(hipMemcpyAsync(kcopy.ptr, keys_in, (size_t)n * 8, hipMemcpyDeviceToDevice, s));
    BOLT_HIP(hipMemcpyAsync(vcopy.ptr, vals_in, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    kin = kcopy.ptr;
    vin = vcopy.ptr;
  }
  prof_begin(s);
  BOLT_TRY(radix_sort_u64_pairs(s, kin, vin, n, reinterpret_cast<uint64_t*>(keys_out), vals_out, 64, x, x));
  prof_end(s);
  return BOLT_OK;
}

// ORDER BY by packed keys.  *done = false when there are too many fields: the
// caller then sorts field by field.
static int sort_packed(hipStream_t s, const bolt_column_t* keys, int32_t n_keys, const int32_t* descending,
                       const int32_t* nulls_first, int64_t n, uint64_t* k0, uint64_t* k1, uint32_t* p0,
                       uint32_t* out_rows, bool* done) {
  OrderFields of;
  memset(&of, 0, sizeof of);
  int total = 0;
  for (int k = 0; k < n_keys; k++) {
    const bolt_column_t& c = keys[k];
    if (of.n + 3 > kMaxFields) return BOLT_OK;
    OrderField f;
    memset(&f, 0, sizeof f);
    f.d = c.data;
    f.v = c.validity;
    f.dt = c.dtype;
    f.desc = descending ? descending[k] : 0;
    f.nulls_first = nulls_first ? nulls_first[k] : 1;
    if (c.validity) {
      f.kind = kFieldNull;
      f.bits = 1;
      of.f[of.n++] = f;
      total += 1;
    }
    f.bits = c.dtype == BOLT_BOOL ? 1 : c.dtype == BOLT_DEC128 ? 64 : dtype_size(c.dtype) * 8;
    if (c.dtype == BOLT_DEC128) {
      f.kind = kFieldDecHigh;
      of.f[of.n++] = f;
      total += 64;
    }
    f.kind = kFieldValue;
    of.f[of.n++] = f;
    total += f.bits;
  }
  int rest[kMaxFields];  // bits of each field that no key has held yet
  for (int q = 0; q < of.n; q++) rest[q] = of.f[q].bits;
  if (total > 64) {
    // the fields' own ranges: a date, a count or the high word of a decimal
    // needs far fewer bits than its type
    DevBuf<unsigned long long> range;
    unsigned long long h[2 * kMaxFields];
    BOLT_TRY(range.alloc(2 * kMaxFields, s));
    BOLT_TRY(fill_u32(range.ptr, 0, 4 * kMaxFields, s));
    field_range_kernel<<<dim3(grid_for(n, 256, 4, 1024), of.n), 256, 0, s>>>(of, n, range.ptr);
    BOLT_HIP(hipGetLastError());
    BOLT_TRY(read_back(s, {{h, range.ptr, sizeof h}}));
    for (int q = 0; q < of.n; q++) {
      OrderField& f = of.f[q];
      if (f.kind == kFieldNull) continue;
      const uint64_t lo = ~(uint64_t)h[2 * q], hi = h[2 * q + 1];
      f.min = lo <= hi ? lo : 0;  // no valid row: every image is skipped
      const uint64_t r = lo <= hi ? hi - lo : 0;
      rest[q] = r ? 64 - __builtin_clzll(r) : 0;
    }
  }
  // the next `left` bits of the fields to the next key; how many there were
  auto take = [&](int left) -> int {
    int taken = 0;
    for (int q = 0; q < of.n; q++) {
      OrderField& f = of.f[q];
      f.width = std::min(rest[q], left - taken);
      f.drop = rest[q] -= f.width;
      taken += f.width;
    }
    return taken;
  };
  total = take(64);
  pack_fields_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(of, n, k0, p0);
  BOLT_HIP(hipGetLastError());
  BOLT_TRY(radix_sort_u64_pairs(s, k0, p0, n, k1, out_rows, std::max(total, 1), 0, 0));
  *done = true;
  const int64_t per = (n + kTieGrid - 1) / kTieGrid;
  const int chunks = (int)((n + per - 1) / per);
  DevBuf<uint32_t> heads;
  DevBuf<unsigned long long> work;
  for (;;) {
    int first = 0;
    while (first < of.n && rest[first] == 0) first++;
    if (first == of.n) return BOLT_OK;
    if (!heads.ptr) {
      BOLT_TRY(heads.alloc(kTieGrid + 2, s));
      BOLT_TRY(work.alloc(kTieGrid, s));
    }
    uint32_t* res = heads.ptr + kTieGrid;
    uint32_t h[2];
    tie_count_kernel<<<chunks, 256, 0, s>>>(k1, n, per, heads.ptr, work.ptr);
    tie_order_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(of, first, k1, n, out_rows, heads.ptr, work.ptr, chunks,
                                                        (unsigned long long)(kTieWork * (double)n), res);
    BOLT_HIP(hipGetLastError());
    BOLT_TRY(read_back(s, {{h, res, 8}}));
    if (h[0] == 0) return BOLT_OK;
    const int rank_bits = h[1] > 1 ? 32 - __builtin_clz(h[1] - 1) : 0;
    total = take(64 - rank_bits);
    rank_pack_kernel<<<chunks, 256, 0, s>>>(of, k1, n, per, heads.ptr, out_rows, k0);
    BOLT_HIP(hipGetLastError());
    BOLT_TRY(radix_sort_u64_pairs(s, k0, out_rows, n, k1, p0, std::max(rank_bits + total, 1), 0, 0));
    BOLT_HIP(hipMemcpyAsync(out_rows, p0, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
  }
}

extern "C" int bolt_sort_last_plan(int32_t* plan, int32_t* passes) {
  if (plan) *plan = t_sort_plan;
  if (passes) *passes = t_sort_passes;
  return BOLT_OK;
}

extern "C" int bolt_sort_indices(bolt_stream_t stream, const bolt_column_t* keys, int32_t n_keys,
                                 const int32_t* descending, const int32_t* nulls_first, uint32_t* out_rows) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  if (n_keys < 1 || keys == nullptr) return set_error(BOLT_ERR_PLAN, "bolt_sort_indices: no sort keys");
  const int64_t n = keys[0].length;
  for (int k = 0; k < n_keys; k++) {
    if (keys[k].length != n) return set_error(BOLT_ERR_PLAN, "bolt_sort_indices: key columns differ in length");
    int dt = keys[k].dtype;
    if (!(dt == BOLT_I32 || dt == BOLT_I64 || dt == BOLT_F32 || dt == BOLT_F64 || dt == BOLT_DATE32 || dt == BOLT_BOOL ||
          dt == BOLT_DEC128))
      return set_error(BOLT_ERR_UNSUPPORTED, "bolt_sort_indices: sort key dtype %s not supported", dtype_name(dt));
  }
  if (n == 0) return BOLT_OK;
  if (n >= (1ll << 30)) return set_error(BOLT_ERR_PLAN, "bolt_sort_indices: %lld rows exceeds 2^30", (long long)n);
  DevBuf<uint64_t> k0, k1;
  DevBuf<uint32_t> p0;
  BOLT_TRY(k0.alloc((size_t)n, s));
  BOLT_TRY(k1.alloc((size_t)n, s));
  BOLT_TRY(p0.alloc((size_t)n, s));
  bool done = false;
  if (getenv("BOLT_SORT_LSD") == nullptr)
    BOLT_TRY(sort_packed(s, keys, n_keys, descending, nulls_first, n, k0.ptr, k1.ptr, p0.ptr, out_rows, &done));
  if (done) {
    BOLT_HIP(hipStreamSynchronize(s));
    return BOLT_OK;
  }
  iota_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(out_rows, n);
  BOLT_HIP(hipGetLastError());
  // least significant key first; each step is a stable sort of the current
  // permutation, so earlier (more significant) keys win ties last
  for (int k = n_keys - 1; k >= 0; k--) {
    const bolt_column_t& c = keys[k];
    const int bits = c.dtype == BOLT_BOOL ? 1 : c.dtype == BOLT_DEC128 ? 64 : dtype_size(c.dtype) * 8;
    const int desc = descending ? descending[k] : 0;
    const int nf = nulls_first ? nulls_first[k] : 1;
    // value (a Decimal128 as its unsigned low word, then its signed high
    // word), then the NULL rank: least significant first
    std::vector<int> modes{0};
    if (c.dtype == BOLT_DEC128) modes.push_back(2);
    if (c.validity) modes.push_back(1);
    for (int mode : modes) {
      order_key_kernel<<<grid_for(n, 256, 4), 256, 0, s>>>(c.data, c.validity, c.dtype, bits, desc, nf, mode, out_rows,
                                                          k0.ptr, n);
      BOLT_HIP(hipGetLastError());
      BOLT_TRY(radix_sort_u64_pairs(s, k0.ptr, out_rows, n, k1.ptr, p0.ptr, mode == 1 ? 1 : bits, 0, 0));
      BOLT_HIP(hipMemcpyAsync(out_rows, p0.ptr, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    }
  }
  BOLT_HIP(hipStreamSynchronize(s));
  return BOLT_OK;
}

extern "C" int bolt_sort_limit(bolt_stream_t stream, const bolt_column_t* keys, int32_t n_keys,
                               const int32_t* descending, const int32_t* nulls_first, int64_t offset, int64_t limit,
                               uint32_t* out_rows, int64_t* n_out) {
  BOLT_CHECK_DEVICE();
  clear_error();
  hipStream_t s = (hipStream_t)stream;
  *n_out = 0;
  if (n_keys < 1 || keys == nullptr) return set_error(BOLT_ERR_PLAN, "bolt_sort_limit: no sort keys");
  if (offset < 0 || limit < 0) return set_error(BOLT_ERR_PLAN, "bolt_sort_limit: negative offset or limit");
  const int64_t n = keys[0].length;
  if (n >= (1ll << 31)) return set_error(BOLT_ERR_PLAN, "bolt_sort_limit: %lld rows exceeds 2^31", (long long)n);
  // execute_limit (src/exec/limit.rs:18): min(limit, n - offset) rows, none past the end
  const int64_t m = offset >= n ? 0 : (limit < n - offset ? limit : n - offset);
  if (m == 0) {
    for (int k = 0; k < n_keys; k++)
      if (keys[k].length != n) return set_error(BOLT_ERR_PLAN, "bolt_sort_limit: key columns differ in length");
    return BOLT_OK;
  }
  const int64_t K = offset + m;  // rows of the order that must be exact
  std::vector<int32_t> desc(n_keys + 1, 0), nf(n_keys + 1, 1);
  for (int k = 0; k < n_keys; k++) {
    desc[k] = descending ? descending[k] : 0;
    nf[k] = nulls_first ? nulls_first[k] : 1;
  }
  // The full sort, then the slice.
  auto full_sort = [&]() -> int {
    DevBuf<uint32_t> perm;
    BOLT_TRY(perm.alloc((size_t)n, s));
    BOLT_TRY(bolt_sort_indices(stream, keys, n_keys, desc.data(), nf.data(), perm.ptr));
    BOLT_HIP(hipMemcpyAsync(out_rows, perm.ptr + offset, (size_t)m * 4, hipMemcpyDeviceToDevice, s));
    BOLT_HIP(hipStreamSynchronize(s));
    *n_out = m;
    return BOLT_OK;
  };
  // inputs of up to 2^20 rows (where the sort is launch-bound and a select
  // saves nothing), or a limit that reaches a quarter of the rows
  if (n <= (1 << 20) || K * 4 >= n) return full_sort();
  for (int k = 0; k < n_keys; k++) {
    if (keys[k].length != n) return set_error(BOLT_ERR_PLAN, "bolt_sort_limit: key columns differ in length");
    const int dt = keys[k].dtype;
    if (!(dt == BOLT_I32 || dt == BOLT_I64 || dt == BOLT_F32 || dt == BOLT_F64 || dt == BOLT_DATE32 || dt == BOLT_BOOL ||
          dt == BOLT_DEC128))
      return set_error(BOLT_ERR_UNSUPPORTED, "bolt_sort_limit: sort key dtype %s not supported", dtype_name(dt));
  }
  const bolt_column_t& c0 = keys[0];
  TopKey tk;
  tk.d = c0.data;
  tk.v = c0.validity;
  tk.dt = c0.dtype;
  tk.bits = c0.dtype == BOLT_BOOL ? 1 : (c0.dtype == BOLT_DEC128 ? 64 : dtype_size(c0.dtype) * 8);
  tk.desc = desc[0];
  tk.nulls_first = nf[0];
  const int kw = c0.dtype == BOLT_BOOL ? 1 : dtype_size(c0.dtype);  // 16 for Decimal128
  // Radix select, most significant digit first: after each pass `prefix`
  // holds the top 64 - hi bits of T, `below` the rows with a smaller prefix
  // and `eq` those with the same one; stop once the tie bucket is small.
  const unsigned hgrid = grid_for(n, kSelBlock, kSelUnroll, 512);
  DevBuf<uint32_t> hist, part;
  BOLT_TRY(hist.alloc(kSelBins, s));
  BOLT_TRY(part.alloc((size_t)hgrid * kSelBins, s));
  std::vector<uint32_t> h(kSelBins);
  uint64_t prefix = 0;
  int hi = tk.bits;  // every image is below 2^bits (coarse_of)
  int64_t below = 0, need = K, eq = n;
  const unsigned grid = grid_for(n, 256, kSelUnroll, 4096);
  const unsigned cgrid = grid_for(n, 256, kSelUnroll, 1024);  // a streaming read's grid (see the aggregates)
  // Candidates guessed in the first pass: the rows whose first digit is at
  // most spec_bound, where the K-th row's digit lies when the keys are spread
  // (about K * 2^14 / n); capacity for twice the expected count.
  const uint64_t spec_bound = (uint64_t)((double)K * (double)kSelBins / (double)n) + 1;
  const int64_t spec_cap = (int64_t)std::min<double>(
      (double)n, 2.0 * (double)(spec_bound + 1) * (double)n / (double)kSelBins + 65536.0);
  DevBuf<uint32_t> spec;
  DevBuf<unsigned long long> spec_cnt;
  BOLT_TRY(spec.alloc((size_t)spec_cap, s));
  BOLT_TRY(spec_cnt.alloc(1, s));
  BOLT_TRY(fill_u32(spec_cnt.ptr, 0, 2, s));
  unsigned long long spec_got = 0;
  int first_digit = -1;
  DevBuf<uint32_t> cand;
  DevBuf<unsigned long long> cnt;
  BOLT_TRY(cnt.alloc(4, s));
  BOLT_TRY(fill_u32(cnt.ptr, 0, 2, s));
  int64_t sampled = -1;  // candidates collected below the sample's bound
  int64_t sample_bytes = kTopSampleBytes;
  if (const char* e = getenv("BOLT_TOPK_SAMPLE_BYTES")) sample_bytes = atoll(e);  // testing
  if (n * kw >= sample_bytes && K <= n / 64) {
    // rank of the bound: K's share of the sample and a few deviations more
    constexpr int S = 8192;
    const double share = (double)K * S / (double)n;
    const int r = (int)std::min<double>(S, std::ceil(share + 4.0 * std::sqrt(share) + 4.0));
    const int64_t expect = (int64_t)((double)r * (double)n / S);
    const int64_t cap = 4 * expect + 65536;  // at r = 5 one sample in a hundred finds twice what is expected
    DevBuf<uint64_t> samp;
    BOLT_TRY(samp.alloc(2 * S + 4, s));
    BOLT_TRY(cand.alloc((size_t)cap, s));
    uint64_t* plan = samp.ptr + 2 * S;
    unsigned long long* least = reinterpret_cast<unsigned long long*>(plan + 2);
    BOLT_TRY(fill_u32(least, 0xFFFFFFFFu, 2, s));
    topk_sample_kernel<<<S / kSampleList, kSampleList, 0, s>>>(tk, n, S, samp.ptr);
    split_merge_kernel<S / kSampleList><<<S / 64, 64, 0, s>>>(samp.ptr, samp.ptr + S);
    topk_bound_kernel<<<1, 64, 0, s>>>(samp.ptr + S, S, r, plan);
    const uint64_t ties = (uint64_t)r + (uint64_t)r / 2 + 2;  // tied beyond that: more rows than `cap` are likely
#define COLLECT_LAUNCH(W, DT) \
  topk_collect_kernel<W, DT><<<cgrid, 256, 0, s>>>(tk, n, 0, 0, cand.ptr, cnt.ptr, cap, plan, ties, least)
    switch (tk.dt) {
      case BOLT_BOOL: COLLECT_LAUNCH(1, BOLT_BOOL); break;
      case BOLT_I32: case BOLT_DATE32: COLLECT_LAUNCH(4, BOLT_I32); break;
      case BOLT_F32: COLLECT_LAUNCH(4, BOLT_F32); break;
      case BOLT_I64: COLLECT_LAUNCH(8, BOLT_I64); break;
      case BOLT_F64: COLLECT_LAUNCH(8, BOLT_F64); break;
      default: COLLECT_LAUNCH(16, BOLT_DEC128); break;
    }
#undef COLLECT_LAUNCH
    BOLT_HIP(hipGetLastError());
    unsigned long long got = 0;
    uint64_t bound[3];  // the bound, its rank, the smallest image collected
    BOLT_TRY(read_back(s, {{&got, cnt.ptr, 8}, {bound, plan, 24}}));
    if (got >= (unsigned long long)K && got <= (unsigned long long)cap) {
      // every row up to the bound, the K first among them; their images agree
      // above bit hi
      sampled = (int64_t)got;
      hi = bound[0] != bound[2] ? 64 - __builtin_clzll(bound[0] ^ bound[2]) : 0;
      prefix = hi < 64 ? bound[0] >> hi : 0;
      eq = sampled;
    }
    BOLT_TRY(fill_u32(cnt.ptr, 0, 2, s));
  }
  while (hi > 0 && sampled < 0) {
    const int width = hi >= kSelBits ? kSelBits : hi;
    const int shift = hi - width;
    uint32_t* sp = first_digit < 0 ? spec.ptr : nullptr;
#define HIST_LAUNCH(WW)                                                                                         \
  topk_hist_kernel<WW><<<hgrid, kSelBlock, 0, s>>>(tk, n, shift, width, prefix, part.ptr, spec_bound, sp,       \
                                                   spec_cnt.ptr, spec_cap)
    switch (kw) {
      case 1: HIST_LAUNCH(1); break;
      case 4: HIST_LAUNCH(4); break;
      case 8: HIST_LAUNCH(8); break;
      default: HIST_LAUNCH(16); break;
    }
#undef HIST_LAUNCH
    BOLT_TRY(fill_u32(hist.ptr, 0, (size_t)1 << width, s));
    topk_hist_sum_kernel<<<dim3((unsigned)(((1 << width) + 255) / 256), 32), 256, 0, s>>>(part.ptr, (int)hgrid,
                                                                                        1 << width, hist.ptr);
    BOLT_HIP(hipGetLastError());
    unsigned long long got_now = 0;
    BOLT_TRY(read_back(s, {{h.data(), hist.ptr, (size_t)(1 << width) * 4}, {&got_now, spec_cnt.ptr, 8}}));
    if (first_digit < 0) spec_got = got_now;
    int64_t cum = 0;
    int d = 0;
    for (; d < (1 << width); d++) {
      if (cum + (int64_t)h[d] >= need) break;
      cum += h[d];
    }
    if (d == (1 << width)) return set_error(BOLT_ERR_OTHER, "bolt_sort_limit: radix select lost rows");
    if (first_digit < 0) first_digit = d;
    below += cum;
    need -= cum;
    eq = h[d];
    prefix = (prefix << width) | (uint64_t)d;
    hi = shift;
    if (eq <= (1 << 16)) break;
  }
  const int64_t Cx = below + eq;  // rows whose image >> hi <= prefix
  if (Cx * 2 > n) return full_sort();  // the leading key ties too often to narrow the rows
  // The candidates: the first pass's guess when it holds every row of the
  // K-th row's first digit and below (a superset of the Cx rows, which the
  // steps below accept), else a collect pass for exactly the Cx rows.
  const uint32_t* cptr;
  int64_t C;
  if (sampled >= 0) {
    cptr = cand.ptr;
    C = sampled;
  } else if (first_digit >= 0 && (uint64_t)first_digit <= spec_bound && (int64_t)spec_got <= spec_cap) {
    cptr = spec.ptr;
    C = (int64_t)spec_got;
  } else {
    BOLT_TRY(cand.alloc((size_t)Cx, s));
    switch (kw) {
      case 1: topk_collect_kernel<1><<<grid, 256, 0, s>>>(tk, n, hi, prefix, cand.ptr, cnt.ptr, Cx); break;
      case 4: topk_collect_kernel<4><<<grid, 256, 0, s>>>(tk, n, hi, prefix, cand.ptr, cnt.ptr, Cx); break;
      case 8: topk_collect_kernel<8><<<grid, 256, 0, s>>>(tk, n, hi, prefix, cand.ptr, cnt.ptr, Cx); break;
      default: topk_collect_kernel<16><<<grid, 256, 0, s>>>(tk, n, hi, prefix, cand.ptr, cnt.ptr, Cx); break;
    }
    BOLT_HIP(hipGetLastError());
    unsigned long long got = 0;
    BOLT_TRY(read_back(s, {{&got, cnt.ptr, 8}}));
    if ((int64_t)got != Cx)
      return set_error(BOLT_ERR_OTHER, "bolt_sort_limit: collected %llu candidates, expected %lld", got, (long long)Cx);
    cptr = cand.ptr;
    C = Cx;
  }
  // One key without NULLs (its image is then exact): narrow the candidates
  // further and sort the few that remain in one workgroup.
  if (n_keys == 1 && !c0.validity && kw != 16 && c0.dtype != BOLT_BOOL && K <= kSmallSort / 2) {
    // continue the select inside the bucket of the first one: `below` rows
    // precede it, the K-th row is the need-th of its `eq`
    uint64_t p2 = prefix;
    int hi2 = hi;
    int64_t below2 = below, need2 = need, eq2 = eq;
    const unsigned ngrid = (unsigned)((C + 255) / 256);
    const unsigned hcgrid = (unsigned)std::min<int64_t>(64, (C + kSelBlock - 1) / kSelBlock);
    while (hi2 > 0 && below2 + eq2 > kSmallSort) {
      const int width = hi2 >= kSelBits ? kSelBits : hi2;
      const int shift = hi2 - width;
      BOLT_TRY(fill_u32(hist.ptr, 0, (size_t)1 << width, s));
      switch (kw) {
        case 1: topk_cand_hist_kernel<1><<<hcgrid, kSelBlock, 0, s>>>(tk, cptr, C, shift, width, p2, hist.ptr); break;
        case 4: topk_cand_hist_kernel<4><<<hcgrid, kSelBlock, 0, s>>>(tk, cptr, C, shift, width, p2, hist.ptr); break;
        default: topk_cand_hist_kernel<8><<<hcgrid, kSelBlock, 0, s>>>(tk, cptr, C, shift, width, p2, hist.ptr); break;
      }
      BOLT_HIP(hipGetLastError());
      BOLT_TRY(read_back(s, {{h.data(), hist.ptr, (size_t)(1 << width) * 4}}));
      int64_t cum = 0;
      int d = 0;
      for (; d < (1 << width); d++) {
        if (cum + (int64_t)h[d] >= need2) break;
        cum += h[d];
      }
      if (d == (1 << width)) return set_error(BOLT_ERR_OTHER, "bolt_sort_limit: candidate select lost rows");
      below2 += cum;
      need2 -= cum;
      eq2 = h[d];
      p2 = (p2 << width) | (uint64_t)d;
      hi2 = shift;
    }
    int64_t C2 = below2 + eq2;
    // More rows tie on the K-th row's whole key than one workgroup sorts:
    // the order among them is by row id, so select the need2-th smallest
    // row id of the tie (14, 14 and 4 bits) and keep the tied rows up to it.
    uint32_t rmax = 0xFFFFFFFFu;
    if (C2 > kSmallSort && hi2 == 0 && below2 + need2 <= kSmallSort) {
      uint32_t rpre = 0;
      int rhi = 32;
      int64_t need3 = need2;
      while (rhi > 0) {
        const int width = rhi >= kSelBits ? kSelBits : rhi;
        const int shift = rhi - width;
        BOLT_TRY(fill_u32(hist.ptr, 0, (size_t)1 << width, s));
        switch (kw) {
          case 1: topk_tie_hist_kernel<1><<<ngrid, 256, 0, s>>>(tk, cptr, C, p2, shift, width, rpre, hist.ptr); break;
          case 4: topk_tie_hist_kernel<4><<<ngrid, 256, 0, s>>>(tk, cptr, C, p2, shift, width, rpre, hist.ptr); break;
          default: topk_tie_hist_kernel<8><<<ngrid, 256, 0, s>>>(tk, cptr, C, p2, shift, width, rpre, hist.ptr); break;
        }
        BOLT_HIP(hipGetLastError());
        BOLT_TRY(read_back(s, {{h.data(), hist.ptr, (size_t)(1 << width) * 4}}));
        int64_t cum = 0;
        int d = 0;
        for (; d < (1 << width); d++) {
          if (cum + (int64_t)h[d] >= need3) break;
          cum += h[d];
        }
        if (d == (1 << width)) return set_error(BOLT_ERR_OTHER, "bolt_sort_limit: tie select lost rows");
        need3 -= cum;
        rpre = (rpre << width) | (uint32_t)d;
        rhi = shift;
      }
      rmax = rpre;  // row ids are distinct: exactly need2 tied rows are <= rmax
      C2 = below2 + need2;
    }
    if (C2 <= kSmallSort) {
      DevBuf<uint32_t> cand2;
      BOLT_TRY(cand2.alloc((size_t)C2, s));
      BOLT_TRY(fill_u32(cnt.ptr, 0, 2, s));
      switch (kw) {
        case 1: topk_cand_collect_kernel<1><<<ngrid, 256, 0, s>>>(tk, cptr, C, hi2, p2, cand2.ptr, cnt.ptr, C2, rmax); break;
        case 4: topk_cand_collect_kernel<4><<<ngrid, 256, 0, s>>>(tk, cptr, C, hi2, p2, cand2.ptr, cnt.ptr, C2, rmax); break;
        default: topk_cand_collect_kernel<8><<<ngrid, 256, 0, s>>>(tk, cptr, C, hi2, p2, cand2.ptr, cnt.ptr, C2, rmax); break;
      }
      BOLT_HIP(hipGetLastError());
      int npow = 1;
      while (npow < C2) npow <<= 1;
      switch (kw) {
        case 1: topk_small_sort_kernel<1><<<1, 1024, 0, s>>>(tk, cand2.ptr, (int)C2, npow, (int)offset, (int)m, out_rows); break;
        case 4: topk_small_sort_kernel<4><<<1, 1024, 0, s>>>(tk, cand2.ptr, (int)C2, npow, (int)offset, (int)m, out_rows); break;
        default: topk_small_sort_kernel<8><<<1, 1024, 0, s>>>(tk, cand2.ptr, (int)C2, npow, (int)offset, (int)m, out_rows); break;
      }
      BOLT_HIP(hipGetLastError());
      unsigned long long got2 = 0;
      BOLT_TRY(read_back(s, {{&got2, cnt.ptr, 8}}));
      if ((int64_t)got2 != C2)
        return set_error(BOLT_ERR_OTHER, "bolt_sort_limit: narrowed to %llu candidates, expected %lld", got2,
                         (long long)C2);
      *n_out = m;
      return BOLT_OK;
    }
  }
  // Sort the candidates by every key, then by row id (the full sort is stable).
  std::vector<DevBuf<uint8_t>> vals(n_keys), valid(n_keys);
  std::vector<bolt_column_t> ck(n_keys + 1);
  for (int k = 0; k < n_keys; k++) {
    const int w = dtype_size(keys[k].dtype);
    BOLT_TRY(vals[k].alloc((size_t)C * w, s));
    memset(&ck[k], 0, sizeof ck[k]);
    ck[k].data = vals[k].ptr;
    if (keys[k].validity) {
      BOLT_TRY(valid[k].alloc((size_t)((C + 7) / 8 + 8), s));
      ck[k].validity = valid[k].ptr;
    }
    BOLT_TRY(bolt_take(stream, &keys[k], cptr, C, &ck[k]));
  }
  memset(&ck[n_keys], 0, sizeof ck[n_keys]);
  ck[n_keys].data = const_cast<uint32_t*>(cptr);  // row ids < 2^31: ascending as Int32
  ck[n_keys].length = C;
  ck[n_keys].dtype = BOLT_I32;
  DevBuf<uint32_t> perm;
  BOLT_TRY(perm.alloc((size_t)C, s));
  BOLT_TRY(bolt_sort_indices(stream, ck.data(), n_keys + 1, desc.data(), nf.data(), perm.ptr));
  topk_emit_kernel<<<(unsigned)((m + 255) / 256), 256, 0, s>>>(cptr, perm.ptr, offset, m, out_rows);
  BOLT_HIP(hipGetLastError());
  BOLT_HIP(hipStreamSynchronize(s));
  *n_out = m;
  return BOLT_OK;
}
