// sort_split.h — the splitter sort: (64-bit key, u32 value) pairs of up to
// 2^25 rows, any key distribution.  Included by sort.hip only.
//
// A radix sort by fixed digits needs keys that spread over those digits:
// floats around a common magnitude, dates or group keys put most rows in a few
// buckets of their top bytes, and the plain LSD sort then runs eight passes
// over HBM.  Here the buckets come from the data: a stratified sample is
// ranked, its quantiles are the splitters, and each key's bucket number (its
// code, up to 16 bits) is the rank of its splitter interval, found by binary
// search in LDS, with the interval cut linearly in up to four.  One stable onesweep
// pass (two above 2^17 rows) by the code's digits groups the rows by bucket,
// and one workgroup sorts each bucket of a few hundred rows in LDS, in place.
//   * A value that is drawn twice as a splitter gets a bucket of its own
//     ([v, v + 1)), of any size, which needs no further sort: the passes are
//     stable.
//   * A bucket of different keys above the LDS sort's capacity (a value or a
//     narrow range that the sample missed) makes the caller fall back to LSD
//     passes from the untouched input.
//   * Up to 6,144 rows one workgroup sorts alone: one launch.
// Uniform int64 keys, whole call, before (LSD or digit buckets) and now: 5,000
// rows 214 -> 17 us, 20,000 232 -> 93, 100,000 234 -> 107, 1M 304 -> 206, 5M
// 958 -> 427, 30M 1752 -> 1076 (by digits, with these bucket sorts).
#pragma once

namespace bolt {

constexpr int64_t kSplitMax = (int64_t)1 << 25;    // above: the digit hybrid (its buckets are 16 bits of digits)
constexpr int64_t kSplitFirst = (int64_t)1 << 23;  // above: a histogram of the keys' bytes first
constexpr int64_t kSplitOnePass = (int64_t)1 << 17;  // up to here 256 buckets of 512 rows on average
constexpr int kCodeBlock = 1024;

// Splitter list of a sorted sample of S keys, for G (a power of two) intervals:
// splitter p (1 .. G - 1) is the (p - 1)-th of G - 1 quantiles, the smallest and
// the largest sample among them; a repeated one becomes the value after it.
struct Splitters {
  const uint64_t* sorted;
  int S, G, sub_bits;  // every interval is cut in 2^sub_bits (up to 4) linearly
};

__device__ __forceinline__ uint64_t sample_quantile(const Splitters& sp, int p) {
  return sp.sorted[(uint32_t)(p - 1) * (uint32_t)(sp.S - 1) / (uint32_t)(sp.G - 2)];  // below 2^28
}
__device__ __forceinline__ uint64_t splitter(const Splitters& sp, int p) {
  if (p <= 0) return 0;
  if (p >= sp.G) return ~0ull;
  const uint64_t v = sample_quantile(sp, p);
  return p > 1 && v != ~0ull && sample_quantile(sp, p - 1) == v ? v + 1 : v;
}
// Smallest key of code b: code(key) >= b exactly when key >= code_start(b).
__device__ __forceinline__ uint64_t code_start(const Splitters& sp, int b) {
  const int p = b >> sp.sub_bits, q = b & ((1 << sp.sub_bits) - 1);
  const uint64_t lo = splitter(sp, p);
  if (q == 0) return lo;
  const uint64_t r = splitter(sp, p + 1) - lo, unit = r >> sp.sub_bits;
  const uint64_t off = unit ? (uint64_t)q * unit : (uint64_t)q;
  return lo + (off < r ? off : r);
}

// Steps of a bitonic sort in LDS of `size` elements: every comparator sorts
// ascending (the first step of a merge mirrors its second half), so positions
// past `size` act as +infinity and are skipped.  `cmpx(a, b)` orders elements
// a < b.  The 64 pairs of a wave lie in one stretch of 128 elements when the
// stride is at most 64, so only longer strides need the workgroup's barrier.
template <int BLOCK, typename F>
__device__ __forceinline__ void lds_bitonic(int size, F cmpx) {
  int npow = 2;
  while (npow < size) npow <<= 1;
  for (int len = 2; len <= npow; len <<= 1)
    for (int st = len >> 1; st > 0; st >>= 1) {
      if (st > 64 || (st == 64 && len > 128) || (st == len >> 1 && len > 128)) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int q = threadIdx.x; q < npow / 2; q += BLOCK) {
        const int off = q & (st - 1), base = (q - off) * 2;
        const int a = base + off;
        const int b = st == len >> 1 ? base + 2 * st - 1 - off : a + st;
        if (b < size) cmpx(a, b);
      }
    }
  __syncthreads();
}

// The sample: one row of each of S equal strata, at a scattered place within
// it, sorted in lists of 1024.  The workgroups behind those of the lists, if any,
// read all keys for the bits that vary: workgroup g's share of the keys has the
// bits one_zero[2 g] set in some key, one_zero[2 g + 1] clear in some.
constexpr int kSampleList = 1024;
constexpr int kVaryRows = 8;      // keys in flight per lane
constexpr int kVaryGrid = 256;
__global__ __launch_bounds__(kSampleList) void split_sample_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                   uint64_t in_xor, int S,
                                                                   uint64_t* __restrict__ lists,
                                                                   uint64_t* __restrict__ one_zero) {
  __shared__ uint64_t k[kSampleList];
  if ((int)blockIdx.x >= S / kSampleList) {
    const int g = (int)blockIdx.x - S / kSampleList, grid = (int)gridDim.x - S / kSampleList;
    const int64_t stride = (int64_t)grid * kSampleList;
    uint64_t one = 0, zero = 0;
    for (int64_t i0 = (int64_t)g * kSampleList + threadIdx.x; i0 < n; i0 += stride * kVaryRows) {
      uint64_t x[kVaryRows];
#pragma unroll
      for (int u = 0; u < kVaryRows; u++) x[u] = keys[i0 + u * stride < n ? i0 + u * stride : i0];
#pragma unroll
      for (int u = 0; u < kVaryRows; u++) {
        one |= x[u];
        zero |= ~x[u];
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      one |= __shfl_xor(one, m);
      zero |= __shfl_xor(zero, m);
    }
    if ((threadIdx.x & 63) == 0) {
      k[threadIdx.x >> 6] = one;
      k[64 + (threadIdx.x >> 6)] = zero;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      uint64_t r = 0;
      for (int w = 0; w < kSampleList / 64; w++) r |= k[64 * threadIdx.x + w];
      one_zero[2 * g + threadIdx.x] = r;
    }
    return;
  }
  const int j = blockIdx.x * kSampleList + threadIdx.x;
  const int64_t lo = (int64_t)j * n / S, hi = (int64_t)(j + 1) * n / S;
  const uint32_t h = (uint32_t)j * 0x9E3779B1u;
  k[threadIdx.x] = keys[lo + (int64_t)(((uint64_t)h * (uint64_t)(hi - lo)) >> 32)] ^ in_xor;
  __syncthreads();
  lds_bitonic<kSampleList>(kSampleList, [&](int a, int b) {
    const uint64_t x = k[a], y = k[b];
    if (x > y) {
      k[a] = y;
      k[b] = x;
    }
  });
  lists[j] = k[threadIdx.x];
}

// Merges the LISTS sorted lists: the rank of a key is its place in its own list
// plus, by binary search, the keys of the others that precede it (equal keys
// of earlier lists do).  The searches of all lists run interleaved; one wave
// per workgroup spreads their scattered reads over the CUs.
template <int LISTS>
__global__ __launch_bounds__(64) void split_merge_kernel(const uint64_t* __restrict__ lists,
                                                          uint64_t* __restrict__ sorted) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  const uint64_t k = lists[j];
  const int own = j / kSampleList;  // block-uniform
  int at[LISTS];
#pragma unroll
  for (int l = 0; l < LISTS; l++) at[l] = -1;  // last key that precedes k
#pragma unroll 1
  for (int step = kSampleList / 2; step > 0; step >>= 1) {
#pragma unroll
    for (int l = 0; l < LISTS; l++) {
      const uint64_t x = lists[l * kSampleList + at[l] + step];
      if (l < own ? x <= k : x < k) at[l] += step;
    }
  }
  uint32_t r = (uint32_t)(j & (kSampleList - 1));
#pragma unroll
  for (int l = 0; l < LISTS; l++) {
    if (l == own) continue;
    // the steps above reach 1023 of the 1024 keys
    const uint64_t x = lists[l * kSampleList + at[l] + 1];
    r += (uint32_t)(at[l] + 1) + ((l < own ? x <= k : x < k) ? 1u : 0u);
  }
  sorted[r] = k;
}

// *out = the sample's distinct keys.
__global__ __launch_bounds__(1024) void split_distinct_kernel(const uint64_t* __restrict__ sorted, int S,
                                                              uint32_t* __restrict__ out) {
  __shared__ uint32_t wsum[16];
  uint32_t c = 0;
  for (int i = threadIdx.x; i < S; i += 1024) c += i == 0 || sorted[i] != sorted[i - 1] ? 1u : 0u;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) c += __shfl_xor(c, m);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) c += wsum[w];
    *out = c;
  }
}

// Code of every key, and the counts of both digits of the codes (hist[0..255]:
// the low b1 bits, hist[256..511]: the rest).  Bound by the LDS searches, 6 to
// 14 dependent reads a key, four keys in flight per lane.
__global__ __launch_bounds__(kCodeBlock) void split_code_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                uint64_t in_xor, Splitters sp, int b1,
                                                                uint16_t* __restrict__ codes,
                                                                uint32_t* __restrict__ hist) {
  extern __shared__ uint64_t spl[];  // [G + 1]
  __shared__ uint32_t h[512];
  for (int p = threadIdx.x; p <= sp.G; p += kCodeBlock) spl[p] = splitter(sp, p);
  for (int i = threadIdx.x; i < 512; i += kCodeBlock) h[i] = 0;
  __syncthreads();
  constexpr int R = 4;
  const uint32_t m1 = (1u << b1) - 1;
  const int64_t stride = (int64_t)gridDim.x * kCodeBlock;
  for (int64_t i0 = (int64_t)blockIdx.x * kCodeBlock + threadIdx.x; i0 < n; i0 += stride * R) {
    uint64_t k[R];
    int p[R];
#pragma unroll
    for (int u = 0; u < R; u++) {
      const int64_t i = i0 + u * stride;
      k[u] = keys[i < n ? i : n - 1] ^ in_xor;
      p[u] = 0;
    }
    for (int step = sp.G >> 1; step > 0; step >>= 1) {
#pragma unroll
      for (int u = 0; u < R; u++)
        if (spl[p[u] + step] <= k[u]) p[u] += step;
    }
#pragma unroll
    for (int u = 0; u < R; u++) {
      uint32_t c = (uint32_t)p[u];
      if (sp.sub_bits) {
        const uint64_t lo = spl[p[u]], d = k[u] - lo;
        uint64_t unit = (spl[p[u] + 1] - lo) >> sp.sub_bits;
        if (unit == 0) unit = 1;
        uint32_t q = (uint32_t)(d >= unit);
        if (sp.sub_bits == 2) q += (uint32_t)(d >= 2 * unit) + (uint32_t)(d >= 3 * unit);
        c = (c << sp.sub_bits) + q;
      }
      const int64_t i = i0 + u * stride;
      if (i < n) {
        codes[i] = (uint16_t)c;
        atomicAdd(&h[c & m1], 1u);
        atomicAdd(&h[256 + (c >> b1)], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 512; i += kCodeBlock)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// Exclusive scans of the two digits' counts (block 0: low, block 1: high),
// 257 entries each.
__global__ __launch_bounds__(256) void split_scan_kernel(const uint32_t* __restrict__ hist,
                                                         uint32_t* __restrict__ offs) {
  __shared__ uint32_t wtot[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t c = hist[blockIdx.x * 256 + t];
  uint32_t inc = c;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t v = __shfl_up(inc, d);
    if (lane >= d) inc += v;
  }
  if (lane == 63) wtot[wave] = inc;
  __syncthreads();
  for (int w = 0; w < wave; w++) inc += wtot[w];
  uint32_t* o = offs + blockIdx.x * 257;
  o[t] = inc - c;
  if (t == 255) o[256] = inc;
}

// start[b] = first row of code b, b = 0 .. C (rows are grouped by code).
__global__ __launch_bounds__(256) void split_bounds_kernel(const uint64_t* __restrict__ keys, int64_t n, uint64_t x,
                                                           Splitters sp, int C, uint32_t* __restrict__ start) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b > C) return;
  int64_t lo = 0, hi = n;
  if (b == C) lo = n;
  else if (b > 0) {
    const uint64_t first = code_start(sp, b);
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((keys[mid] ^ x) < first) lo = mid + 1;
      else hi = mid;
    }
  }
  start[b] = (uint32_t)lo;
}

// ---- bucket sorts in LDS ------------------------------------------------------
//
// Stable sort of rows [s0, s0 + size) by key: one counting pass on the 10 to 12
// bits below the top bit of the bucket's key range, then an insertion sort of
// each sub-bucket by (key, position).  The values
// stay in memory and are gathered at the end (all of them before the first is
// overwritten), which leaves LDS for more workgroups.  Buckets with a sub-bucket above kSubMax rows
// take a bitonic network instead, which suits any keys.
template <int BLOCK, int ITEMS>
struct SplitLds {
  static constexpr int kMax = BLOCK * ITEMS;
  static constexpr int kCnt = BLOCK * 4;
  uint64_t k[kMax];
  uint16_t idx[kMax];
  uint32_t cnt[kCnt];
  uint64_t red[2][BLOCK / 64];
  uint32_t tot[BLOCK / 64];
  uint32_t big;
};
constexpr uint32_t kSubMax = 12;  // longer insertion sorts cost more than the network (576 steps for 48 rows)

template <int BLOCK, int ITEMS>
__device__ __forceinline__ void split_local_sort(SplitLds<BLOCK, ITEMS>& L, const uint64_t* kin, const uint32_t* vin,
                                                 uint64_t* kout, uint32_t* vout, int64_t s0, int size, uint64_t in_xor,
                                                 uint64_t out_xor) {
  using Lds = SplitLds<BLOCK, ITEMS>;
  constexpr int kWaves = BLOCK / 64;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  uint64_t k[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const int i = j * BLOCK + t;
    const int ic = i < size ? i : size - 1;
    k[j] = kin[s0 + ic] ^ in_xor;
  }
  uint64_t mn = ~0ull, mx = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    mn = k[j] < mn ? k[j] : mn;
    mx = k[j] > mx ? k[j] : mx;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const uint64_t a = __shfl_xor(mn, m), b = __shfl_xor(mx, m);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  if (lane == 0) {
    L.red[0][wave] = mn;
    L.red[1][wave] = mx;
  }
  for (int i = t; i < Lds::kCnt; i += BLOCK) L.cnt[i] = 0;
  if (t == 0) L.big = 0;
  __syncthreads();
  for (int w = 0; w < kWaves; w++) {
    mn = L.red[0][w] < mn ? L.red[0][w] : mn;
    mx = L.red[1][w] > mx ? L.red[1][w] : mx;
  }
  if (mn == mx) {  // block-uniform: equal keys keep their order
    if (kin != kout) {
#pragma unroll
      for (int j = 0; j < ITEMS; j++) {
        const int i = j * BLOCK + t;
        if (i < size) {
          kout[s0 + i] = k[j] ^ out_xor;
          vout[s0 + i] = vin[s0 + i];
        }
      }
    }
    return;
  }
  constexpr int kCntBits = Lds::kCnt == 1024 ? 10 : Lds::kCnt == 2048 ? 11 : 12;
  static_assert(Lds::kCnt == 1 << kCntBits, "counter bits");
  const int h = 63 - __clzll(mx - mn);  // top bit of the range
  const int dsh = h >= kCntBits ? h - (kCntBits - 1) : 0;
#pragma unroll
  for (int j = 0; j < ITEMS; j++)
    if (j * BLOCK + t < size) atomicAdd(&L.cnt[(uint32_t)((k[j] - mn) >> dsh)], 1u);
  __syncthreads();
  {
    const uint32_t c0 = L.cnt[4 * t], c1 = L.cnt[4 * t + 1], c2 = L.cnt[4 * t + 2], c3 = L.cnt[4 * t + 3];
    const uint32_t local = c0 + c1 + c2 + c3;
    uint32_t inc = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t x = __shfl_up(inc, d);
      if (lane >= d) inc += x;
    }
    if (lane == 63) L.tot[wave] = inc;
    if (max(max(c0, c1), max(c2, c3)) > kSubMax) L.big = 1;
    __syncthreads();
    uint32_t carry = 0;
    for (int w = 0; w < wave; w++) carry += L.tot[w];
    const uint32_t ex = carry + inc - local;
    L.cnt[4 * t] = ex;
    L.cnt[4 * t + 1] = ex + c0;
    L.cnt[4 * t + 2] = ex + c0 + c1;
    L.cnt[4 * t + 3] = ex + c0 + c1 + c2;
  }
  __syncthreads();
  if (L.big == 0) {
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int i = j * BLOCK + t;
      if (i < size) {
        const uint32_t at = atomicAdd(&L.cnt[(uint32_t)((k[j] - mn) >> dsh)], 1u);
        L.k[at] = k[j];
        L.idx[at] = (uint16_t)i;
      }
    }
    __syncthreads();
    // cnt[d] is now the end of sub-bucket d
    for (int d = t; d < Lds::kCnt; d += BLOCK) {
      const int b = d ? (int)L.cnt[d - 1] : 0, e = (int)L.cnt[d];
      for (int x = b + 1; x < e; x++) {
        const uint64_t w = L.k[x];
        const uint16_t wi = L.idx[x];
        int y = x - 1;
        while (y >= b && (L.k[y] > w || (L.k[y] == w && L.idx[y] > wi))) {
          L.k[y + 1] = L.k[y];
          L.idx[y + 1] = L.idx[y];
          y--;
        }
        L.k[y + 1] = w;
        L.idx[y + 1] = wi;
      }
    }
    __syncthreads();
    uint32_t vv[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int i = j * BLOCK + t;
      vv[j] = vin[s0 + (i < size ? L.idx[i] : 0)];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int i = j * BLOCK + t;
      if (i < size) {
        kout[s0 + i] = L.k[i] ^ out_xor;
        vout[s0 + i] = vv[j];
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const int i = j * BLOCK + t;
    if (i < size) {
      L.k[i] = k[j];
      L.idx[i] = (uint16_t)i;
    }
  }
  __syncthreads();
  lds_bitonic<BLOCK>(size, [&](int a, int b) {
    const uint64_t ka = L.k[a], kb = L.k[b];
    const uint16_t ia = L.idx[a], ib = L.idx[b];
    if (ka > kb || (ka == kb && ia > ib)) {
      L.k[a] = kb;
      L.k[b] = ka;
      L.idx[a] = ib;
      L.idx[b] = ia;
    }
  });
    uint32_t vv[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int i = j * BLOCK + t;
      vv[j] = vin[s0 + (i < size ? L.idx[i] : 0)];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int i = j * BLOCK + t;
      if (i < size) {
        kout[s0 + i] = L.k[i] ^ out_xor;
        vout[s0 + i] = vv[j];
      }
    }
}

// Rows of the three bucket kernels.
// The first holds nearly all buckets (20 KB of LDS: eight workgroups a CU).
constexpr int kSplitSmall = 256 * 6;
constexpr int kSplitMid = 512 * 8;
constexpr int kSplitLarge = 1024 * 10;
constexpr int kSplitWhole = 1024 * 6;  // a whole input, by one workgroup

// A bucket of one value only, by construction of its splitters.
__device__ __forceinline__ bool code_constant(const Splitters& sp, int b, int C) {
  const uint64_t v = code_start(sp, b);
  return v == ~0ull || (b + 1 < C && code_start(sp, b + 1) == v + 1);
}

// One workgroup per bucket; larger buckets are left to split_list_kernel.
__global__ __launch_bounds__(256) void split_small_kernel(uint64_t* keys, uint32_t* vals,
                                                          const uint32_t* __restrict__ start, uint64_t x) {
  __shared__ SplitLds<256, 6> L;
  const uint32_t s0 = start[blockIdx.x];
  const int64_t size = (int64_t)start[blockIdx.x + 1] - s0;
  if (size < 2 || size > kSplitSmall) return;
  split_local_sort(L, keys, vals, keys, vals, s0, (int)size, x, x);
}

// Each workgroup looks at LOOK buckets and sorts those of above `lo` rows that
// it holds.  In the last such kernel err is set for a bucket of different keys
// that does not fit (`sp.sorted` null: buckets by digits, none of which is
// known to be constant).
template <int BLOCK, int ITEMS, int LOOK, bool LAST>
__global__ __launch_bounds__(BLOCK) void split_list_kernel(uint64_t* keys, uint32_t* vals,
                                                           const uint32_t* __restrict__ start, int C, Splitters sp,
                                                           int lo, uint64_t x, uint32_t* __restrict__ err) {
  __shared__ SplitLds<BLOCK, ITEMS> L;
  __shared__ int list[LOOK];
  __shared__ int n_list;
  if (threadIdx.x == 0) n_list = 0;
  __syncthreads();
  const int b = blockIdx.x * LOOK + threadIdx.x;
  if (threadIdx.x < LOOK && b < C) {
    const int64_t size = (int64_t)start[b + 1] - start[b];
    if (size > lo) {
      if (size <= BLOCK * ITEMS) list[atomicAdd(&n_list, 1)] = b;
      else if (LAST && !(sp.sorted && code_constant(sp, b, C))) atomicOr(err, 1u);
    }
  }
  __syncthreads();
  for (int q = 0; q < n_list; q++) {
    const uint32_t s0 = start[list[q]];
    split_local_sort(L, keys, vals, keys, vals, s0, (int)(start[list[q] + 1] - s0), x, x);
    __syncthreads();
  }
}

static void launch_bucket_sorts(uint64_t* keys, uint32_t* vals, const uint32_t* start, int C, const Splitters& sp,
                                uint64_t x, uint32_t* err, hipStream_t s) {
  split_small_kernel<<<C, 256, 0, s>>>(keys, vals, start, x);
  // a few hundred buckets: one launch for all larger ones
  const bool few = C <= 256;
  if (!few)
    split_list_kernel<512, 8, 16, false><<<(C + 15) / 16, 512, 0, s>>>(keys, vals, start, C, sp, kSplitSmall, x, err);
  if (few)
    split_list_kernel<1024, 10, 4, true><<<(C + 3) / 4, 1024, 0, s>>>(keys, vals, start, C, sp, kSplitSmall, x, err);
  else
    split_list_kernel<1024, 10, 64, true><<<(C + 63) / 64, 1024, 0, s>>>(keys, vals, start, C, sp, kSplitMid, x, err);
}

// An input of up to kSplitWhole rows.
__global__ __launch_bounds__(1024) void split_whole_kernel(const uint64_t* kin, const uint32_t* vin, uint64_t* kout,
                                                           uint32_t* vout, int n, uint64_t in_xor, uint64_t out_xor) {
  __shared__ SplitLds<1024, 6> L;
  split_local_sort(L, kin, vin, kout, vout, 0, n, in_xor, out_xor);
}

}  // namespace bolt
