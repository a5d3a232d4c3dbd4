// reduce_common.h — block-level reduction of aggregate accumulators and the
// deterministic finishing kernel shared by the scalar-aggregate and the
// join-aggregate operators.
#pragma once

#include "ops_common.h"

namespace bolt {

constexpr int kReduceBlock = 256;
constexpr int kWaves = kReduceBlock / 64;

// Reduce NA accumulators across a 256-thread block; thread 0 writes them to
// out[0..NA).  `ops` is read from the uniform AggList.
template <int NA>
__device__ __forceinline__ void block_reduce_store(Acc (&acc)[NA], const AggList& aggs, Acc* out) {
  __shared__ Acc sh[kWaves][NA];
  int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < NA; a++) wave_reduce_acc(acc[a], aggs.a[a].op, aggs.a[a].dtype);
  if (lane == 0) {
#pragma unroll
    for (int a = 0; a < NA; a++) sh[wave][a] = acc[a];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int a = 0; a < NA; a++) {
      Acc r = sh[0][a];
      for (int w = 1; w < kWaves; w++) acc_merge(r, sh[w][a], aggs.a[a].op, aggs.a[a].dtype);
      out[a] = r;
    }
  }
}

// Block a folds the `n_parts` per-block partials of aggregate a (layout
// [part][stride], this list's aggregates from offset `first`) in a fixed order,
// so float results do not depend on scheduling.  One block per aggregate: the
// kernel is bound by the latency of its reads and of the reduction's steps,
// which the aggregates then share instead of queueing for (8192 partials of
// three aggregates: 50 us in one block, 14 us now).
__global__ __launch_bounds__(kReduceBlock) inline void finish_partials_kernel(const Acc* __restrict__ parts,
                                                                             int n_parts, int stride, int first,
                                                                             AggList aggs, Acc* __restrict__ out) {
  const int a = blockIdx.x;
  const int op = aggs.a[a].op, dtype = aggs.a[a].dtype;
  Acc acc[1];
  acc_init(acc[0], op);
  constexpr int kU = 4;  // partials in flight per lane
  for (int p0 = threadIdx.x; p0 < n_parts; p0 += kU * kReduceBlock) {
    Acc x[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int p = p0 + u * kReduceBlock < n_parts ? p0 + u * kReduceBlock : p0;
      x[u] = parts[(int64_t)p * stride + first + a];
    }
#pragma unroll
    for (int u = 0; u < kU; u++)
      if (p0 + u * kReduceBlock < n_parts) acc_merge(acc[0], x[u], op, dtype);
  }
  AggList one;
  one.a[0] = aggs.a[a];
  one.n = 1;
  block_reduce_store<1>(acc, one, out + a);
}

// Launch the finishing kernel for `na` aggregates whose partials sit at offset
// `first` of rows of `stride` accumulators.
int launch_finish(int na, const Acc* parts, int n_parts, int stride, int first, const AggList& chunk, Acc* out,
                  hipStream_t s);

// Split an AggList into chunks of at most 4 (kernels are instantiated for
// 1..4 aggregates so that accumulators stay in registers).
inline AggList agg_chunk(const AggList& all, int first, int count) {
  AggList c;
  c.n = count;
  for (int i = 0; i < count; i++) c.a[i] = all.a[first + i];
  return c;
}

}  // namespace bolt
