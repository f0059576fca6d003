// optk_batch.h -- the persistent work loop of the batched trace, shared by
// the float64 and float32 forms (device code; include after
// optk_internal.h).
//
// A launch holds as many blocks as the device keeps resident.  Each block
// takes work tiles (block * rays_per_thread rays of one instance) from a
// global counter until the queue is empty, so instances with 1k rays and
// instances with 64k rays load-balance.  Per tile, the block traces the
// instance's rays -- the records read through the constant address space at
// a uniform index, scalar loads as in the single-system kernels -- and
// reduces per-path statistics of the final positions with wave shuffles and
// one LDS pass: one float64 atomic per statistic per tile.  (Records staged
// in LDS came back in vector registers, and with them every index and branch
// condition they hold: the coatings' records then cost chains of vector
// loads.  Tolerance batch of 256 spectrographs, float32: 1468 us staged,
// 1111 us.)
#pragma once

#include "optk_internal.h"

namespace optk {

#define OPTK_BATCH_MAX_WAVES 8  // 512 threads per block at most

__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// sums acc[0..5] over the block and adds them to stats[0..5]
__device__ __forceinline__ void block_accumulate(double acc[6], double *stats,
                                                 double (*s_red)[6]) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int waves = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int k = 0; k < 6; ++k) acc[k] = wave_sum(acc[k]);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 6; ++k) s_red[wave][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double s = 0.0;
    for (int w = 0; w < waves; ++w) s += s_red[w][threadIdx.x];
    if (s != 0.0) unsafeAtomicAdd(&stats[threadIdx.x], s);
  }
  __syncthreads();
}

// Tracer: select(instance) points it at that instance's records; trace(i, path0, path1, emit) traces ray i along paths path0 ..
// path1 - 1 and calls emit(path, x, y, intensity, unvignetted) for each.
// Two paths at a time share the part of the trace before the orders split.
template <class Tracer>
__device__ __forceinline__ void batch_loop(const BatchArgs &A, Tracer &tr) {
  __shared__ int s_tile;
  __shared__ double s_red[OPTK_BATCH_MAX_WAVES][6];
  const int tid = threadIdx.x;
  const int block = blockDim.x;
  for (;;) {
    if (tid == 0) s_tile = atomicAdd(A.counter, 1);
    __syncthreads();
    const int64_t t = __builtin_amdgcn_readfirstlane(s_tile);
    if (t >= A.num_tiles) break;  // uniform: every thread read the same s_tile
    const BatchTile tile = A.tiles[t];
    tr.select(__builtin_amdgcn_readfirstlane(tile.instance));
    const int paths = tr.num_paths();
    for (int path0 = 0; path0 < paths; path0 += 2) {
      const int path1 = path0 + 2 < paths ? path0 + 2 : paths;
      double acc[2][6] = {{0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
      for (int j = 0; j < A.rays_per_thread; ++j) {
        const int local = tid + j * block;
        if (local < tile.count) {
          tr.trace(tile.start + local, path0, path1,
                   [&](int path, double x, double y, double inten, bool unv) {
                     // a ray that does not count adds zeros (its values may
                     // be infinite: a select, not a product)
                     const double v[6] = {unv ? 1.0 : 0.0, unv ? inten : 0.0, unv ? x : 0.0,
                                          unv ? y : 0.0,   unv ? x * x : 0.0, unv ? y * y : 0.0};
#pragma unroll
                     for (int k = 0; k < 6; ++k) {
                       acc[0][k] += path == path0 ? v[k] : 0.0;
                       acc[1][k] += path == path0 ? 0.0 : v[k];
                     }
                   });
        }
      }
      double *stats = A.stats + ((int64_t)tile.instance * A.num_paths + path0) * OPTK_BATCH_STATS;
      block_accumulate(acc[0], stats, s_red);
      if (path1 - path0 > 1) block_accumulate(acc[1], stats + OPTK_BATCH_STATS, s_red);
    }
    // every thread is past its read of s_tile
    __syncthreads();
  }
}

__device__ __forceinline__ void stage_words(void *dst, const void *src, size_t bytes) {
  uint64_t *d = reinterpret_cast<uint64_t *>(dst);
  const uint64_t *s = reinterpret_cast<const uint64_t *>(src);
  const int words = (int)(bytes / 8);
  for (int w = threadIdx.x; w < words; w += blockDim.x) d[w] = s[w];
}

}  // namespace optk
