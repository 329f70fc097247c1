// Block-level helpers of the kernels: scans, reductions and the mapping of
// workgroups to contiguous chunks of the data.  Every kernel that uses them
// runs workgroups of TPB threads.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "lsg_kernels.hpp"

namespace lsg {

static constexpr int TPB = 256;

// Block-wide exclusive scan of one value per thread (256 threads, 4 waves).
__device__ inline uint32_t blockExclusiveScan(uint32_t v, uint32_t &total) {
  __shared__ uint32_t wsum[TPB / 64];
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[wid] = x;
  __syncthreads();
  uint32_t woff = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < TPB / 64; ++k) {
    uint32_t s = wsum[k];
    if (k < wid) woff += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return x - v + woff;
}

__device__ inline uint32_t blockSum(uint32_t v) {
  uint32_t t;
  blockExclusiveScan(v, t);
  return t;
}

// Logical block index: workgroups are dispatched round-robin over the 8 XCDs
// (each with its own L2), so consecutive logical blocks are mapped to the
// same XCD; a contiguous 1/8 of the data then lives in one L2 and stencil
// neighbours (rows above and below) are found there.
static constexpr uint32_t NUM_XCD = 8;
__device__ inline uint32_t logicalBlock() {
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t xcd = b % NUM_XCD, k = b / NUM_XCD;
  const uint32_t per = nb / NUM_XCD, rem = nb % NUM_XCD;
  return xcd * per + (xcd < rem ? xcd : rem) + k;
}

// Contiguous chunk [lo, hi) of the (logical) block for a device-side size n;
// chunks are multiples of `align` items (the packed keep flags of the
// compaction are written one 64-bit word per wave).
__device__ inline uint32_t chunkSize(uint32_t n, uint32_t align) {
  const uint32_t per = (n + gridDim.x - 1) / gridDim.x;
  return (per + align - 1) / align * align;
}
__device__ inline void blockChunk(uint32_t n, uint32_t &lo, uint32_t &hi, uint32_t align = 64) {
  const uint32_t per = chunkSize(n, align);
  lo = logicalBlock() * per;
  hi = lo + per;
  if (lo > n) lo = n;
  if (hi > n) hi = n;
}

// Sum of partials[0 .. logical block) computed by the whole block.  The
// partials (SCAN_BLOCKS_MAX + 1 counts, 256-byte aligned) are read four at a
// time, every thread's loads issued before the first is used (a loop that
// adds each count as it arrives waits once per load).
__device__ inline uint32_t blockOffset(const uint32_t *partials) {
  static_assert(SCAN_BLOCKS_MAX <= 4 * 4 * TPB, "four uint4 loads per thread cover the partials");
  const uint32_t me = logicalBlock();
  const uint4 *p4 = reinterpret_cast<const uint4 *>(partials);
  uint4 v[4];
  LSG_UNROLL
  for (int r = 0; r < 4; ++r) {
    const uint32_t q = threadIdx.x + (uint32_t)r * TPB;
    v[r] = (4u * q < me) ? p4[q] : make_uint4(0u, 0u, 0u, 0u);
  }
  uint32_t s = 0;
  LSG_UNROLL
  for (int r = 0; r < 4; ++r) {
    const uint32_t k = 4u * (threadIdx.x + (uint32_t)r * TPB);
    s += (k < me ? v[r].x : 0u) + (k + 1 < me ? v[r].y : 0u) + (k + 2 < me ? v[r].z : 0u) + (k + 3 < me ? v[r].w : 0u);
  }
  return blockSum(s);
}

// Block-wide exclusive scan of one 0/1 flag per thread via wave ballots.
__device__ inline uint32_t blockBallotScan(bool k, uint32_t &total, uint64_t &waveMask) {
  __shared__ uint32_t wc[TPB / 64];
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const uint64_t m = (uint64_t)__ballot(k ? 1 : 0);
  const uint32_t lp = (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull));
  if (lane == 0) wc[wid] = (uint32_t)__builtin_popcountll(m);
  __syncthreads();
  uint32_t woff = 0, tot = 0;
#pragma unroll
  for (int q = 0; q < TPB / 64; ++q) {
    uint32_t c = wc[q];
    if (q < wid) woff += c;
    tot += c;
  }
  __syncthreads();
  total = tot;
  waveMask = m;
  return woff + lp;
}

// Block max of non-negative doubles (as ordered bit patterns), then one
// atomicMax per block.
__device__ inline void blockMaxAtomic(unsigned long long v, unsigned long long *dst) {
  __shared__ unsigned long long sm[TPB / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    unsigned long long y = __shfl_down(v, o, 64);
    v = (y > v) ? y : v;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) sm[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = sm[0];
    for (int k = 1; k < TPB / 64; ++k) m = (sm[k] > m) ? sm[k] : m;
    if (m) atomicMax(dst, m);
  }
  __syncthreads();
}

__device__ inline unsigned long long blockSumU64(unsigned long long v) {
  __shared__ unsigned long long sm2[TPB / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) sm2[wid] = v;
  __syncthreads();
  unsigned long long t = 0;
  if (threadIdx.x == 0)
    for (int k = 0; k < TPB / 64; ++k) t += sm2[k];
  __syncthreads();
  return t;
}

}  // namespace lsg
