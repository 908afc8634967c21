// Reorder between the accumulators' half-spectrum layout main[kz][ky][kx] +
// nyq[kx][ky] (kz < m, the kz = m plane apart) and the reference's
// [kx][ky][kz], kz <= m.
#pragma once
#include <hip/hip_runtime.h>

namespace mdsf {

// A block moves one ky's tile of kHalfX kx by kHalfK kz through LDS, so that
// both sides are read and written along their own rows: 256-byte runs of kx on
// one side, 512-byte runs of kz on the other.  Element by element in the
// reference's order, the reads of the other side fetched a cache line per value:
// a sum of 512^3 took 1,274 us, one of 256^3 104 us (at the card's copy rate:
// 222 and 28).
constexpr int kHalfX = 32, kHalfK = 64, kHalfThreads = 256;

inline unsigned half_tiles(int nx, int ny, int m) {
  return (unsigned)((long long)((m + 1 + kHalfK - 1) / kHalfK) * ((nx + kHalfX - 1) / kHalfX) * ny);
}

// main / nyq -> out[x][y][kz]: get(kz, y, x) -> V for kz < m, nyq(x, y) -> V,
// put(x, y, kz, V).  One block per tile, kHalfThreads threads.
template <typename V, typename Get, typename Nyq, typename Put>
__device__ __forceinline__ void half_to_rows(int nx, int ny, int m, Get get, Nyq nyq, Put put) {
  __shared__ V t[kHalfK][kHalfX + 1];
  const int tk = (m + 1 + kHalfK - 1) / kHalfK, tx = (nx + kHalfX - 1) / kHalfX;
  const unsigned b = blockIdx.x;
  const int k0 = (int)(b % tk) * kHalfK, x0 = (int)((b / tk) % tx) * kHalfX;
  const int y = (int)(b / ((unsigned)tk * tx));
  const int i = threadIdx.x % kHalfX, r = threadIdx.x / kHalfX;
#pragma unroll
  for (int k = r; k < kHalfK; k += kHalfThreads / kHalfX)
    if (x0 + i < nx && k0 + k <= m) t[k][i] = k0 + k < m ? get(k0 + k, y, x0 + i) : nyq(x0 + i, y);
  __syncthreads();
  const int k = threadIdx.x % kHalfK, q = threadIdx.x / kHalfK;
#pragma unroll
  for (int x = q; x < kHalfX; x += kHalfThreads / kHalfK)
    if (x0 + x < nx && k0 + k <= m) put(x0 + x, y, k0 + k, t[k][x]);
}

// in[x][y][kz] -> main / nyq: get(x, y, kz) -> V, put(kz, y, x, V) for kz < m,
// nyq(x, y, V).
template <typename V, typename Get, typename Put, typename Nyq>
__device__ __forceinline__ void rows_to_half(int nx, int ny, int m, Get get, Put put, Nyq nyq) {
  __shared__ V t[kHalfK][kHalfX + 1];
  const int tk = (m + 1 + kHalfK - 1) / kHalfK, tx = (nx + kHalfX - 1) / kHalfX;
  const unsigned b = blockIdx.x;
  const int k0 = (int)(b % tk) * kHalfK, x0 = (int)((b / tk) % tx) * kHalfX;
  const int y = (int)(b / ((unsigned)tk * tx));
  const int k = threadIdx.x % kHalfK, q = threadIdx.x / kHalfK;
#pragma unroll
  for (int x = q; x < kHalfX; x += kHalfThreads / kHalfK)
    if (x0 + x < nx && k0 + k <= m) t[k][x] = get(x0 + x, y, k0 + k);
  __syncthreads();
  const int i = threadIdx.x % kHalfX, r = threadIdx.x / kHalfX;
#pragma unroll
  for (int kk = r; kk < kHalfK; kk += kHalfThreads / kHalfX)
    if (x0 + i < nx && k0 + kk <= m) {
      if (k0 + kk < m) put(k0 + kk, y, x0 + i, t[kk][i]);
      else nyq(x0 + i, y, t[kk][i]);
    }
}

}  // namespace mdsf
