// small_cube.h -- a whole cube of edge 8 or 16 per work-group: the plain 3D
// transform, and the convolution, as one launch that reads the cube once and
// writes it once.
//
// A 16^3 cube is 32 KiB: N^2 threads hold it with one line of N points each, so
// a line's DFT (one radix-N step) needs no exchange at all and the lines of the
// three axes are turned into each other through LDS.  As five axis passes
// (x, y, z*H*z, y^-1, x^-1), such a cube is five launches whose kernels each
// take 2-3 us for 64 KiB of traffic; here it is one: back-to-back calls on one
// 16^3 cube 15.7 -> 6.0 us each.  What bounds it is the launch and the chain of
// one work-group (load, six transforms, six exchanges, store).  The lines are
// transformed in the order of the axis passes with the same DFT code, so the
// results are the same bits.
#pragma once
#include "fft_core.h"

namespace cfk {

template <int N>
struct CubeCfg {
  static_assert(Shape<N>::P == N, "a line per thread: edges whose line is one radix step");
  static constexpr int THREADS = N * N, P = N;
  // (z, y, x) at z*PZ + y*PY + x: at N = 16 a half-wave's 8-byte accesses along
  // any axis fall on 32 different bank pairs (one pair of lanes shares one in
  // the rows of x), at N = 8 nearly so
  static constexpr int PY = N + 1, PZ = N * PY;
  static constexpr int LDS = N * PZ;
};

// MODE 0 forward transform, 1 inverse, 2 forward * H then inverse with `scale`
template <int N, int MODE>
__device__ __forceinline__ void cube_kernel(const float2* in, float2* out, const float2* H, long long hstride,
                                            float scale, int ntotal) {
  using K = CubeCfg<N>;
  constexpr int PY = K::PY, PZ = K::PZ;
  __shared__ float2 lds[K::LDS];
  const int cube = blockIdx.x;
  if (cube >= ntotal) return;
  const int l = threadIdx.x, lo = l % N, hi = l / N;
  const float2* src = in + (size_t)cube * (N * N * N) + l;
  float2* dst = out + (size_t)cube * (N * N * N) + l;
  float2* const xline = lds + hi * PZ + lo * PY;  // thread (y = lo, z = hi), x = m
  float2* const yline = lds + hi * PZ + lo;       // thread (x = lo, z = hi), y = m at m * PY
  float2* const zline = lds + hi * PY + lo;       // thread (x = lo, y = hi), z = m at m * PZ
  float2 v[N], h[MODE == 2 ? N : 1];
  // the thread's z line: consecutive lanes, consecutive addresses
#pragma unroll
  for (int m = 0; m < N; ++m) v[m] = src[m * N * N];
  if constexpr (MODE == 2) {  // in flight while the forward half runs
    const float2* hp = H + (size_t)cube * hstride + l;
#pragma unroll
    for (int m = 0; m < N; ++m) h[m] = hp[m * N * N];
  }
  if constexpr (MODE != 1) {
#pragma unroll
    for (int m = 0; m < N; ++m) zline[m * PZ] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = xline[m];
    DFT<N, false>::run(v);
#pragma unroll
    for (int m = 0; m < N; ++m) xline[m] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = yline[m * PY];
    DFT<N, false>::run(v);
#pragma unroll
    for (int m = 0; m < N; ++m) yline[m * PY] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = zline[m * PZ];
    DFT<N, false>::run(v);
  }
  if constexpr (MODE == 2) {
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = cmul(v[m], h[m]);
  }
  if constexpr (MODE != 0) {
    // (each thread overwrites only the z line it has read itself)
    DFT<N, true>::run(v);
#pragma unroll
    for (int m = 0; m < N; ++m) zline[m * PZ] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = yline[m * PY];
    DFT<N, true>::run(v);
#pragma unroll
    for (int m = 0; m < N; ++m) yline[m * PY] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = xline[m];
    DFT<N, true>::run(v);
#pragma unroll
    for (int m = 0; m < N; ++m) xline[m] = cscale(v[m], scale);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = zline[m * PZ];
  }
#pragma unroll
  for (int m = 0; m < N; ++m) dst[m * N * N] = v[m];
}

}  // namespace cfk
