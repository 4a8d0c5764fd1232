// fft_two_pass.h -- the plain 256^3 transform, natural order in and out, in two
// passes over the cube (4 volume transfers) instead of one per axis (6).
//
// z is split four-step style, z = 64*z1 + z2 and kz = k1 + 4*k2:
//   X[k1 + 4 k2] = sum_z2 W_64^(z2 k2) W_256^(z2 k1) [ sum_z1 x[64 z1 + z2] W_4^(z1 k1) ]
//   first : tile (z2, 16 adjacent x): y FFT of the 64 lines (z1, x), 4-point DFT
//           over z1; reads runs of 16 points of the natural cube (whole 128-byte
//           lines), writes one contiguous block of the workspace
//   second: tile (k1, ky): twiddle, 64-point DFT over z2 (16 by 4), x FFT of the
//           64 rows k2; reads runs of 16 points, writes whole rows
// INV: the conjugate transform (unnormalised), the same passes.
// A tile is 16384 points (1024 threads); its exchanges move real parts, then
// imaginary parts, so that two work-groups share a CU's LDS.  Both passes are
// bound by memory, and what decides is the run length, which the two tile sizes
// fix together (points of a first and a second tile have
// 16384 * 16384 / 256^3 = 16 points in common): one 256^3 transform takes 97 us
// (5.5 TB/s) against 133-143 in three axis passes; with runs of 2 points read
// from the cube (z1 = 16, 2 x, 8192-point tiles) 132, with runs of 8 (z1 = 4,
// 8 x) 111.  The cube is read, and the result written, once: both go past the
// memory-side cache, which keeps the workspace (98 -> 97 us).
#pragma once
#include "three_pass.h"

namespace cfk {

struct Fft2Geo {
  static constexpr int N = 256, X = 16, Z1 = 4, Z2 = N / Z1;
  static constexpr int LINES = Z1 * X, A_THREADS = LINES * 16, A_TILES = Z2 * (N / X);
  static constexpr int B_THREADS = Z2 * 16, B_TILES = Z1 * N;
  // second pass, rows (k2) of the half-width exchange: 272 = 16 (mod 64), so that
  // 4 rows by 16 points fall on 64 different banks in both directions
  static constexpr int ROW = N + 16;
  // workspace [x/X][z2][k1][ky][x%X]
  __device__ __forceinline__ static int work_index(int x, int z2, int k1, int ky) {
    return ((((x / X) * Z2 + z2) * Z1 + k1) * N + ky) * X + x % X;
  }
};

// First pass, point y of line l = (z1, x%X): 64 lines per y, the groups of 16
// permuted by y so that 4 consecutive y at one z1 fall on different banks too.
struct Fft2Lds {
  float* p;
  int l;
  __device__ __forceinline__ static int at(int y, int l) { return y * Fft2Geo::LINES + (l ^ ((y & 3) * Fft2Geo::X)); }
  __device__ __forceinline__ void st(int y, float v) const { p[at(y, l)] = v; }
  __device__ __forceinline__ float ld(int y) const { return p[at(y, l)]; }
};

template <bool INV>
__device__ __forceinline__ void fft2_first_kernel(const float2* in, float2* out, const float2* tw, int ntotal) {
  using G = Fft2Geo;
  constexpr int N = G::N, X = G::X, Z1 = G::Z1;
  __shared__ float lds[N * G::LINES];
  __shared__ float2 tw_s[N];
  const int tile = (int)blockIdx.x;
  if (tile >= ntotal) return;
  const size_t cube = (size_t)(tile / G::A_TILES) * N * N * N;
  const int tt = tile % G::A_TILES, z2 = tt / (N / X), x0 = (tt % (N / X)) * X;
  const int l = threadIdx.x % G::LINES, yt = threadIdx.x / G::LINES;  // line (z1, x), points y = yt + 16 m
  const Fft2Lds line{lds, l};
  float2 v[16];
  {
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(in + cube, (unsigned)(N * N * N * sizeof(float2)));
    const unsigned voff = (unsigned)(((((l / X) * G::Z2 + z2) * N + yt) * N + x0 + l % X) * sizeof(float2));
#pragma unroll
    for (int m = 0; m < 16; ++m) v[m] = buffer_ld2_nt(rs, voff, (unsigned)(16 * m * N * sizeof(float2)));
  }
  stage_twiddles<N, G::A_THREADS>(tw_s, tw);
  fft_line_half<N, INV>(v, yt, line, tw_s);
  // rows (ky, x%X), consecutive in the block: row r of the thread is threadIdx + 1024 r
  float2 u[4][Z1];
  const int q = threadIdx.x, xl = q % X;
#pragma unroll
  for (int m = 0; m < 16; ++m) line.st(yt + 16 * m, v[m].x);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int z1 = 0; z1 < Z1; ++z1) u[r][z1].x = lds[Fft2Lds::at(q / X + 64 * r, z1 * X + xl)];
  __syncthreads();  // every real part read before the imaginary parts overwrite them
#pragma unroll
  for (int m = 0; m < 16; ++m) line.st(yt + 16 * m, v[m].y);
  __syncthreads();
  float2* dst = out + cube + G::work_index(x0, z2, 0, 0) + q;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int z1 = 0; z1 < Z1; ++z1) u[r][z1].y = lds[Fft2Lds::at(q / X + 64 * r, z1 * X + xl)];
    DFT<Z1, INV>::run(u[r]);  // u[k1]
#pragma unroll
    for (int k1 = 0; k1 < Z1; ++k1) dst[k1 * N * X + G::A_THREADS * r] = u[r][k1];
  }
}

template <bool INV>
__device__ __forceinline__ void fft2_second_kernel(const float2* in, float2* out, const float2* tw, int ntotal) {
  using G = Fft2Geo;
  constexpr int N = G::N, X = G::X, Z1 = G::Z1;
  __shared__ float f[G::Z2 * G::ROW];
  __shared__ float2 tw_s[N];
  const int tile = (int)blockIdx.x;
  if (tile >= ntotal) return;
  const size_t cube = (size_t)(tile / G::B_TILES) * N * N * N;
  const int tt = tile % G::B_TILES, k1 = tt / N, ky = tt % N;
  // column x, thread t of its 4 (lanes 16 apart): z2 = t + 4 m
  const int t = threadIdx.x / 16 % 4, x = threadIdx.x / 64 * 16 + threadIdx.x % 16;
  float2 v[16];
  {
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(in + cube, (unsigned)(N * N * N * sizeof(float2)));
    const unsigned voff = (unsigned)(G::work_index(x, t, k1, ky) * sizeof(float2));
#pragma unroll
    for (int m = 0; m < 16; ++m) v[m] = buffer_ld2(rs, voff, (unsigned)(4 * m * Z1 * N * X * sizeof(float2)));
  }
  stage_twiddles<N, G::B_THREADS>(tw_s, tw);
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = cmulw<INV>(v[m], tw_s[k1 * (t + 4 * m)]);
  // 64 = 16 * 4: DFT over m, then 4 x 4 transposes over the threads t:
  // register 4g + j of thread t is what thread j had for k = 4g + t
  DFT<16, INV>::run(v);
  xpose_swap_stage<1, 2>(v);
  xpose_swap_stage<0, 1>(v);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
#pragma unroll
    for (int j = 1; j < 4; ++j) v[4 * g + j] = cmulw<INV>(v[4 * g + j], tw_s[4 * j * (4 * g + t)]);  // W_64^(j k)
    DFT<4, INV>::run(v + 4 * g);  // register 4g + i: k2 = 4g + t + 16 i
  }
  // columns -> rows k2 (16 threads of a DPP row, x = rt + 16 m), real then imaginary parts
  const int rt = threadIdx.x % 16, row = threadIdx.x / 16;
  float* const colp = f + t * G::ROW + x;
  const float* const rowp = f + row * G::ROW + rt;
  float2 u[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) colp[(j / 4 * 4 + j % 4 * 16) * G::ROW] = v[j].x;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; ++m) u[m].x = rowp[16 * m];
  __syncthreads();  // every real part read before the imaginary parts overwrite them
#pragma unroll
  for (int j = 0; j < 16; ++j) colp[(j / 4 * 4 + j % 4 * 16) * G::ROW] = v[j].y;
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; ++m) u[m].y = rowp[16 * m];
  fft_line<N, INV, true>(u, rt, RowLds{nullptr}, tw_s);  // a row: lanes of one wave
  const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(out + cube, (unsigned)(N * N * N * sizeof(float2)));
  const unsigned voff = (unsigned)((((k1 + Z1 * row) * N + ky) * N + rt) * sizeof(float2));
#pragma unroll
  for (int m = 0; m < 16; ++m) buffer_st2_nt(rs, voff, (unsigned)(16 * m * sizeof(float2)), u[m]);
}

}  // namespace cfk
