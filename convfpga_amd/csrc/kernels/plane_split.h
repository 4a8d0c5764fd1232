// plane_split.h -- one 64^3 cube of the plane plan with its y transform split over
// the passes, y = 8*y1 + y2 and ky = k1 + 8*k2, bit for bit the plane passes' result:
//   rows_fwd : a wave transforms the 8 rows y1 of one (z, y2) along x and takes
//              the 8-point DFT over y1; no barrier, 512-byte rows in and out
//   mid      : a tile (k1, 2 adjacent x) of all z and y2: twiddle and 8-point DFT
//              over y2, z FFT, product with the (natural order) spectrum, and back
//   rows_inv : twiddle, 8-point DFT over k1, x FFT of the rows, final scale
// Value (k1, y2) of plane z is kept in row 8*k1 + y2 of the plane: every pass
// reads and writes the same rows, so all run in place in the output.
// The 64-point column transform of a plane (radix 8 by 8) is cut between its two
// radix steps; the steps themselves, their order (x, y, z and back) and their
// twiddles stay, hence the same bits.
// For one cube, whose passes are three launches of a few microseconds bound by
// one tile's chain of loads, exchanges and stores: the plane passes run 64
// work-groups of 512 threads (a quarter of the CUs), these 128 of 256 and 256 of
// 128, with shorter chains: 13.3 -> 12.4 us per convolution on one signal, 13.8 ->
// 12.3 on 2 GiB of them in turn, 14.3 -> 13.7 with a filter each.  Batches fill the
// GPU with planes and move whole lines in every pass: 2 cubes 15.9 us with the
// plane passes against 16.3, 16 cubes 44.5 against 68; wider middle tiles (4, 8,
// 16 x) come level at 4 to 8 cubes and lose above.
#pragma once
#include "three_pass.h"

namespace cfk {

struct PlaneSplit {
  static constexpr int N = 64, WAVES = 4, THREADS = 64 * WAVES;  // rows passes: a tile per wave
  static constexpr int TILES = N * 8;                            // (z, y2) per cube
  static constexpr int PITCH = N + 8;                            // float2 per row y1: 8 rows x 8 points conflict-free
  static constexpr int WAVE_LDS = 8 * PITCH;
};

template <bool INV>
__device__ __forceinline__ void rows64_kernel(const float2* in, float2* out, const float2* tw, float scale, int ntotal) {
  using G = PlaneSplit;
  constexpr int N = G::N;
  __shared__ float2 lds[G::WAVES * G::WAVE_LDS];
  __shared__ float2 tw_s[N];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if ((int)blockIdx.x >= ntotal) return;
  const int tile = (int)blockIdx.x * G::WAVES + wave;  // (plane, y2)
  const int y2 = tile % 8;
  const int rt = lane % 8, y1 = lane / 8;  // row y1, points x = rt + 8 m; column x = lane
  float2* const seg = lds + wave * G::WAVE_LDS;
  const size_t plane = (size_t)(tile / 8) * N * N;
  float2 v[8];
  const float2* src = in + plane + (INV ? y2 * N + lane : (8 * y1 + y2) * N + rt);
#pragma unroll
  for (int m = 0; m < 8; ++m) v[m] = src[INV ? 8 * m * N : 8 * m];
  stage_twiddles<N, G::THREADS>(tw_s, tw);
  float2* const rowp = seg + y1 * G::PITCH + rt;
  if constexpr (!INV) {
    fft_line<N, false, true>(v, rt, RowLds{seg + y1 * G::PITCH}, tw_s);  // (N + N/16 <= PITCH)
#pragma unroll
    for (int m = 0; m < 8; ++m) rowp[8 * m] = v[m];
    lds_sync<true>();
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = seg[j * G::PITCH + lane];
    DFT<8, false>::run(v);  // v[k1]
    float2* dst = out + plane + y2 * N + lane;
#pragma unroll
    for (int k1 = 0; k1 < 8; ++k1) dst[8 * k1 * N] = v[k1];
  } else {
#pragma unroll
    for (int k1 = 1; k1 < 8; ++k1) v[k1] = cmulw<true>(v[k1], tw_s[k1 * y2]);
    DFT<8, true>::run(v);  // v[y1]
#pragma unroll
    for (int j = 0; j < 8; ++j) seg[j * G::PITCH + lane] = v[j];
    lds_sync<true>();
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = rowp[8 * m];
    lds_sync<true>();
    fft_line<N, true, true>(v, rt, RowLds{seg + y1 * G::PITCH}, tw_s);
    float2* dst = out + plane + (8 * y1 + y2) * N + rt;
#pragma unroll
    for (int m = 0; m < 8; ++m) dst[8 * m] = cscale(v[m], scale);
  }
}

struct MidSplit {
  static constexpr int N = 64, GM = 2, THREADS = 64 * GM, LINES = 8 * GM, TILES = 8 * (N / GM);
  static constexpr int SIBLINGS = 16 / GM;  // tiles that share 128-byte lines
  static constexpr int PITCH = LINES + 1;
  static constexpr int LDS = N * PITCH;
};
__device__ __forceinline__ void mid64_kernel(const float2* in, float2* out, const float2* H, const float2* tw,
                                             long long hstride, int ntotal) {
  using G = MidSplit;
  constexpr int N = G::N, GM = G::GM, PITCH = G::PITCH;
  static_assert(G::TILES % (8 * G::SIBLINGS) == 0, "tile count must be a multiple of 8*siblings");
  __shared__ float2 lds[G::LDS];
  __shared__ float2 tw_s[N];
  const int tile = xcd_group_tile<G::SIBLINGS>((int)blockIdx.x);
  if (tile >= ntotal) return;
  const int cube = tile / G::TILES, tt = tile % G::TILES, k1 = tt / (N / GM), x0 = tt % (N / GM) * GM;
  const int xl = threadIdx.x % GM, z = threadIdx.x / GM;          // (z, x): the 8 values of y2 / k2
  const int l = threadIdx.x % G::LINES, zt = threadIdx.x / G::LINES;  // line (k2, x), points z = zt + 8 m
  const size_t base = (size_t)cube * N * N * N + (size_t)(z * N + 8 * k1) * N + x0 + xl;
  float2 v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = in[base + j * N];
  stage_twiddles<N, G::THREADS>(tw_s, tw);
#pragma unroll
  for (int j = 1; j < 8; ++j) v[j] = cmulw<false>(v[j], tw_s[j * k1]);
  DFT<8, false>::run(v);  // v[k2]
  const PitchLds<PITCH> view{lds + l};
  float2* const zp = lds + z * PITCH + xl;  // k2 at k2 * GM
#pragma unroll
  for (int j = 0; j < 8; ++j) zp[j * GM] = v[j];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 8; ++m) v[m] = view.ld(zt + 8 * m);
  __syncthreads();
  fft_line<N, false>(v, zt, view, tw_s);
  const float2* hp = H + (size_t)cube * hstride + (size_t)(zt * N + k1 + 8 * (l / GM)) * N + x0 + l % GM;
#pragma unroll
  for (int m = 0; m < 8; ++m) v[m] = cmul(v[m], hp[8 * m * N * N]);
  fft_line<N, true>(v, zt, view, tw_s);
#pragma unroll
  for (int m = 0; m < 8; ++m) view.st(zt + 8 * m, v[m]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = zp[j * GM];
  DFT<8, true>::run(v);  // v[y2]
#pragma unroll
  for (int j = 0; j < 8; ++j) out[base + j * N] = v[j];
}

}  // namespace cfk
