// plane_pair.h -- the plane plan's passes for a batch of 64^3 and a batch of 32^3
// cubes in one launch per pass: the work-groups of the 32^3 tiles follow those of
// the 64^3 tiles.  A pass that waits for the one before costs 4-5 us from its
// launch, its first loads and its tail alone, more than 16 cubes of 32^3 take to
// move (4 MiB a pass); in one launch the two batches share it: 8 x 64^3 and
// 16 x 32^3 as one graph 53 -> 38 us.  The tiles are the plane passes' own, with
// the 32^3 planes four to a work-group of the 64^3 plane's 512 threads (35 KiB of
// LDS, 33 registers: the four 64^3 work-groups per CU of the plane pass itself);
// the results are the same bits.
#pragma once
#include "../geometry.h"
#include "axis_passes.h"
#include "three_pass.h"

namespace cfk {

// One batch's part of a launch (cfgeo::PairPart of the host).
struct PairPart {
  const float2* in;
  float2* out;
  const float2* H;
  const float2* tw;
  long long hstride;
  float scale;
  int groups;  // work-groups
};
static_assert(sizeof(PairPart) == sizeof(cfgeo::PairPart), "pair descriptor");

template <int N, bool INV>
__device__ __forceinline__ void pair_plane_part(const PairPart& p, int group, float2* lds, float2* tw_s) {
  using K = PlaneCfg<N>;
  constexpr int SUB = cfgeo::pair_threads / K::THREADS;  // planes side by side
  const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / K::THREADS), x = threadIdx.x % K::THREADS;
  const PlanePass<N, INV> k{p.in, p.out, tw_s, lds + g * K::LDS, p.scale, x % K::T, x / K::T, x % N, x / N};
  typename PlanePass<N, INV>::Regs r;
  k.load(group * SUB + g, r);
  stage_twiddles<N, cfgeo::pair_threads>(tw_s, p.tw);
  k.process(group * SUB + g, r);
}

template <bool INV>
__device__ __forceinline__ void pair_plane_kernel(const PairPart& a, const PairPart& b) {
  constexpr int L32 = cfgeo::pair_threads / PlaneCfg<32>::THREADS * PlaneCfg<32>::LDS;
  __shared__ float2 lds[PlaneCfg<64>::LDS > L32 ? PlaneCfg<64>::LDS : L32];
  __shared__ float2 tw_s[64];
  const int g = (int)blockIdx.x;
  if (g < a.groups)
    pair_plane_part<64, INV>(a, g, lds, tw_s);
  else if (g - a.groups < b.groups)
    pair_plane_part<32, INV>(b, g - a.groups, lds, tw_s);
}

template <int N>
__device__ __forceinline__ void pair_z_part(const PairPart& p, int tile, float2* lds, float2* tw_s) {
  using K = ColCfg<N>;
  static_assert(K::THREADS == cfgeo::pair_z_threads, "one z tile per work-group");
  const int x = threadIdx.x;
  const ColPass<N, 2, 2> k{p.in, p.out, p.H, tw_s, lds, p.hstride, x % K::C, (x / K::C) % K::T, x / (K::C * K::T)};
  typename ColPass<N, 2, 2>::Regs r;
  k.load(tile, r);
  stage_twiddles<N, K::THREADS>(tw_s, p.tw);
  k.process(tile, r);
}

__device__ __forceinline__ void pair_z_kernel(const PairPart& a, const PairPart& b) {
  __shared__ float2 lds[ColCfg<64>::LDS > ColCfg<32>::LDS ? ColCfg<64>::LDS : ColCfg<32>::LDS];
  __shared__ float2 tw_s[64];
  const int g = (int)blockIdx.x;
  if (g < a.groups)
    pair_z_part<64>(a, g, lds, tw_s);
  else if (g - a.groups < b.groups)
    pair_z_part<32>(b, g - a.groups, lds, tw_s);
}

}  // namespace cfk
