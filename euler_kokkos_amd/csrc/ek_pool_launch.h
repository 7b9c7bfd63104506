// ek_pool_launch.h -- instantiation and launch of the job-pool kernels for one real type.
// Included by exactly one translation unit per precision (ek_pool_fp64.hip, ek_pool_fp32.hip).
#pragma once

#include "ek_pool_kernels.h"

namespace ek {
namespace pool {

// 2D tiles the autotuner chooses from (Tile2Of, SmallTile2: ek_hydro.h); the first until tuned.
// us per step of 24 ragged jobs of up to 320^2, then 100 of up to 512^2 in FP64 / 256 in FP32:
// FP64 16x12 47.6, 389; 24x8 44.5, 400; 12x16 44.3, 397; small 61.0, 581. FP32 32x8 29.0, 558;
// 32x16 27.5, 559; 16x16 26.2, 555; small 38.8, 929. 8 jobs of up to 64^2: small 6.9 and 5.8, the
// others 7.3 to 7.6.
struct PoolTile2 {
  int x, y, nt;
  bool cmp;
};
constexpr int N2VARIANTS = 4;
template <class T>
constexpr PoolTile2 pool_tile2(int v)
{
  using L = Tile2Of<T>;
  using S = SmallTile2;
  switch (v) {
    case 0: return sizeof(T) == 8 ? PoolTile2{ L::X, L::Y, L::NT, L::CMP } : PoolTile2{ 32, 8, 256, false };
    case 1: return { S::X, S::Y, S::NT, S::CMP };
    case 2: return sizeof(T) == 8 ? PoolTile2{ 24, 8, 256, true } : PoolTile2{ L::X, L::Y, L::NT, L::CMP };
    default: return sizeof(T) == 8 ? PoolTile2{ 12, 16, 256, true } : PoolTile2{ 16, 16, 256, false };
  }
}
// 3D column tile (the z chunk depth is the tuned parameter)
constexpr int P3X = 16, P3Y = 8, P3T = 256;

template <class T>
using Pool2Fn = void (*)(const T*, T*, const PoolJob<T>*, const PoolWork*, TimeSlot*, int);

template <class T, int V, int ST>
inline Pool2Fn<T> pick2v()
{
  constexpr PoolTile2 t = pool_tile2<T>(V);
  return hydro2d_pool_step<T, t.x, t.y, t.nt, RS_HLLC, ST, t.cmp>;
}

template <class T>
inline Pool2Fn<T> pick2(int variant, int st)
{
  switch (variant * 2 + (st == 1 ? 0 : 1)) {
    case 0: return pick2v<T, 0, 1>();
    case 1: return pick2v<T, 0, 2>();
    case 2: return pick2v<T, 1, 1>();
    case 3: return pick2v<T, 1, 2>();
    case 4: return pick2v<T, 2, 1>();
    case 5: return pick2v<T, 2, 2>();
    case 6: return pick2v<T, 3, 1>();
    default: return pick2v<T, 3, 2>();
  }
}

template <class T>
inline Pool2Fn<T> pick3(int st)
{
  if (st == 1)
    return hydro3d_pool_step<T, P3X, P3Y, P3T, RS_HLLC, 1>;
  return hydro3d_pool_step<T, P3X, P3Y, P3T, RS_HLLC, 2>;
}

template <class T>
inline hipError_t launch_step(int dim, int variant, int st, const T* Ua, T* Ub, const PoolJob<T>* jobs,
                              const PoolWork* work, int nwork, TimeSlot* ts, int slot, hipStream_t s)
{
  if (nwork <= 0)
    return hipSuccess;
  const Pool2Fn<T> f = dim == 2 ? pick2<T>(variant, st) : pick3<T>(st);
  const int nt = dim == 2 ? pool_tile2<T>(variant).nt : P3T;
  in_launches(nwork, nt, [&](unsigned first, unsigned count) {
    hipLaunchKernelGGL(f, dim3(count), dim3(nt), 0, s, Ua, Ub, jobs, work + first, ts, slot);
  });
  return hipGetLastError();
}

} // namespace pool
} // namespace ek
