// ek_mhd_launch.h -- instantiation and launch of the 2D MHD kernels for one real type.
// Included by exactly one translation unit per precision (ek_mhd_fp64.hip, ek_mhd_fp32.hip).
#pragma once

#include "ek_mhd.h"

namespace ek {
namespace mhd {

// Tiles of the 2D MHD step. A launch lasts as long as the CU with the most blocks: about
// A + B * ceil(blocks / 256) us, A and B measured on grids of 48^2 to 1024^2 (Orszag-Tang, HLLD)
// for each tile; the launch takes the tile with the smallest. us per step, FP64 14x6 / 14x10 /
// 27x11: 140^2 11.7 / 13.5 / 18.2, 200^2 16.0 / 18.1 / 18.2, 300^2 35 / 23.1 / 28.2, 700^2 155 /
// 83.4 / 84.8, 1024^2 328 / 179 / 169 (14x14 in 81 KB: 16.6, 16.7, 22.5, 93.4, 197; 30x10 174,
// 20x15 179 at 1024^2). FP32 14x6 / 14x10 / 30x14: 140^2 8.7 / 10.3 / 14.8, 240^2 11.5 / 11.9 /
// 14.8, 300^2 14.9 / 14.1 / 15.0, 420^2 24.4 / 18.2 / 19.8, 700^2 56 / 38.6 / 37.8, 1024^2 115 /
// 80.9 / 80.3 (27x11 86, 32x13 78 to 80).
template <class T>
struct M2Small {
  static constexpr bool F64 = sizeof(T) == 8;
  static constexpr int X = 14, Y = 6, NT = 320, WPE = F64 ? 4 : 8;
  static constexpr double A = F64 ? 5.7 : 6.5, B = F64 ? 5.6 : 1.9;
};
template <class T>
struct M2Mid {
  static constexpr bool F64 = sizeof(T) == 8;
  static constexpr int X = 14, Y = 10, NT = 256, WPE = F64 ? 4 : 8;
  static constexpr double A = F64 ? 7.9 : 8.0, B = F64 ? 5.4 : 2.2;
};
template <class T>
struct M2Large {
  static constexpr bool F64 = sizeof(T) == 8;
  static constexpr int X = F64 ? 27 : 30, Y = F64 ? 11 : 14, NT = 512, WPE = F64 ? 4 : 6;
  static constexpr double A = F64 ? 7.0 : 8.7, B = F64 ? 11.3 : 5.8;
};

template <class T>
using MStepFn = void (*)(const T*, T*, Geom<T>, Gas<T>, StepCtl);

template <class T, class M, int RS>
inline MStepFn<T> pick(int st)
{
  if (st == 1)
    return mhd2d_step<T, M::X, M::Y, M::NT, RS, 1, M::WPE>;
  return mhd2d_step<T, M::X, M::Y, M::NT, RS, 2, M::WPE>;
}

template <class M, class T>
inline long long blocks_of(const Geom<T>& geo)
{
  return (long long)((geo.nx + M::X - 1) / M::X) * ((geo.ny + M::Y - 1) / M::Y);
}

template <class M, class T>
inline double estimate(const Geom<T>& geo)
{
  return M::A + M::B * (double)((blocks_of<M>(geo) + 255) / 256);
}

template <class T, class M>
inline void launch_tiles(int rs, int st, const T* Uin, T* Uout, const Geom<T>& geo, const Gas<T>& gas,
                         const StepCtl& ctl, hipStream_t s)
{
  MStepFn<T> f;
  switch (rs) {
    case RS_HLL: f = pick<T, M, RS_HLL>(st); break;
    case RS_LLF: f = pick<T, M, RS_LLF>(st); break;
    default: f = pick<T, M, RS_HLLD>(st); break;
  }
  StepCtl part = ctl;
  in_launches(blocks_of<M>(geo), M::NT, [&](unsigned first, unsigned count) {
    part.tile0 = first;
    hipLaunchKernelGGL(f, dim3(count), dim3(M::NT), 0, s, Uin, Uout, geo, gas, part);
  });
}

template <class T>
inline hipError_t launch_step(int rs, int st, const T* Uin, T* Uout, const Geom<T>& geo, const Gas<T>& gas,
                              const StepCtl& ctl, hipStream_t s)
{
  const double small = estimate<M2Small<T>>(geo), mid = estimate<M2Mid<T>>(geo);
  if (estimate<M2Large<T>>(geo) < (small < mid ? small : mid))
    launch_tiles<T, M2Large<T>>(rs, st, Uin, Uout, geo, gas, ctl, s);
  else if (small < mid)
    launch_tiles<T, M2Small<T>>(rs, st, Uin, Uout, geo, gas, ctl, s);
  else
    launch_tiles<T, M2Mid<T>>(rs, st, Uin, Uout, geo, gas, ctl, s);
  return hipGetLastError();
}

template <class T>
inline hipError_t launch_inv_dt(const T* U, const Geom<T>& geo, const Gas<T>& gas, unsigned long long* dst,
                                unsigned long long* spread, int nspread,
                  hipStream_t s)
{
  long long nb = (geo.vstride + 255) / 256;
  if (nb > 4096)
    nb = 4096;
  hipLaunchKernelGGL((mhd2d_inv_dt_kernel<T, 256>), dim3((unsigned)nb), dim3(256), 0, s, U, geo, gas, dst, spread, nspread);
  return hipGetLastError();
}

} // namespace mhd
} // namespace ek
