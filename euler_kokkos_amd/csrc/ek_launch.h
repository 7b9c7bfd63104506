// ek_launch.h -- kernel instantiation and launch for one real type. Included by exactly one
// translation unit per precision: ek_fp64.hip (built with -ffp-contract=off, the bit-exact
// path) and ek_fp32.hip (FP32 bulk path, contraction allowed).
#pragma once

#include "ek_hydro.h"
#include "ek_hydro3d.h"

namespace ek {

// 3D tiles: T3X x T3Y columns marching over z-chunks (ek_hydro3d.h; N3T threads: one per
// primitive column of the tile and its 2-cell halo).
//
// 2D tiles (Tile2Of, ek_hydro.h). A grid that leaves CUs idle takes small ones with so many
// threads that every phase is one pass; a step of it then lasts as long as its fullest CU, so
// the line lies where the small tiles put no more blocks on one CU than the large ones do
// (FP64, us per step, small / large tiles: 128^2 6.9 / 7.3, 200^2 8.2 / 7.4, 256^2 8.3 / 8.8,
// 280^2 9.5 / 8.8, 512^2 19.6 / 16.0). In FP32 a second block on a CU costs the small tiles little
// (64^2 5.9 / 7.8, 200^2 6.4 / 7.8, 256^2 6.5 / 7.9, 320^2 8.1 / 7.9, 512^2 12.7 / 9.8).
template <class T>
inline bool small_tile2(int nx, int ny)
{
  constexpr long long CUS = 256;
  using S = SmallTile2;
  using L = Tile2Of<T>;
  const long long ns = (long long)((nx + S::X - 1) / S::X) * ((ny + S::Y - 1) / S::Y);
  const long long nl = (long long)((nx + L::X - 1) / L::X) * ((ny + L::Y - 1) / L::Y);
  return ns <= CUS || (ns <= 2 * CUS && (sizeof(T) == 4 || nl > CUS));
}

template <class T>
using Step2Fn = void (*)(const T*, T*, Geom<T>, Gas<T>, StepCtl);
template <class T>
using Step3Fn = void (*)(const T*, T*, Geom<T>, Gas<T>, StepCtl, int, int, int, int);

template <class T, class C, int RS>
inline Step2Fn<T> pick2(int st)
{
  if (st == 0)
    return hydro2d_step<T, C::X, C::Y, C::NT, RS, 0, C::CMP>;
  if (st == 1)
    return hydro2d_step<T, C::X, C::Y, C::NT, RS, 1, C::CMP>;
  return hydro2d_step<T, C::X, C::Y, C::NT, RS, 2, C::CMP>;
}
template <class T, class C>
inline void launch2(int rs, int st, const T* Uin, T* Uout, const Geom<T>& geo, const Gas<T>& gas, const StepCtl& ctl,
                    hipStream_t s)
{
  Step2Fn<T> f;
  switch (rs) {
    case RS_APPROX: f = pick2<T, C, RS_APPROX>(st); break;
    case RS_LLF: f = pick2<T, C, RS_LLF>(st); break;
    case RS_HLL: f = pick2<T, C, RS_HLL>(st); break;
    default: f = pick2<T, C, RS_HLLC>(st); break;
  }
  const long long blocks = (long long)((geo.nx + C::X - 1) / C::X) * ((geo.ny + C::Y - 1) / C::Y);
  StepCtl part = ctl;
  in_launches(blocks, C::NT, [&](unsigned first, unsigned count) {
    part.tile0 = first;
    hipLaunchKernelGGL(f, dim3(count), dim3(C::NT), 0, s, Uin, Uout, geo, gas, part);
  });
}
template <class T, int TX, int TY, int RS>
inline Step3Fn<T> pick3(int st)
{
  if (st == 0)
    return hydro3d_step<T, TX, TY, N3T, RS, 0>;
  if (st == 1)
    return hydro3d_step<T, TX, TY, N3T, RS, 1>;
  return hydro3d_step<T, TX, TY, N3T, RS, 2>;
}
template <class T, int TX, int TY>
inline void launch3(int rs, int st, const T* Uin, T* Uout, const Geom<T>& geo, const Gas<T>& gas, const StepCtl& ctl,
                    int cz, hipStream_t s)
{
  Step3Fn<T> f;
  switch (rs) {
    case RS_APPROX: f = pick3<T, TX, TY, RS_APPROX>(st); break;
    case RS_LLF: f = pick3<T, TX, TY, RS_LLF>(st); break;
    default: f = pick3<T, TX, TY, RS_HLLC>(st); break;
  }
  const int ntx = (geo.nx + TX - 1) / TX, nty = (geo.ny + TY - 1) / TY, nch = (geo.nz + cz - 1) / cz;
  hipLaunchKernelGGL(f, dim3(ntx * nty * nch), dim3(N3T), 0, s, Uin, Uout, geo, gas, ctl, cz, ntx, nty, nch);
}

template <class T>
inline hipError_t launch_step(int dim, int rs, int st, const T* Uin, T* Uout, const Geom<T>& geo,
                              const Gas<T>& gas, const StepCtl& ctl, int cz, hipStream_t s)
{
  if (dim == 2) {
    if (small_tile2<T>(geo.nx, geo.ny))
      launch2<T, SmallTile2>(rs, st, Uin, Uout, geo, gas, ctl, s);
    else
      launch2<T, Tile2Of<T>>(rs, st, Uin, Uout, geo, gas, ctl, s);
  } else if (cz < 0) { // hydro3d_z_chunk's sign
    launch3<T, T3Y, T3X>(rs, st, Uin, Uout, geo, gas, ctl, -cz, s);
  } else {
    launch3<T, T3X, T3Y>(rs, st, Uin, Uout, geo, gas, ctl, cz, s);
  }
  return hipGetLastError();
}

template <class T>
inline hipError_t launch_inv_dt(int dim, const T* U, const Geom<T>& geo, const Gas<T>& gas,
                                unsigned long long* dst, unsigned long long* spread, int nspread,
                  hipStream_t s)
{
  const long long n = geo.vstride;
  long long nb = (n + 255) / 256;
  if (nb > 4096)
    nb = 4096;
  if (dim == 2)
    hipLaunchKernelGGL((inv_dt_kernel<T, 2, 256>), dim3((unsigned)nb), dim3(256), 0, s, U, geo, gas, dst, spread, nspread, n);
  else
    hipLaunchKernelGGL((inv_dt_kernel<T, 3, 256>), dim3((unsigned)nb), dim3(256), 0, s, U, geo, gas, dst, spread, nspread, n);
  return hipGetLastError();
}

template <class T>
inline hipError_t launch_budget(int nv, const T* U, long long ncell, long long vstride, double* partial,
                                int nblocks, hipStream_t s)
{
  if (nv == 4)
    hipLaunchKernelGGL((budget_kernel<T, 4, 256>), dim3(nblocks), dim3(256), 0, s, U, ncell, vstride, partial);
  else if (nv == 5)
    hipLaunchKernelGGL((budget_kernel<T, 5, 256>), dim3(nblocks), dim3(256), 0, s, U, ncell, vstride, partial);
  else
    hipLaunchKernelGGL((budget_kernel<T, 8, 256>), dim3(nblocks), dim3(256), 0, s, U, ncell, vstride, partial);
  return hipGetLastError();
}

template <class T>
inline hipError_t launch_ref_to_soa(int dim, const double* R, T* U, const Geom<T>& geo, int gw, int nbvar,
                                    int isize, int jsize, int ksize, hipStream_t s)
{
  long long nb = (geo.vstride + 255) / 256;
  if (nb > 65535)
    nb = 65535;
  if (dim == 2)
    hipLaunchKernelGGL((ref_to_soa<T, 2>), dim3((unsigned)nb), dim3(256), 0, s, R, U, geo, gw, nbvar, isize, jsize, ksize);
  else
    hipLaunchKernelGGL((ref_to_soa<T, 3>), dim3((unsigned)nb), dim3(256), 0, s, R, U, geo, gw, nbvar, isize, jsize, ksize);
  return hipGetLastError();
}

template <class T>
inline hipError_t launch_soa_to_ref(int dim, const T* U, double* R, const Geom<T>& geo, int gw, int nbvar,
                                    int isize, int jsize, int ksize, int mhd, hipStream_t s)
{
  const long long n = (long long)isize * jsize * (dim == 3 ? ksize : 1);
  long long nb = (n + 255) / 256;
  if (nb > 65535)
    nb = 65535;
  if (dim == 2)
    hipLaunchKernelGGL((soa_to_ref<T, 2>), dim3((unsigned)nb), dim3(256), 0, s, U, R, geo, gw, nbvar, isize, jsize, ksize, mhd);
  else
    hipLaunchKernelGGL((soa_to_ref<T, 3>), dim3((unsigned)nb), dim3(256), 0, s, U, R, geo, gw, nbvar, isize, jsize, ksize, mhd);
  return hipGetLastError();
}

} // namespace ek
