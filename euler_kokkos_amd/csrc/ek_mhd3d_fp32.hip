// ek_mhd3d_fp32.hip -- 3D MHD step pipeline, float instantiation.
#include "ek_internal.h"
#include "ek_mhd3d.h"
#include "ek_pool_mhd3d.h"

namespace ek {
namespace fp32 {

template <int RS, int ST>
static hipError_t launch3(const float* Uin, float* Uout, float* S, const mhd3::Work3& w, const Geom<float>& geo,
                          const Gas<float>& gas, const StepCtl& ctl, hipStream_t s)
{
  const unsigned nb = (unsigned)((w.PN + 255) / 256);
  const long long nu = (geo.vstride + 255) / 256;
  const unsigned ni = (unsigned)(nu < mhd3::MHD3_UPDATE_BLOCKS ? nu : mhd3::MHD3_UPDATE_BLOCKS);
  hipLaunchKernelGGL(mhd3::padprims_kernel<float>, dim3(nb), dim3(256), 0, s, Uin, S, w, geo, gas, ctl);
  hipLaunchKernelGGL(mhd3::efield_kernel<float>, dim3(nb), dim3(256), 0, s, S, w, ctl);
  const mhd3::FluxGrid fg = mhd3::flux_grid(geo);
  hipLaunchKernelGGL((mhd3::fluxemf_kernel<float, RS, ST>), dim3(fg.ntx * fg.nty * fg.ntz), dim3(mhd3::FCN), 0, s, S, w, geo,
                     gas, ctl, fg.cz, fg.ntx, fg.nty);
  hipLaunchKernelGGL(mhd3::update_kernel<float>, dim3(ni), dim3(256), 0, s, Uin, S, Uout, w, geo, gas, ctl);
  return hipGetLastError();
}

hipError_t mhd3_step(int rs, int st, const float* Uin, float* Uout, float* scratch, const Geom<float>& geo,
                     const Gas<float>& gas, const StepCtl& ctl, hipStream_t s)
{
  mhd3::Work3 w;
  w.nx = geo.nx;
  w.ny = geo.ny;
  w.nz = geo.nz;
  w.PX = geo.nx + 6;
  w.PY = geo.ny + 6;
  w.PZ = geo.nz + 6;
  w.PN = (long long)w.PX * w.PY * w.PZ;
  const bool st1 = st == 1;
  switch (rs) {
    case RS_HLL: return st1 ? launch3<RS_HLL, 1>(Uin, Uout, scratch, w, geo, gas, ctl, s)
                            : launch3<RS_HLL, 2>(Uin, Uout, scratch, w, geo, gas, ctl, s);
    case RS_LLF: return st1 ? launch3<RS_LLF, 1>(Uin, Uout, scratch, w, geo, gas, ctl, s)
                            : launch3<RS_LLF, 2>(Uin, Uout, scratch, w, geo, gas, ctl, s);
    default: return st1 ? launch3<RS_HLLD, 1>(Uin, Uout, scratch, w, geo, gas, ctl, s)
                        : launch3<RS_HLLD, 2>(Uin, Uout, scratch, w, geo, gas, ctl, s);
  }
}

hipError_t mhd3_inv_dt(const float* U, const Geom<float>& geo, const Gas<float>& gas, unsigned long long* dst,
                       unsigned long long* spread, int nspread,
                  hipStream_t s)
{
  long long nb = (geo.vstride + 255) / 256;
  if (nb > 4096)
    nb = 4096;
  hipLaunchKernelGGL(mhd3::inv_dt3_kernel<float>, dim3((unsigned)nb), dim3(256), 0, s, U, geo, gas, dst, spread, nspread);
  return hipGetLastError();
}

long long mhd3_scratch_elems(int nx, int ny, int nz)
{
  return (long long)mhd3::A_TOTAL * (nx + 6) * (ny + 6) * (long long)(nz + 6);
}

hipError_t pool_mhd3_step(int rs, int st, const float* Ua, float* Ub, float* W, const PoolJobM<float>* jobs,
                          const PoolWork* wp, int np, const PoolWork* wf, int nf, const PoolWork* wu, int nu,
                          TimeSlot* ts, int slot, int ugrid, hipStream_t s)
{
  return pool::mhd3_step<float>(rs, st, Ua, Ub, W, jobs, wp, np, wf, nf, wu, nu, ts, slot, ugrid, s);
}

int pool_mhd3_update_grid(int cus)
{
  return pool::mhd3_update_grid<float>(cus);
}

} // namespace fp32
} // namespace ek
