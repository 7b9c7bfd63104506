// ek_pool_mhd3d.h -- 3D MHD jobs of the job pool: one pool step runs the four kernels of
// the 3D MHD pipeline (ek_mhd3d.h) once each over every active job.
//
// Every job keeps its state in the pool's arena (same offset in both ping-pong buffers) and
// its own padded work area in the pool's work buffer. Three work lists describe the active
// jobs: (job, 4096-cell chunk of the padded grid) items for the two padded-grid kernels, which
// run one block per 256 cells of them; (job, column tile, z-chunk) items for the flux/EMF
// kernel, one block each; and (job, 4096-cell chunk of the interior) items for the update, a
// persistent grid whose blocks walk contiguous ranges of them; a job's first interior chunk
// keeps the job's time bookkeeping. Each job reads its own dt from its own time slots. The
// per-cell code is the single-grid pipeline's (padprims_cell ... update_cell), so a job's
// result is its single-grid ek_run result.
#pragma once

#include "ek_mhd3d.h"
#include "ek_pool_kernels.h"

namespace ek {

template <class T>
struct PoolJobM {
  long long off;   // element offset of the job's state in each arena buffer
  long long woff;  // element offset of the job's work area in the work buffer
  int slot0;       // index of the job's first TimeSlot (3 per job)
  int nStepmax;
  int cz;          // z planes per flux/EMF item
  double cfl, tEnd;
  mhd3::Work3 w;
  Geom<T> geo;
  Gas<T> gas;
};

// cells per work item: padded-grid kernels, update. A block of the update walks its range in
// units of 256 cells (one per thread), reading the item and its job record again for every
// unit: kept across units, the record's fields and the array bases derived from them would take
// the scalar registers that the scalar-base addressing of the per-cell code needs.
constexpr int MP_CHUNK = 4096;
constexpr int MU_CHUNK = 4096;
constexpr int UNITS_P = MP_CHUNK / 256, UNITS_U = MU_CHUNK / 256;

template <class T>
__device__ __forceinline__ StepCtl pool_ctl(const PoolJobM<T>& J, TimeSlot* ts, int slot)
{
  StepCtl ctl;
  ctl.ts = ts + J.slot0;
  ctl.spread = nullptr;
  ctl.nspread = 1;
  ctl.slot = slot;
  ctl.mode = 0;
  ctl.dt_given = 0.0;
  ctl.cfl = J.cfl;
  ctl.tEnd = J.tEnd;
  ctl.nStepmax = J.nStepmax;
  return ctl;
}

// One unit (256 padded cells) per block: the block reads its item, the item's job record and
// the job's dt, then `body` runs for this thread's padded cell c. One unit per block lets the
// hardware overlap those dependent reads across the many resident blocks; persistent blocks
// walking ranges of units serialized them with every unit's cell loads (0.78 against 0.60 ms per
// 128^3 FP32 job).
template <class T, class Body>
__device__ __forceinline__ void pool_padded_unit(const PoolJobM<T>* __restrict__ jobs,
                                                 const PoolWork* __restrict__ work, TimeSlot* ts, int slot,
                                                 Body body)
{
  const int u = blockIdx.x;
  const int q = u / UNITS_P, r = u - q * UNITS_P;
  const PoolWork it = work[q];
  const PoolJobM<T> J = jobs[it.job];
  double dt;
  if (!mhd3::step_dt(pool_ctl(J, ts, slot), dt))
    return;
  const unsigned c = ((unsigned)it.tx * (unsigned)UNITS_P + (unsigned)r) * 256u + threadIdx.x;
  if ((long long)c < J.w.PN)
    body(J, c);
}

template <class T>
__global__ __launch_bounds__(256) void mhd3_pool_padprims(const T* __restrict__ Ua, T* __restrict__ W,
                                                          const PoolJobM<T>* __restrict__ jobs,
                                                          const PoolWork* __restrict__ work, TimeSlot* ts, int slot)
{
  pool_padded_unit<T>(jobs, work, ts, slot, [&](const PoolJobM<T>& J, unsigned c) {
    int i, j, k;
    mhd3::split3(c, (unsigned)J.w.PX, (unsigned)J.w.PY, i, j, k);
    mhd3::padprims_cell<T>(Ua + J.off, W + J.woff, J.w, J.geo, J.gas, i, j, k);
  });
}

template <class T>
__global__ __launch_bounds__(256) void mhd3_pool_efield(T* __restrict__ W, const PoolJobM<T>* __restrict__ jobs,
                                                        const PoolWork* __restrict__ work, TimeSlot* ts, int slot)
{
  pool_padded_unit<T>(jobs, work, ts, slot, [&](const PoolJobM<T>& J, unsigned c) {
    int i, j, k;
    mhd3::split3(c, (unsigned)J.w.PX, (unsigned)J.w.PY, i, j, k);
    mhd3::efield_cell<T>(W + J.woff, J.w, i, j, k);
  });
}

// Trace, fluxes and EMFs: one block per (job, tile, z-chunk) item.
template <class T, int RS, int ST>
__global__ __launch_bounds__(mhd3::FCN) __attribute__((amdgpu_waves_per_eu(mhd3::FCW<T>))) void mhd3_pool_fluxemf(T* __restrict__ W, const PoolJobM<T>* __restrict__ jobs,
                                                               const PoolWork* __restrict__ work, TimeSlot* ts,
                                                               int slot)
{
  const PoolWork it = work[xcd_order(blockIdx.x, gridDim.x)];
  const PoolJobM<T> J = jobs[it.job];
  double dt;
  if (!mhd3::step_dt(pool_ctl(J, ts, slot), dt))
    return;
  mhd3::fluxemf_columns<T, RS, ST>(W + J.woff, J.w, J.geo, J.gas, dt, 3 + it.tx * mhd3::FCX, 3 + it.ty * mhd3::FCY,
                                   3 + it.tz_first * J.cz, min(3 + (it.tz_first + 1) * J.cz, 3 + mhd3::nfaces(J.geo, 2)));
}

// Items of block b: a contiguous range of the work list, so neighbouring tiles of a job run
// one after the other on the same XCD (their halo lines meet in that XCD's L2).
__device__ __forceinline__ void pool_range(int nwork, int& w0, int& w1)
{
  const int per = nwork / (int)gridDim.x, rem = nwork % (int)gridDim.x;
  const int b = blockIdx.x;
  w0 = b * per + (b < rem ? b : rem);
  w1 = w0 + per + (b < rem ? 1 : 0);
}

// Update. A block's range holds consecutive units of few jobs: the block keeps a running CFL
// maximum and adds it to a job's next slot once, when its units of that job end. The job's
// first unit keeps the job's time bookkeeping. (Contiguous ranges measured faster than
// grid-strided units here: 0.78 against 0.88 ms per 128^3 FP32 job in a pool of 8.)
template <class T>
__global__ __launch_bounds__(256) void mhd3_pool_update(const T* __restrict__ Ua, const T* __restrict__ W, T* __restrict__ Ub,
                                                        const PoolJobM<T>* __restrict__ jobs,
                                                        const PoolWork* __restrict__ work, int nwork, TimeSlot* ts,
                                                        int slot)
{
  __shared__ double sred[4];
  int u0, u1;
  pool_range(UNITS_U * nwork, u0, u1);
  double local = 0.0;
  int pending = -1;  // TimeSlot word index of the job whose maximum `local` holds
  int pjob = -1;
  for (int u = u0; u < u1; u++) {
    const int q = u / UNITS_U, r = u - q * UNITS_U;
    const PoolWork it = work[q];
    if (pending >= 0 && it.job != pjob) {
      block_max_to<256>(&ts[pending].invdt_bits, local, sred);
      local = 0.0;
      pending = -1;
    }
    const PoolJobM<T> J = jobs[it.job];
    const StepCtl ctl = pool_ctl(J, ts, slot);
    const bool first = (it.tz_first & 1) != 0 && r == 0;
    double dt;
    TimeSlot cur;
    if (!step_begin(ctl, first, dt, cur))
      continue;
    pending = J.slot0 + (slot + 1) % 3;
    pjob = it.job;
    const T dtdx = T(dt / J.geo.dx), dtdy = T(dt / J.geo.dy), dtdz = T(dt / J.geo.dz);
    const long long c = ((long long)it.tx * UNITS_U + r) * 256 + threadIdx.x;
    if (c < J.geo.vstride) {
      const double sv = mhd3::update_cell<T>(Ua + J.off, W + J.woff, Ub + J.off, J.w, J.geo, J.gas, dtdx, dtdy, dtdz, c);
      local = (sv > local || !(sv == sv)) ? sv : local;
    }
    if (first && threadIdx.x < 64)
      step_end_bookkeeping(ctl, cur, dt);
  }
  if (pending >= 0)
    block_max_to<256>(&ts[pending].invdt_bits, local, sred);
}

namespace pool {

// persistent grid of the update kernel: CUs x blocks that fit on one CU at once
template <class T>
inline int mhd3_update_grid(int cus)
{
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(mhd3_pool_update<T>), 256, 0) !=
          hipSuccess ||
      n < 1)
    n = 1;
  return cus * n;
}

template <class T, int RS, int ST>
inline hipError_t mhd3_launch(const T* Ua, T* Ub, T* W, const PoolJobM<T>* jobs, const PoolWork* wp, int np,
                              const PoolWork* wf, int nf, const PoolWork* wu, int nu, TimeSlot* ts, int slot,
                              int ugrid, hipStream_t s)
{
  if (np <= 0 || nf <= 0 || nu <= 0)
    return hipSuccess;
  hipLaunchKernelGGL(mhd3_pool_padprims<T>, dim3(UNITS_P * np), dim3(256), 0, s, Ua, W, jobs, wp, ts, slot);
  hipLaunchKernelGGL(mhd3_pool_efield<T>, dim3(UNITS_P * np), dim3(256), 0, s, W, jobs, wp, ts, slot);
  hipLaunchKernelGGL((mhd3_pool_fluxemf<T, RS, ST>), dim3(nf), dim3(mhd3::FCN), 0, s, W, jobs, wf, ts, slot);
  hipLaunchKernelGGL(mhd3_pool_update<T>, dim3((unsigned)(ugrid < UNITS_U * nu ? ugrid : UNITS_U * nu)), dim3(256), 0, s,
                     Ua, W, Ub, jobs, wu, nu, ts, slot);
  return hipGetLastError();
}

template <class T>
inline hipError_t mhd3_step(int rs, int st, const T* Ua, T* Ub, T* W, const PoolJobM<T>* jobs, const PoolWork* wp,
                            int np, const PoolWork* wf, int nf, const PoolWork* wu, int nu, TimeSlot* ts, int slot,
                            int ugrid, hipStream_t s)
{
  auto go = [&](auto f) { return f(Ua, Ub, W, jobs, wp, np, wf, nf, wu, nu, ts, slot, ugrid, s); };
  const bool st1 = st == 1;
  switch (rs) {
    case RS_HLL: return st1 ? go(mhd3_launch<T, RS_HLL, 1>) : go(mhd3_launch<T, RS_HLL, 2>);
    case RS_LLF: return st1 ? go(mhd3_launch<T, RS_LLF, 1>) : go(mhd3_launch<T, RS_LLF, 2>);
    default: return st1 ? go(mhd3_launch<T, RS_HLLD, 1>) : go(mhd3_launch<T, RS_HLLD, 2>);
  }
}

} // namespace pool
} // namespace ek
