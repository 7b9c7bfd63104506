// ek_pool_kernels.h -- batched steps of many independent grids (a job pool) in one launch.
//
// Every job keeps its own state in a shared device arena (two ping-pong buffers, the job at
// the same element offset in both), its own geometry, gas constants and time slots. One
// launch advances every active job by one step of its own dt: block b runs item b of a work
// list of (job, tile) items with the same per-tile code as the single-grid kernels
// (hydro2d_tile / hydro3d_column), so a job's results are those of its single-grid run.
// Each job's first tile keeps that job's time bookkeeping; every tile reduces its CFL term
// into one of the job's CFL words (PoolJob::spread).
//
// A tile is short and starts with a chain of dependent reads (item, job record, time slot, CFL
// words, cells), so what counts is how many tiles are in flight and how long their closing
// atomics queue: on one word per job they serialize (about 70 ns each). us per step in a persistent
// grid walking ranges of the list with one word per job -> with one block per item, the items in
// XCD order and 32 words per job: 24 blasts of edges 64-320 60 -> 29 FP32, 72 -> 46 FP64; 128 of
// edges 64-512 FP32 372 -> 289; 64 of them FP64 402 -> 245; 3D jobs (six of edges 64-128) 278 -> 201
// and 606 -> 484. Figures for other numbers of words beside pool_word.
#pragma once

#include "ek_hydro.h"
#include "ek_hydro3d.h"

namespace ek {

// CFL words per slot of a job
constexpr int POOL_NSPREAD = 32;
constexpr long long POOL_SPREAD_ELEMS = 3LL * POOL_NSPREAD * SPREAD_STRIDE;

template <class T>
struct PoolJob {
  long long off;   // element offset of the job's state in each arena buffer
  int slot0;       // index of the job's first TimeSlot (3 per job)
  int nStepmax;
  int cz;          // z planes per column chunk (3D)
  unsigned long long* spread; // the job's extra CFL words (POOL_SPREAD_ELEMS), or null
  int ntx, nty;    // tiles per axis
  double cfl, tEnd;
  Geom<T> geo;
  Gas<T> gas;
};

struct PoolWork {
  int job;
  int tx, ty;
  int tz_first; // z chunk * 2 + (1 if this item does the job's bookkeeping)
};

// Position in the work list of the item that block b of n runs, and which of its job's CFL words
// takes its term: words in turn both along an XCD's blocks (8 apart in b, one item of the list
// after another, and so one job's for many blocks) and across the XCDs (where a job that fills the
// launch runs on all of them at once). us per step, 1 / 4 / 8 / 16 / 32 / 64 words, FP32: 128 jobs of
// edges 64-512 546, 310, 292, 290, 289, 288; 24 of edges 64-320 48, 30, 29, 28, 29, 28; one of 1024^2
// 150, 74, 56, 42, 33, 30; one of 512^2 (16 words and more) 10.7, 10.8, 10.8; in FP64 64's longer
// reads show (six 3D jobs 484, 484, 484, 484, 484, 486). By block number alone the items of a job
// that run side by side on one XCD meet on two of 16 words: 128 jobs 326 to 378, one of 1024^2 35 to
// 41, one of 512^2 10.3.
__host__ __device__ __forceinline__ unsigned pool_item(unsigned b, unsigned n) { return xcd_order(b, n); }
__host__ __device__ __forceinline__ unsigned pool_word(unsigned b)
{
  return (b / 8 + b % 8 * (POOL_NSPREAD / 8)) & (unsigned)(POOL_NSPREAD - 1);
}

template <class T, int TX, int TY, int NT, int RS, int ST, bool CMP>
__global__ __launch_bounds__(NT) void hydro2d_pool_step(const T* __restrict__ Ua, T* __restrict__ Ub,
                                                        const PoolJob<T>* __restrict__ jobs,
                                                        const PoolWork* __restrict__ work,
                                                        TimeSlot* ts, int slot)
{
  __shared__ double sred[NT / 64];
  const PoolWork it = work[pool_item(blockIdx.x, gridDim.x)];
  const PoolJob<T> J = jobs[it.job];
  StepCtl ctl;
  ctl.ts = ts + J.slot0;
  ctl.spread = J.spread;
  ctl.nspread = POOL_NSPREAD;
  ctl.slot = slot;
  ctl.mode = 0;
  ctl.dt_given = 0.0;
  ctl.cfl = J.cfl;
  ctl.tEnd = J.tEnd;
  ctl.nStepmax = J.nStepmax;
  const bool first = (it.tz_first & 1) != 0;
  Loaded2<T, TX, TY, NT> in;
  hydro2d_load<T, TX, TY, NT>(Ua + J.off, J.geo, it.tx * TX, it.ty * TY, in);
  double dt;
  TimeSlot cur;
  if (!step_begin(ctl, first, dt, cur))
    return;
  const double local =
      hydro2d_tile<T, TX, TY, NT, RS, ST, CMP>(Ua + J.off, Ub + J.off, J.geo, J.gas, dt, it.tx * TX, it.ty * TY, in);
  block_max_to<NT>(invdt_word(ctl, (slot + 1) % 3, pool_word(blockIdx.x)), local, sred);
  if (first && threadIdx.x < 64)
    step_end_bookkeeping(ctl, cur, dt);
}

// Occupancy targets: FP64 3 waves per SIMD (what the shared memory allows anyway); FP32 5,
// which its shared memory also allows (93 registers, no spills).
template <class T, int TX, int TY, int NT, int RS, int ST>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 3 : 5))) void hydro3d_pool_step(const T* __restrict__ Ua, T* __restrict__ Ub,
                                                        const PoolJob<T>* __restrict__ jobs,
                                                        const PoolWork* __restrict__ work,
                                                        TimeSlot* ts, int slot)
{
  __shared__ double sred[NT / 64];
  const PoolWork it = work[pool_item(blockIdx.x, gridDim.x)];
  const PoolJob<T> J = jobs[it.job];
  StepCtl ctl;
  ctl.ts = ts + J.slot0;
  ctl.spread = J.spread;
  ctl.nspread = POOL_NSPREAD;
  ctl.slot = slot;
  ctl.mode = 0;
  ctl.dt_given = 0.0;
  ctl.cfl = J.cfl;
  ctl.tEnd = J.tEnd;
  ctl.nStepmax = J.nStepmax;
  const bool first = (it.tz_first & 1) != 0;
  double dt, local;
  TimeSlot cur;
  auto begin = [&](double& d) {
    const bool go = step_begin(ctl, first, dt, cur);
    d = dt;
    return go;
  };
  if (!hydro3d_column<T, TX, TY, NT, RS, ST, false>(Ua + J.off, Ub + J.off, J.geo, J.gas, begin, it.tx * TX,
                                                    it.ty * TY, (it.tz_first >> 1) * J.cz, J.cz, local))
    return;
  block_max_to<NT>(invdt_word(ctl, (slot + 1) % 3, pool_word(blockIdx.x)), local, sred);
  if (first && threadIdx.x < 64)
    step_end_bookkeeping(ctl, cur, dt);
}

} // namespace ek
