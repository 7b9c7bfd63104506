// ek_mhd3d.h -- 3D MHD MUSCL-Hancock step (HLLD fluxes, 3D constrained transport) for gfx950.
//
// One step is SolverMHDMuscl<3>::godunov_unsplit_impl, impl 0 (src/muscl/SolverMHDMuscl.cpp:
// 462-512), as a pipeline of kernels over a ghost-padded SoA work area (x fastest, 3 ghost
// layers each side, so padded index (i,j,k) is the reference's U(i,j,k)):
//   padprims: interior state -> padded face fields, ghosts through the boundary map, and the
//             primitives with the right/top/front face fields (ConvertToPrimitivesFunctor3D_MHD)
//   efield  : edge electric fields (ComputeElecFieldFunctor3D)
//   fluxemf : the half-step record of every cell (trace_unsplit_mhd_3d_simpler) in LDS: centred
//             state, face fields and half slopes, 35 values, from which each of the 6 face
//             states and 12 edge states is the centre plus one or two half slopes, and the
//             transverse face-field slopes (ComputeMagSlopesFunctor3D); from them, with the
//             reference's own additions and floors, 3 Riemann problems and 3 edge EMFs per cell
//             (ComputeFluxesAndStoreFunctor3D_MHD, ComputeEmfAndStoreFunctor3D)
//   update  : flux update, CT update and the CFL term of the new state (UpdateFunctor3D_MHD,
//             UpdateEmfFunctor3D, ComputeDtFunctor3D_MHD), with the device time bookkeeping
// Every kernel reads the step's dt from the device time slot.
#pragma once

#include "ek_mhd.h"

namespace ek {
namespace mhd3 {

using namespace ek::mhd;

// Work-area layout. All arrays have PN = PX*PY*PZ elements.
struct Work3 {
  int PX, PY, PZ;
  long long PN;
  int nx, ny, nz;
};

// offsets (in arrays of PN elements) inside the scratch block
enum {
  A_B = 0,            // padded face fields IA, IB, IC (A_B + v - IA)
  A_Q = 3,            // primitives, 8
  A_E = 11,           // Ex, Ey, Ez
  A_FLUX = 14,        // Fx, Fy, Fz: 3 x 5 (ID IP IU IV IW of the update, unrotated)
  A_EMF = 29,         // EMF x, y, z
  A_TOTAL = 32
};

// Half-step record of a cell: K_C + v the centred state (component order of the state),
// K_AL..K_CR the six face fields, then the half slopes along x, y and z, each group
// holding ID IP IU IV IW at 0..4 and the two transverse field components at 5, 6
// (x: IB IC; y: IA IC; z: IA IB).
enum { K_C = 0, K_AL = 8, K_AR, K_BL, K_BR, K_CL, K_CR, K_X = 14, K_Y = 21, K_Z = 28, K_N = 35 };

// Lower faces per row of cells along `axis` that a step computes: one more than cells, except on
// a periodic axis, where face n is face 0 (the ghosts on both sides are copies of the same
// cells, so its values are bitwise those) and whoever computes face 0 stores it as face n too.
template <class T>
__host__ __device__ inline bool wraps(const Geom<T>& geo, int axis)
{
  return geo.bc[2 * axis] == BC_PERIODIC && geo.bc[2 * axis + 1] == BC_PERIODIC;
}
template <class T>
__host__ __device__ inline int nfaces(const Geom<T>& geo, int axis)
{
  return (axis == 0 ? geo.nx : axis == 1 ? geo.ny : geo.nz) + (wraps(geo, axis) ? 0 : 1);
}

// padded linear index (below 2^30: the host keeps every array below 4 GiB)
__device__ __forceinline__ unsigned pidx(const Work3& w, int i, int j, int k)
{
  return ((unsigned)k * (unsigned)w.PY + (unsigned)j) * (unsigned)w.PX + (unsigned)i;
}

// Element at a 32-bit byte offset from a wave-uniform array base: the access addresses as a
// scalar base + one 32-bit lane offset per cell, instead of a 64-bit address per (array,
// cell), which takes two registers and 64-bit adds each. Each array of one grid is below
// 4 GiB (checked by the host). The base is the same in every lane; passing it through
// readfirstlane keeps the compiler from folding the array offset into a 64-bit per-lane
// address. Used in the trace and the update; the pad and E-field kernels keep plain indexing,
// with which the compiler spaces their loads better.
typedef char __attribute__((address_space(1))) * gbytes_t;

template <class T>
__device__ __forceinline__ gbytes_t sbase(const T* base)
{
  const unsigned long long a = reinterpret_cast<unsigned long long>(base);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return (gbytes_t)(((unsigned long long)hi << 32) | lo);
}

template <class T>
__device__ __forceinline__ T ldb(const T* base, unsigned boff)
{
  return *(const T __attribute__((address_space(1)))*)(sbase(base) + boff);
}

template <class T>
__device__ __forceinline__ void stb(T* base, unsigned boff, T x)
{
  *(T __attribute__((address_space(1)))*)(sbase(base) + boff) = x;
}

// (i, j, k) of linear index c in a box of X x Y x (any) cells. 32-bit division: the host
// keeps every work-area array below 4 GiB, so every index here is below 2^30 (a 64-bit
// division would cost each thread a long software sequence).
__device__ __forceinline__ void split3(unsigned c, unsigned X, unsigned Y, int& i, int& j, int& k)
{
  const unsigned r = c / X;
  const unsigned z = r / Y;
  i = (int)(c - r * X);
  j = (int)(r - z * Y);
  k = (int)z;
}

template <class T>
__device__ __forceinline__ bool cell_of(const Work3& w, int& i, int& j, int& k)
{
  // XCD order: the rows and planes a cell's neighbours are on were read on the same XCD (per step
  // 64^3 FP64 126.4 -> 122.9 us, FP32 64.9 -> 63.9; 97x64x110 312 -> 307 and 149 -> 146; 128^3 FP64
  // 897 -> 896, FP32 388 -> 382; the update in that order was up to 3 % slower)
  const unsigned c = xcd_order(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (c >= (unsigned long long)w.PN)
    return false;
  split3(c, (unsigned)w.PX, (unsigned)w.PY, i, j, k);
  return true;
}

// step_begin without the finished-slot forwarding (the update kernel owns it)
__device__ __forceinline__ bool step_dt(const StepCtl& c, double& dt)
{
  const TimeSlot cur = c.ts[c.slot];
  if (c.mode == 0) {
    if (cur.finished || cur.t >= (c.tEnd - 1e-14) || cur.it >= c.nStepmax)
      return false;
    dt = c.cfl / bits_to_double(invdt_gather(c, c.slot, cur.invdt_bits));
    if (cur.t + dt > c.tEnd)
      dt = c.tEnd - cur.t;
  } else {
    dt = c.dt_given;
  }
  return true;
}

// pad + prims in one pass. The padded face fields: ghost values as SolverBase::make_boundaries
// fills them (X, then Y, then Z passes; reflecting axes negate the normal momentum and the
// normal face field). On i < PX-1, j < PY-1, k < PZ-1 also the primitives
// (ConvertToPrimitivesFunctor3D_MHD), whose right / top / front face fields are the padded
// values of those neighbours, read from the interior state through the same map.
template <class T>
__device__ __forceinline__ void padprims_cell(const T* __restrict__ U, T* __restrict__ S, const Work3& w,
                                              const Geom<T>& geo, const Gas<T>& gas, int i, int j, int k)
{
  bool fx, fy, fz;
  const int si = bc_map(i - 3, w.nx, geo.bc[0], geo.bc[1], fx);
  const int sj = bc_map(j - 3, w.ny, geo.bc[2], geo.bc[3], fy);
  const int sk = bc_map(k - 3, w.nz, geo.bc[4], geo.bc[5], fz);
  const long long vs = geo.vstride;
  const long long o = ((long long)sk * w.ny + sj) * w.nx + si;
  const long long po = pidx(w, i, j, k), PN = w.PN;
  T u[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    T x = U[v * vs + o];
    if ((fx && (v == IU || v == IA)) || (fy && (v == IV || v == IB)) || (fz && (v == IW || v == IC)))
      x = x * T(-1);
    if (v >= IA)
      S[(A_B + v - IA) * PN + po] = x;
    u[v] = x;
  }
  if (i >= w.PX - 1 || j >= w.PY - 1 || k >= w.PZ - 1)
    return;
  // the padded IA of (i+1,j,k), IB of (i,j+1,k), IC of (i,j,k+1): only the reflection
  // along the field's own axis negates it
  bool gx, gy, gz;
  const int si1 = bc_map(i - 2, w.nx, geo.bc[0], geo.bc[1], gx);
  const int sj1 = bc_map(j - 2, w.ny, geo.bc[2], geo.bc[3], gy);
  const int sk1 = bc_map(k - 2, w.nz, geo.bc[4], geo.bc[5], gz);
  T mx = U[IA * vs + ((long long)sk * w.ny + sj) * w.nx + si1];
  T my = U[IB * vs + ((long long)sk * w.ny + sj1) * w.nx + si];
  T mz = U[IC * vs + ((long long)sk1 * w.ny + sj) * w.nx + si];
  if (gx)
    mx = mx * T(-1);
  if (gy)
    my = my * T(-1);
  if (gz)
    mz = mz * T(-1);
  T q[NV];
  constoprim<T>(gas, u, mx, my, mz, q);
#pragma unroll
  for (int v = 0; v < NV; v++)
    S[(A_Q + v) * PN + po] = q[v];
}

template <class T>
__global__ __launch_bounds__(256) void padprims_kernel(const T* __restrict__ U, T* __restrict__ S, Work3 w,
                                                       Geom<T> geo, Gas<T> gas, StepCtl ctl)
{
  double dt;
  if (!step_dt(ctl, dt))
    return;
  int i, j, k;
  if (!cell_of<T>(w, i, j, k))
    return;
  padprims_cell<T>(U, S, w, geo, gas, i, j, k);
}

// edge electric fields on 1 <= i,j,k < size-1
template <class T>
__device__ __forceinline__ void efield_cell(T* __restrict__ S, const Work3& w, int i, int j, int k)
{
  if (i < 1 || j < 1 || k < 1 || i >= w.PX - 1 || j >= w.PY - 1 || k >= w.PZ - 1)
    return;
  const long long PN = w.PN, o = pidx(w, i, j, k);
  const long long sx = 1, sy = w.PX, sz = (long long)w.PX * w.PY;
  const T* Q = S + A_Q * PN;
  const T* Bp = S + A_B * PN;
  auto q = [&](int v, long long off) -> T { return Q[v * PN + o + off]; };
  auto u = [&](int v, long long off) -> T { return Bp[(v - IA) * PN + o + off]; };
  T vv, ww, uu, A, B, C;
  vv = T(0.25) * (q(IV, -sy - sz) + q(IV, -sy) + q(IV, -sz) + q(IV, 0));
  ww = T(0.25) * (q(IW, -sy - sz) + q(IW, -sy) + q(IW, -sz) + q(IW, 0));
  B = T(0.5) * (u(IB, -sz) + u(IB, 0));
  C = T(0.5) * (u(IC, -sy) + u(IC, 0));
  S[(A_E + 0) * PN + o] = vv * C - ww * B;
  uu = T(0.25) * (q(IU, -sx - sz) + q(IU, -sx) + q(IU, -sz) + q(IU, 0));
  ww = T(0.25) * (q(IW, -sx - sz) + q(IW, -sx) + q(IW, -sz) + q(IW, 0));
  A = T(0.5) * (u(IA, -sz) + u(IA, 0));
  C = T(0.5) * (u(IC, -sx) + u(IC, 0));
  S[(A_E + 1) * PN + o] = ww * A - uu * C;
  uu = T(0.25) * (q(IU, -sx - sy) + q(IU, -sx) + q(IU, -sy) + q(IU, 0));
  vv = T(0.25) * (q(IV, -sx - sy) + q(IV, -sx) + q(IV, -sy) + q(IV, 0));
  A = T(0.5) * (u(IA, -sy) + u(IA, 0));
  B = T(0.5) * (u(IB, -sx) + u(IB, 0));
  S[(A_E + 2) * PN + o] = uu * B - vv * A;
}

template <class T>
__global__ __launch_bounds__(256) void efield_kernel(T* __restrict__ S, Work3 w, StepCtl ctl)
{
  double dt;
  if (!step_dt(ctl, dt))
    return;
  int i, j, k;
  if (!cell_of<T>(w, i, j, k))
    return;
  efield_cell<T>(S, w, i, j, k);
}

// Inputs of the 3D trace of one cell, gathered from wherever the caller keeps them.
template <class T>
struct TraceIn {
  T qc[NV];                  // primitives of the cell
  T dqx[NV], dqy[NV], dqz[NV];  // their slopes (slope1 of the neighbours along x, y, z)
  T ELL, ELR, ERL, ERR;      // Ex at (j, k), (j, k+1), (j+1, k), (j+1, k+1)
  T FLL, FLR, FRL, FRR;      // Ey at (i, k), (i, k+1), (i+1, k), (i+1, k+1)
  T GLL, GLR, GRL, GRR;      // Ez at (i, j), (i, j+1), (i+1, j), (i+1, j+1)
  T AL, AR, BL, BR, CL, CR;  // the cell's own face fields (left/right)
};

// The half-step record of one cell (trace_unsplit_mhd_3d_simpler): `put(k, value)` receives
// the 35 values K_C .. K_Z+6.
template <class T, int ST, class Put>
__device__ __forceinline__ void trace_record(const TraceIn<T>& in, const Gas<T>& gas, T dtdx, T dtdy, T dtdz,
                                             Put put)
{
  const T* qc = in.qc;
  const T* dqx = in.dqx;
  const T* dqy = in.dqy;
  const T* dqz = in.dqz;
  const T ELL = in.ELL, ELR = in.ELR, ERL = in.ERL, ERR = in.ERR;
  const T FLL = in.FLL, FLR = in.FLR, FRL = in.FRL, FRR = in.FRR;
  const T GLL = in.GLL, GLR = in.GLR, GRL = in.GRL, GRR = in.GRR;
  T r = qc[ID], p = qc[IP], u = qc[IU], v = qc[IV], ww = qc[IW], A = qc[IA], B = qc[IB], C = qc[IC];
  T AL = in.AL, AR = in.AR, BL = in.BL, BR = in.BR, CL = in.CL, CR = in.CR;
  const T h = T(0.5);
  const T drx = dqx[ID] * h, dpx = dqx[IP] * h, dux = dqx[IU] * h, dvx = dqx[IV] * h, dwx = dqx[IW] * h;
  const T dCx = dqx[IC] * h, dBx = dqx[IB] * h;
  const T dry = dqy[ID] * h, dpy = dqy[IP] * h, duy = dqy[IU] * h, dvy = dqy[IV] * h, dwy = dqy[IW] * h;
  const T dCy = dqy[IC] * h, dAy = dqy[IA] * h;
  const T drz = dqz[ID] * h, dpz = dqz[IP] * h, duz = dqz[IU] * h, dvz = dqz[IV] * h, dwz = dqz[IW] * h;
  const T dAz = dqz[IA] * h, dBz = dqz[IB] * h;
  const T dAx = h * (AR - AL), dBy = h * (BR - BL), dCz = h * (CR - CL);
  const T gamma = gas.gamma0;
  const T sr0 = (-u * drx - dux * r) * dtdx + (-v * dry - dvy * r) * dtdy + (-ww * drz - dwz * r) * dtdz;
  const Inv<T> ir = inv_of(r);
  // (plain: in FP32 the y and z terms fuse into the sum, the x term's product is rounded)
  const T su0 = plain((-u * dux - quot_any(dpx + B * dBx + C * dCx, ir)) * dtdx) +
                (-v * duy + quot_any(B * dAy, ir)) * dtdy + (-ww * duz + quot_any(C * dAz, ir)) * dtdz;
  const T sv0 = (-u * dvx + quot_any(A * dBx, ir)) * dtdx + (-v * dvy - quot_any(dpy + A * dAy + C * dCy, ir)) * dtdy +
                (-ww * dvz + quot_any(C * dBz, ir)) * dtdz;
  const T sw0 = (-u * dwx + quot_any(A * dCx, ir)) * dtdx + (-v * dwy + quot_any(B * dCy, ir)) * dtdy +
                (-ww * dwz - quot_any(dpz + A * dAz + B * dBz, ir)) * dtdz;
  const T sp0 = (-u * dpx - dux * gamma * p) * dtdx + (-v * dpy - dvy * gamma * p) * dtdy +
                (-ww * dpz - dwz * gamma * p) * dtdz;
  const T sA0 = (u * dBy + B * duy - v * dAy - A * dvy) * dtdy + (u * dCz + C * duz - ww * dAz - A * dwz) * dtdz;
  const T sB0 = (v * dAx + A * dvx - u * dBx - B * dux) * dtdx + (v * dCz + C * dvz - ww * dBz - B * dwz) * dtdz;
  const T sC0 = (ww * dAx + A * dwx - u * dCx - C * dux) * dtdx + (ww * dBy + B * dwy - v * dCy - C * dvy) * dtdy;
  const T sAL0 = +(GLR - GLL) * dtdy * h - (FLR - FLL) * dtdz * h;
  const T sAR0 = +(GRR - GRL) * dtdy * h - (FRR - FRL) * dtdz * h;
  const T sBL0 = -(GRL - GLL) * dtdx * h + (ELR - ELL) * dtdz * h;
  const T sBR0 = -(GRR - GLR) * dtdx * h + (ERR - ERL) * dtdz * h;
  const T sCL0 = +(FRL - FLL) * dtdx * h - (ERL - ELL) * dtdy * h;
  const T sCR0 = +(FRR - FLR) * dtdx * h - (ERR - ELR) * dtdy * h;
  r = r + sr0;
  u = u + su0;
  v = v + sv0;
  ww = ww + sw0;
  p = p + sp0;
  A = A + sA0;
  B = B + sB0;
  C = C + sC0;
  AL = AL + sAL0;
  AR = AR + sAR0;
  BL = BL + sBL0;
  BR = BR + sBR0;
  CL = CL + sCL0;
  CR = CR + sCR0;
  put(K_C + ID, r);
  put(K_C + IP, p);
  put(K_C + IU, u);
  put(K_C + IV, v);
  put(K_C + IW, ww);
  put(K_C + IA, A);
  put(K_C + IB, B);
  put(K_C + IC, C);
  put(K_AL, AL);
  put(K_AR, AR);
  put(K_BL, BL);
  put(K_BR, BR);
  put(K_CL, CL);
  put(K_CR, CR);
  put(K_X + 0, drx);
  put(K_X + 1, dpx);
  put(K_X + 2, dux);
  put(K_X + 3, dvx);
  put(K_X + 4, dwx);
  put(K_X + 5, dBx);
  put(K_X + 6, dCx);
  put(K_Y + 0, dry);
  put(K_Y + 1, dpy);
  put(K_Y + 2, duy);
  put(K_Y + 3, dvy);
  put(K_Y + 4, dwy);
  put(K_Y + 5, dAy);
  put(K_Y + 6, dCy);
  put(K_Z + 0, drz);
  put(K_Z + 1, dpz);
  put(K_Z + 2, duz);
  put(K_Z + 3, dvz);
  put(K_Z + 4, dwz);
  put(K_Z + 5, dAz);
  put(K_Z + 6, dBz);
}

// ------------------------------------------------------------------------------------------
// Trace, fluxes and EMFs in one kernel, marching along z. A block owns FCX x FCY columns of
// cells (one wave of 64) and a chunk of planes. Per plane the records of its cells and of
// the row and column before them go to LDS; then wave t runs task t for the 64 cells: 0 the
// three Riemann problems, 1..3 the EMF z, y, x. What the plane above needs of this one (the
// upper z-face state, the two upper edge states of EMF y and x) is kept in LDS beside them, so only
// one plane of records is ever kept and none goes to memory.
//
// Bound by VALU issue and, in the trace, by load latency. With the records in memory (a trace
// kernel writing 35 arrays, a flux/EMF kernel reading them up to four times over: 3 of the 6 GB
// a 128^3 FP64 step moved, its loads saturating the texture addressers at 11 cycles each) the
// two kernels took 845 us (FP64) and 418 us (FP32) at 128^3; this one 630 and 245, the step 1255
// -> 931 and 590 -> 398, and 97x64x110 FP32 180 -> 143. What is kept for the next plane in
// registers instead of LDS: 1145 and 461 us per step (238 registers, or spills).
constexpr int FCX = 16, FCY = 4, FCN = 256;
constexpr int FRX = FCX + 1, FRN = (FCX + 1) * (FCY + 1); // records: one row and column more
// waves per SIMD = blocks per CU: 168 and 80 registers, 46 and 23 KB of LDS
template <class T>
constexpr int FCW = sizeof(T) == 8 ? 3 : 6;
constexpr int K_DB = K_N, K_ALL = K_N + 6; // LDS record: the half-step record, then 6 face-field slopes

template <class T>
struct RecLds {
  const T* s;
  __device__ __forceinline__ T operator()(int kk, int c) const { return s[kk * FRN + c]; }
  __device__ __forceinline__ T db(int m, int c) const { return s[(K_DB + m) * FRN + c]; }
};

// Face state of record c along dir (0..2): maxface -> qm (centre + half slope, FACE_*MAX),
// else qp (centre - half slope); the normal field is the face's own. Floors as the 3D trace
// (trace_unsplit_mhd_3d_simpler): rho by smallr, p by smallp.
template <class T>
__device__ __forceinline__ void face_state(const RecLds<T>& R, int c, int dir, bool maxface, const Gas<T>& gas, T* q)
{
  const int K = K_X + 7 * dir;
#pragma unroll
  for (int v = 0; v < 5; v++)
    q[v] = maxface ? R(K_C + v, c) + R(K + v, c) : R(K_C + v, c) - R(K + v, c);
  const int m1 = dir == 0 ? IB : IA, m2 = dir == 2 ? IB : IC, mn = dir == 0 ? IA : (dir == 1 ? IB : IC);
  q[m1] = maxface ? R(K_C + m1, c) + R(K + 5, c) : R(K_C + m1, c) - R(K + 5, c);
  q[m2] = maxface ? R(K_C + m2, c) + R(K + 6, c) : R(K_C + m2, c) - R(K + 6, c);
  q[mn] = R((maxface ? K_AR : K_AL) + 2 * dir, c);
  q[ID] = emax(gas.smallr, q[ID]);
  q[IP] = emax(gas.smallp, q[IP]);
}

// Edge states 0..3 = RT, RB, LT, LB of a record: over the two transverse directions (X: y, z;
// Y: x, z; Z: x, y) a state is centre + (+-s1 +- s2) (RT ++, RB +-, LT -+, LB --); the two
// transverse face fields are the right or left face value plus or minus its own transverse
// half slope, h*DB at that face (ComputeMagSlopesFunctor3D's slopes, halved as the trace does).
template <class T>
__device__ __forceinline__ T edge_comb(int e, T base, T a, T b)
{
  const T t = e < 2 ? a : -a;
  return base + ((e & 1) == 0 ? t + b : t - b);
}

// Along Z, as the edge solver reads it.
template <class T>
__device__ __forceinline__ Edge<T> edge_along_z(const RecLds<T>& R, int c, int e, const Gas<T>& gas)
{
  const T h = T(0.5);
  const bool p1 = e < 2, p2 = (e & 1) == 0;
  auto comb = [&](int v, int kx, int ky) { return edge_comb(e, R(K_C + v, c), R(K_X + kx, c), R(K_Y + ky, c)); };
  Edge<T> s;
  s.r = emax(gas.smallr, comb(ID, ID, ID));
  s.p = emax(gas.smallp, comb(IP, IP, IP));
  s.u = comb(IU, IU, IU);
  s.v = comb(IV, IV, IV);
  s.c = comb(IC, 6, 6);
  const T sa = p1 ? h * R.db(0, c + 1) : h * R.db(0, c);     // dARy / dALy
  s.a = (p1 ? R(K_AR, c) : R(K_AL, c)) + (p2 ? sa : -sa);
  const T sb = p2 ? h * R.db(2, c + FRX) : h * R.db(2, c);   // dBRx / dBLx
  s.b = (p2 ? R(K_BR, c) : R(K_BL, c)) + (p1 ? sb : -sb);
  return s;
}

// Along X (d = 0) or Y (d = 1), all but the slope of the C face, which belongs to the plane of
// that face: an upper state (RT, LT) is made on its own plane and closed on the next one.
template <class T>
struct OpenEdge {
  T r, p, t, w, f, g, cf;
};

template <class T>
__device__ __forceinline__ OpenEdge<T> open_edge(const RecLds<T>& R, int c, int e, int d, const Gas<T>& gas)
{
  const T h = T(0.5);
  const bool p1 = e < 2, p2 = (e & 1) == 0;
  const int K1 = d == 0 ? K_Y : K_X, vt = d == 0 ? IV : IU;
  auto comb = [&](int v) { return edge_comb(e, R(K_C + v, c), R(K1 + v, c), R(K_Z + v, c)); };
  OpenEdge<T> s;
  s.r = emax(gas.smallr, comb(ID));
  s.p = emax(gas.smallp, comb(IP));
  s.t = comb(vt);
  s.w = comb(IW);
  if (d == 0) {
    s.g = edge_comb(e, R(K_C + IA, c), R(K_Y + 5, c), R(K_Z + 5, c));
    const T sb = p1 ? h * R.db(3, c + FRX) : h * R.db(3, c); // dBRz / dBLz
    s.f = (p1 ? R(K_BR, c) : R(K_BL, c)) + (p2 ? sb : -sb);
  } else {
    s.g = edge_comb(e, R(K_C + IB, c), R(K_X + 5, c), R(K_Z + 6, c));
    const T sa = p1 ? h * R.db(1, c + 1) : h * R.db(1, c); // dARz / dALz
    s.f = (p1 ? R(K_AR, c) : R(K_AL, c)) + (p2 ? sa : -sa);
  }
  s.cf = p2 ? R(K_CR, c) : R(K_CL, c);
  return s;
}

// The whole state, R holding the plane of its C face.
template <class T>
__device__ __forceinline__ Edge<T> close_edge(const RecLds<T>& R, const OpenEdge<T>& o, int c, int e, int d)
{
  const T sc = T(0.5) * R.db(d == 0 ? 5 : 4, c); // dC/dy, dC/dx at the face
  const T C = o.cf + (e < 2 ? sc : -sc);
  Edge<T> s;
  s.r = o.r;
  s.p = o.p;
  if (d == 0) {
    s.u = o.t; s.v = o.w; s.a = o.f; s.b = C; s.c = o.g;
  } else {
    s.u = o.w; s.v = o.t; s.a = C; s.b = o.f; s.c = o.g;
  }
  return s;
}

// Record of padded cell (i, j, k) and the face-field slopes at its left faces, into LDS slot c.
template <class T, int ST>
__device__ __forceinline__ void record_to_lds(const T* __restrict__ S, const Work3& w, const Gas<T>& gas, T dtdx,
                                              T dtdy, T dtdz, int i, int j, int k, T* sR, int c)
{
  const long long PN = w.PN;
  const unsigned o = pidx(w, i, j, k) * (unsigned)sizeof(T), sx = sizeof(T), sy = (unsigned)w.PX * (unsigned)sizeof(T);
  const unsigned sz = (unsigned)(w.PX * w.PY) * (unsigned)sizeof(T);
  auto q = [&](int v, unsigned off) { return ldb(S + (A_Q + v) * PN, off); };
  auto u = [&](int v, unsigned off) { return ldb(S + (A_B + v - IA) * PN, off); };
  auto E = [&](int v, unsigned off) { return ldb(S + (A_E + v) * PN, off); };
  TraceIn<T> in;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const T qc = q(v, o);
    in.qc[v] = qc;
    in.dqx[v] = slope1<T, ST>(qc, q(v, o + sx), q(v, o - sx));
    in.dqy[v] = slope1<T, ST>(qc, q(v, o + sy), q(v, o - sy));
    in.dqz[v] = slope1<T, ST>(qc, q(v, o + sz), q(v, o - sz));
  }
  in.ELL = E(0, o);
  in.ELR = E(0, o + sz);
  in.ERL = E(0, o + sy);
  in.ERR = E(0, o + sy + sz);
  in.FLL = E(1, o);
  in.FLR = E(1, o + sz);
  in.FRL = E(1, o + sx);
  in.FRR = E(1, o + sx + sz);
  in.GLL = E(2, o);
  in.GLR = E(2, o + sy);
  in.GRL = E(2, o + sx);
  in.GRR = E(2, o + sx + sy);
  in.AL = u(IA, o);
  in.AR = u(IA, o + sx);
  in.BL = u(IB, o);
  in.BR = u(IB, o + sy);
  in.CL = u(IC, o);
  in.CR = u(IC, o + sz);
  // slope_unsplit_mhd_3d with xslope_type = min(slope_type, 2) (MHDBaseFunctor3D.h:563-668):
  // dA/dy, dA/dz, dB/dx, dB/dz, dC/dx, dC/dy (full, not halved)
  sR[(K_DB + 0) * FRN + c] = slope1<T, ST>(in.AL, u(IA, o + sy), u(IA, o - sy));
  sR[(K_DB + 1) * FRN + c] = slope1<T, ST>(in.AL, u(IA, o + sz), u(IA, o - sz));
  sR[(K_DB + 2) * FRN + c] = slope1<T, ST>(in.BL, u(IB, o + sx), u(IB, o - sx));
  sR[(K_DB + 3) * FRN + c] = slope1<T, ST>(in.BL, u(IB, o + sz), u(IB, o - sz));
  sR[(K_DB + 4) * FRN + c] = slope1<T, ST>(in.CL, u(IC, o + sx), u(IC, o - sx));
  sR[(K_DB + 5) * FRN + c] = slope1<T, ST>(in.CL, u(IC, o + sy), u(IC, o - sy));
  trace_record<T, ST>(in, gas, dtdx, dtdy, dtdz, [&](int kk, T x) { sR[kk * FRN + c] = x; });
}

// Columns i0.., j0.. over planes [k0, k1) of the padded grid (from 3, nfaces of each): fluxes of
// each cell's lower faces and EMFs of its lower edges (ComputeFluxesAndStoreFunctor3D_MHD,
// ComputeEmfAndStoreFunctor3D).
template <class T, int RS, int ST>
__device__ __forceinline__ void fluxemf_columns(T* __restrict__ S, const Work3& w, const Geom<T>& geo,
                                                const Gas<T>& gas, double dt, int i0, int j0, int k0, int k1)
{
  __shared__ T sR[K_ALL * FRN];
  const T dtdx = T(dt / geo.dx), dtdy = T(dt / geo.dy), dtdz = T(dt / geo.dz);
  const int tid = threadIdx.x, lane = tid & 63;
  const int task = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long PN = w.PN;
  // records: one per thread, the columns past the grid's end clamped to its last (their
  // values reach only cells that are not stored)
  const int ri = min(i0 - 1 + tid % FRX, w.PX - 3), rj = min(j0 - 1 + tid / FRX, w.PY - 3);
  const int lx = lane % FCX, ly = lane / FCX;
  const int c = (ly + 1) * FRX + lx + 1; // this lane's cell among the records
  const bool valid = i0 + lx < 3 + nfaces(geo, 0) && j0 + ly < 3 + nfaces(geo, 1);
  const RecLds<T> R{ sR };
  // what each lane keeps for the plane above: task 0 the cell's upper z-face state, tasks 2 and 3
  // the RT and LT edge states. In LDS, each lane its own column: in registers they would be live
  // through the trace, which has the most of its own.
  __shared__ T sH[NV + 28][64];
  T(*const hold)[64] = sH + (task == 2 ? NV : task == 3 ? NV + 14 : 0);
  auto keep = [&](int n, const OpenEdge<T>& e) {
    hold[n][lane] = e.r; hold[n + 1][lane] = e.p; hold[n + 2][lane] = e.t; hold[n + 3][lane] = e.w;
    hold[n + 4][lane] = e.f; hold[n + 5][lane] = e.g; hold[n + 6][lane] = e.cf;
  };
  auto kept = [&](int n) {
    return OpenEdge<T>{ hold[n][lane], hold[n + 1][lane], hold[n + 2][lane], hold[n + 3][lane],
                        hold[n + 4][lane], hold[n + 5][lane], hold[n + 6][lane] };
  };
  for (int k = k0 - 1; k < k1; k++) {
    if (tid < FRN)
      record_to_lds<T, ST>(S, w, gas, dtdx, dtdy, dtdz, ri, rj, k, sR, tid);
    __syncthreads();
    const bool out = k >= k0 && valid;
    const long long o = pidx(w, i0 + lx, j0 + ly, k);
    // distance to the copy of this cell's faces and edges past the end of a periodic axis, or 0
    const long long cx = lx == 0 && i0 == 3 && wraps(geo, 0) ? w.nx : 0;
    const long long cy = ly == 0 && j0 == 3 && wraps(geo, 1) ? (long long)w.ny * w.PX : 0;
    const long long cz = k == 3 && wraps(geo, 2) ? (long long)w.nz * w.PX * w.PY : 0;
    auto put_flux = [&](int dir, long long d, T f0, T f1, T f2, T f3, T f4) {
      if (!out)
        return;
      T* F = S + (A_FLUX + 5 * dir) * PN + o;
      F[0] = f0; F[PN] = f1; F[2 * PN] = f2; F[3 * PN] = f3; F[4 * PN] = f4;
      if (d) {
        F += d;
        F[0] = f0; F[PN] = f1; F[2 * PN] = f2; F[3 * PN] = f3; F[4 * PN] = f4;
      }
    };
    auto put_emf = [&](int dir, long long d1, long long d2, T e) {
      if (!out)
        return;
      T* F = S + (A_EMF + dir) * PN + o;
      F[0] = e;
      if (d1)
        F[d1] = e;
      if (d2)
        F[d2] = e;
      if (d1 && d2)
        F[d1 + d2] = e;
    };
    if (task == 0) {
      if (k >= k0) {
        T ql[NV], qr[NV], f[NV];
        // x: qm_x(i-1) | qp_x(i)
        face_state<T>(R, c - 1, 0, true, gas, ql);
        face_state<T>(R, c, 0, false, gas, qr);
        riemann<T, RS>(gas, ql, qr, f);
        put_flux(0, cx, f[ID], f[IP], f[IU], f[IV], f[IW]);
        // y: qm_y(j-1) | qp_y(j), IU<->IV and IA<->IB around the solve
        face_state<T>(R, c - FRX, 1, true, gas, ql);
        face_state<T>(R, c, 1, false, gas, qr);
        {
          T t;
          t = ql[IU]; ql[IU] = ql[IV]; ql[IV] = t;
          t = ql[IA]; ql[IA] = ql[IB]; ql[IB] = t;
          t = qr[IU]; qr[IU] = qr[IV]; qr[IV] = t;
          t = qr[IA]; qr[IA] = qr[IB]; qr[IB] = t;
        }
        riemann<T, RS>(gas, ql, qr, f);
        put_flux(1, cy, f[ID], f[IP], f[IV], f[IU], f[IW]);
        // z: qm_z(k-1) | qp_z(k), IU<->IW and IA<->IC around the solve
        face_state<T>(R, c, 2, false, gas, qr);
        {
          T t;
#pragma unroll
          for (int v = 0; v < NV; v++)
            ql[v] = hold[v][lane];
          t = ql[IU]; ql[IU] = ql[IW]; ql[IW] = t;
          t = ql[IA]; ql[IA] = ql[IC]; ql[IC] = t;
          t = qr[IU]; qr[IU] = qr[IW]; qr[IW] = t;
          t = qr[IA]; qr[IA] = qr[IC]; qr[IC] = t;
        }
        riemann<T, RS>(gas, ql, qr, f);
        put_flux(2, cz, f[ID], f[IP], f[IW], f[IV], f[IU]);
      }
      T up[NV];
      face_state<T>(R, c, 2, true, gas, up);
#pragma unroll
      for (int v = 0; v < NV; v++)
        hold[v][lane] = up[v];
    } else if (task == 1) {
      // EMF z: RT(i-1,j-1), RB(i-1,j), LT(i,j-1), LB(i,j) of the Z edges
      if (k >= k0) {
        const T e = emf_z<T>(gas, edge_along_z<T>(R, c - 1 - FRX, 0, gas), edge_along_z<T>(R, c - 1, 1, gas),
                             edge_along_z<T>(R, c - FRX, 2, gas), edge_along_z<T>(R, c, 3, gas));
        put_emf(2, cx, cy, e);
      }
    } else if (task == 2) {
      // EMF y: RT(i-1,k-1), LT(i,k-1) in the RB place, RB(i-1,k) in the LT place, LB(i,k)
      if (k >= k0) {
        const T e = emf_z<T>(gas, close_edge<T>(R, kept(0), c - 1, 0, 1), close_edge<T>(R, kept(7), c, 2, 1),
                             close_edge<T>(R, open_edge<T>(R, c - 1, 1, 1, gas), c - 1, 1, 1),
                             close_edge<T>(R, open_edge<T>(R, c, 3, 1, gas), c, 3, 1));
        put_emf(1, cx, cz, e);
      }
      keep(0, open_edge<T>(R, c - 1, 0, 1, gas));
      keep(7, open_edge<T>(R, c, 2, 1, gas));
    } else {
      // EMF x: RT(j-1,k-1), RB(j-1,k), LT(j,k-1), LB(j,k)
      if (k >= k0) {
        const T e = emf_z<T>(gas, close_edge<T>(R, kept(0), c - FRX, 0, 0),
                             close_edge<T>(R, open_edge<T>(R, c - FRX, 1, 0, gas), c - FRX, 1, 0),
                             close_edge<T>(R, kept(7), c, 2, 0), close_edge<T>(R, open_edge<T>(R, c, 3, 0, gas), c, 3, 0));
        put_emf(0, cy, cz, e);
      }
      keep(0, open_edge<T>(R, c - FRX, 0, 0, gas));
      keep(7, open_edge<T>(R, c, 2, 0, gas));
    }
    __syncthreads(); // every read of this plane's records is done
  }
}

// Tiles of the flux/EMF kernel on a grid and its z-chunk length (z_chunk_of, its constants fitted
// to 11 grids from 20^3 to 160^3 at every chunk length to 40: within 0.8 % of the fastest on
// average, 4.2 % at worst).
struct FluxGrid {
  int ntx, nty, ntz, cz;
};

template <class T>
inline FluxGrid flux_grid(const Geom<T>& geo)
{
  FluxGrid g;
  g.ntx = (nfaces(geo, 0) + FCX - 1) / FCX;
  g.nty = (nfaces(geo, 1) + FCY - 1) / FCY;
  const int n = nfaces(geo, 2);
  g.cz = z_chunk_of((long long)g.ntx * g.nty, n, 256 * FCW<T>, sizeof(T) == 8 ? 0.3 : 0.5, sizeof(T) == 8 ? 0.2 : 0.1, 1, 40);
  g.ntz = (n + g.cz - 1) / g.cz;
  return g;
}

template <class T, int RS, int ST>
__global__ __launch_bounds__(FCN) __attribute__((amdgpu_waves_per_eu(FCW<T>))) void fluxemf_kernel(T* __restrict__ S, Work3 w, Geom<T> geo, Gas<T> gas, StepCtl ctl,
                                                      int cz, int ntx, int nty)
{
  double dt;
  if (!step_dt(ctl, dt))
    return;
  const int b = (int)xcd_order(blockIdx.x, gridDim.x);
  const int tx = b % ntx, ty = (b / ntx) % nty, tz = b / (ntx * nty);
  fluxemf_columns<T, RS, ST>(S, w, geo, gas, dt, 3 + tx * FCX, 3 + ty * FCY, 3 + tz * cz,
                             min(3 + (tz + 1) * cz, 3 + nfaces(geo, 2)));
}

// CFL term of a 3D cell from its new state and new right/top/front face fields
template <class T>
__device__ __forceinline__ double cfl3(const Gas<T>& gas, const T* u, T mx, T my, T mz, const Geom<T>& geo)
{
  if constexpr (sizeof(T) == 8) {
    T q[NV];
    constoprim<T>(gas, u, mx, my, mz, q);
    const T d = q[ID], p = q[IP], a = q[IA], b = q[IB], c = q[IC];
    const T b2 = a * a + b * b + c * c;
    const Inv<T> id = inv_of(d);
    const T c2 = quot(gas.gamma0 * p, id);
    const T d2 = T(0.5) * (quot(b2, id) + c2);
    const T vx = esqrt(d2 + esqrt(d2 * d2 - quot(c2 * a * a, id))) + eabs(q[IU]);
    const T vy = esqrt(d2 + esqrt(d2 * d2 - quot(c2 * b * b, id))) + eabs(q[IV]);
    const T vz = esqrt(d2 + esqrt(d2 * d2 - quot(c2 * c * c, id))) + eabs(q[IW]);
    if (geo.pow2)
      return vx * geo.idx + vy * geo.idy + vz * geo.idz;
    return quot(vx, inv_with(geo.dx, geo.rdx)) + quot(vy, inv_with(geo.dy, geo.rdy)) +
           quot(vz, inv_with(geo.dz, geo.rdz));
  } else {
    return mhd_cfl_widened<3>(gas, u, (double)mx, (double)my, (double)mz, geo.rdx, geo.rdy, geo.rdz);
  }
}

// Flux update, CT update and the CFL term of the new state of interior cell c
// (UpdateFunctor3D_MHD + UpdateEmfFunctor3D + ComputeDtFunctor3D_MHD on the result).
template <class T>
__device__ __forceinline__ double update_cell(const T* __restrict__ Uin, const T* __restrict__ S, T* __restrict__ Uout, const Work3& w,
                                              const Geom<T>& geo, const Gas<T>& gas, T dtdx, T dtdy, T dtdz,
                                              long long c)
{
  const long long n = geo.vstride;
  {
    int ii, jj, kk;
    split3((unsigned)c, (unsigned)w.nx, (unsigned)w.ny, ii, jj, kk);
    const long long PN = w.PN;
    // byte offsets: this cell of the padded grid, its strides, this cell of the output
    const unsigned o = pidx(w, ii + 3, jj + 3, kk + 3) * (unsigned)sizeof(T);
    const unsigned sx = sizeof(T), sy = (unsigned)w.PX * (unsigned)sizeof(T);
    const unsigned sz = (unsigned)(w.PX * w.PY) * (unsigned)sizeof(T);
    const unsigned ob = (unsigned)c * (unsigned)sizeof(T);
    auto at = [&](int a, unsigned off) -> T { return ldb(S + a * PN, off); };
    T u[NV];
#pragma unroll
    for (int v = 0; v < NV; v++)
      u[v] = v < IA ? ldb(Uin + v * n, ob) : at(A_B + v - IA, o);
    constexpr int hv[5] = { ID, IP, IU, IV, IW };
#pragma unroll
    for (int m = 0; m < 5; m++) {
      T a = u[hv[m]];
      a += at(A_FLUX + m, o) * dtdx;
      a -= at(A_FLUX + m, o + sx) * dtdx;
      a += at(A_FLUX + 5 + m, o) * dtdy;
      a -= at(A_FLUX + 5 + m, o + sy) * dtdy;
      a += at(A_FLUX + 10 + m, o) * dtdz;
      a -= at(A_FLUX + 10 + m, o + sz) * dtdz;
      u[hv[m]] = a;
    }
    auto EX = [&](unsigned off) -> T { return at(A_EMF + 0, off); };
    auto EY = [&](unsigned off) -> T { return at(A_EMF + 1, off); };
    auto EZ = [&](unsigned off) -> T { return at(A_EMF + 2, off); };
    u[IA] += (EZ(o + sy) - EZ(o)) * dtdy;
    u[IB] -= (EZ(o + sx) - EZ(o)) * dtdx;
    u[IA] -= (EY(o + sz) - EY(o)) * dtdz;
    u[IB] += (EX(o + sz) - EX(o)) * dtdz;
    u[IC] += (EY(o + sx) - EY(o)) * dtdx;
    u[IC] -= (EX(o + sy) - EX(o)) * dtdy;
#pragma unroll
    for (int v = 0; v < NV; v++)
      stb(Uout + v * n, ob, u[v]);
    // new face fields of the right / top / front neighbours, as the next ghost fill sees them
    T ar, bt, cf;
    if (ii + 1 < w.nx || geo.bc[1] == BC_PERIODIC) {
      const unsigned q = o + sx;
      ar = at(A_B + IA - IA, q);
      ar += (EZ(q + sy) - EZ(q)) * dtdy;
      ar -= (EY(q + sz) - EY(q)) * dtdz;
    } else {
      ar = geo.bc[1] == BC_DIRICHLET ? u[IA] * T(-1) : u[IA];
    }
    if (jj + 1 < w.ny || geo.bc[3] == BC_PERIODIC) {
      const unsigned q = o + sy;
      bt = at(A_B + IB - IA, q);
      bt -= (EZ(q + sx) - EZ(q)) * dtdx;
      bt += (EX(q + sz) - EX(q)) * dtdz;
    } else {
      bt = geo.bc[3] == BC_DIRICHLET ? u[IB] * T(-1) : u[IB];
    }
    if (kk + 1 < w.nz || geo.bc[5] == BC_PERIODIC) {
      const unsigned q = o + sz;
      cf = at(A_B + IC - IA, q);
      cf += (EY(q + sx) - EY(q)) * dtdx;
      cf -= (EX(q + sy) - EX(q)) * dtdy;
    } else {
      cf = geo.bc[5] == BC_DIRICHLET ? u[IC] * T(-1) : u[IC];
    }
    return cfl3<T>(gas, u, ar, bt, cf, geo);
  }
}

// update on the interior (UpdateFunctor3D_MHD + UpdateEmfFunctor3D) into the SoA output.
// A grid-stride loop over a bounded grid (MHD3_UPDATE_BLOCKS): each block ends with one
// atomic max on the time slot, and one short block per 256 cells (27k blocks at 192^3)
// made those atomics cost three quarters of the kernel's time.
constexpr unsigned MHD3_UPDATE_BLOCKS = 2048;

template <class T>
__global__ __launch_bounds__(256) void update_kernel(const T* __restrict__ Uin, const T* __restrict__ S, T* __restrict__ Uout, Work3 w,
                                                     Geom<T> geo, Gas<T> gas, StepCtl ctl)
{
  __shared__ double sred[4];
  double dt;
  TimeSlot cur;
  const bool first_block = blockIdx.x == 0;
  if (!step_begin(ctl, first_block, dt, cur))
    return;
  const T dtdx = T(dt / geo.dx), dtdy = T(dt / geo.dy), dtdz = T(dt / geo.dz);
  const long long n = geo.vstride;
  double local = 0.0;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    const double sv = update_cell<T>(Uin, S, Uout, w, geo, gas, dtdx, dtdy, dtdz, c);
    local = (sv > local || !(sv == sv)) ? sv : local;
  }
  block_max_to<256>(invdt_word(ctl, (ctl.slot + 1) % 3, blockIdx.x), local, sred);
  if (first_block && threadIdx.x < 64)
    step_end_bookkeeping(ctl, cur, dt);
}

// CFL reduction over a 3D MHD state (interior SoA), neighbours' face fields through the
// boundary map
template <class T>
__global__ __launch_bounds__(256) void inv_dt3_kernel(const T* __restrict__ U, Geom<T> geo, Gas<T> gas,
                                                      unsigned long long* dst, unsigned long long* spread,
                                                      int nspread)
{
  __shared__ double sred[4];
  const long long n = geo.vstride;
  const int nx = geo.nx, ny = geo.ny, nz = geo.nz;
  double local = 0.0;
  for (long long c = (long long)blockIdx.x * 256 + threadIdx.x; c < n; c += (long long)gridDim.x * 256) {
    int i, j, k;
    split3((unsigned)c, (unsigned)nx, (unsigned)ny, i, j, k);
    T u[NV];
#pragma unroll
    for (int v = 0; v < NV; v++)
      u[v] = U[v * n + c];
    bool fx, fy, fz;
    const int si = bc_map(i + 1, nx, geo.bc[0], geo.bc[1], fx);
    const int sj = bc_map(j + 1, ny, geo.bc[2], geo.bc[3], fy);
    const int sk = bc_map(k + 1, nz, geo.bc[4], geo.bc[5], fz);
    T mx = U[IA * n + ((long long)k * ny + j) * nx + si];
    T my = U[IB * n + ((long long)k * ny + sj) * nx + i];
    T mz = U[IC * n + ((long long)sk * ny + j) * nx + i];
    if (fx)
      mx = mx * T(-1);
    if (fy)
      my = my * T(-1);
    if (fz)
      mz = mz * T(-1);
    const double s = cfl3<T>(gas, u, mx, my, mz, geo);
    local = (s > local || !(s == s)) ? s : local;
  }
  block_max_to<256>(reduce_word(dst, spread, nspread), local, sred);
}

} // namespace mhd3
} // namespace ek
