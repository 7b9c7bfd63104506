"""3D steps that march over several planes: 8x16 hydro columns (turned) with remainders on every axis,
and the 3D MHD flux/EMF kernel with chunks of three planes and more, a short last chunk and ragged
columns, where what one plane keeps for the next is used plane after plane. FP64 is bitwise the
oracle's, FP32 within three steps' rounding of FP64 (each step rounds a few hundred (hydro) to a
thousand-odd (MHD) FP32 operations per cell: 1e-5 of the norm), a pooled job its single-grid run.
Every case first checks that its grid is launched with the tile and the chunk it is here for."""
import numpy as np
import pytest

from euler_kokkos_amd import native, pool
from euler_kokkos_amd.params import make_params

import test_mhd3d_gpu
import test_min_grids_gpu
import test_parity_gpu

pytestmark = pytest.mark.gpu

W, P = (1, 2, 3, 3, 2, 1), (3,) * 6
# shape, (planes, tile x, tile y) in FP64 and in FP32, None where FP32 takes 16x8 tiles
TURNED = [((7, 40, 30), (2, 8, 16), None), ((23, 97, 61), (2, 8, 16), (2, 8, 16)), ((23, 181, 20), (2, 8, 16), (2, 8, 16)),
          ((101, 75, 130), (12, 8, 16), (7, 8, 16))]
# shape, boundaries, planes per chunk in FP64 and FP32
MHD = [((64, 60, 53), P, 5, 3), ((64, 60, 50), W, 6, 3), ((100, 90, 40), W, 3, 6), ((97, 64, 43), P, 4, 4)]


def hydro(shape, rs, prec):
    return make_params("Hydro_Muscl_3D", *shape, riemann=rs, slope_type="2", cfl="0.5", bc=W, precision=prec)


def run(ekp, U0, steps):
    ctx = native.Context(ekp)
    try:
        ctx.upload(U0)
        ctx.run(steps, steps, 1e30)
        return ctx.download(native.EK_LAYOUT_SOA)
    finally:
        ctx.close()


@pytest.mark.parametrize("rs", ["hllc", "approx", "llf"])
@pytest.mark.parametrize("shape,fp64,fp32", TURNED)
def test_turned_columns(oracle, shape, fp64, fp32, rs):
    ekp = hydro(shape, rs, native.EK_FP64)
    assert native.z_chunk(ekp) == fp64
    U0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), False, 41)
    g, o = test_parity_gpu.run_pair(oracle, ekp, U0, 3)
    print(f"case=turned {shape} {rs}: {np.count_nonzero(g != o)} differ", flush=True)
    assert np.array_equal(g, o)
    if fp32:
        ekp32 = hydro(shape, rs, native.EK_FP32)
        assert native.z_chunk(ekp32) == fp32
        a, b = run(ekp, U0, 3), run(ekp32, U0, 3)
        assert np.linalg.norm(b - a) < 1e-5 * np.linalg.norm(a)


@pytest.mark.parametrize("riemann", ["hlld", "hll", "llf"])
@pytest.mark.parametrize("shape,bc,fp64,fp32", MHD)
def test_mhd_chunks(oracle, shape, bc, fp64, fp32, riemann):
    kw = dict(bc=bc, riemann=riemann, slope_type="1" if riemann == "llf" else "2")
    ekp = test_mhd3d_gpu.m3(*shape, **kw)
    assert native.z_chunk(ekp) == (fp64, 16, 4)
    R0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), True, 42)
    g, o = test_mhd3d_gpu.run_pair(oracle, ekp, R0, 3)
    print(f"case=mhd3d {shape} chunks of {fp64} {riemann}: {np.count_nonzero(g != o)} differ", flush=True)
    assert np.array_equal(g, o)
    ekp32 = test_mhd3d_gpu.m3(*shape, precision=native.EK_FP32, **kw)
    assert native.z_chunk(ekp32) == (fp32, 16, 4)
    a, b = run(ekp, R0, 3), run(ekp32, R0, 3)
    assert np.linalg.norm(b - a) < 1e-5 * np.linalg.norm(a)


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_pooled_mhd_chunks(oracle, prec):
    jobs = []
    for k, (shape, bc) in enumerate((((64, 60, 53), P), ((13, 9, 8), P), ((64, 60, 50), W))):
        ekp = test_mhd3d_gpu.m3(*shape, bc=bc, precision=prec)
        jobs.append((ekp, test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), True, 43 + k)))
    assert native.z_chunk(jobs[0][0])[0] >= 3
    p = pool.Pool(jobs[0][0], 1 << 30, len(jobs))
    try:
        ids = [p.admit(ekp, R0, 4, layout=native.EK_LAYOUT_REFERENCE) for ekp, R0 in jobs]
        p.step(4)
        for jid, (ekp, R0) in zip(ids, jobs):
            assert np.array_equal(p.download(jid), run(ekp, R0, 4))
    finally:
        p.close()
