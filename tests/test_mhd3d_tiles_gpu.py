"""3D MHD at the edges of the flux/EMF kernel's column tiles (16 x 4 cells, chunks of planes): one
cell under, at and over a tile, single-plane chunks, walls and outflow (one face more than
cells), periodic axes (the last face is stored by whoever computes the first) and axes periodic
on one side only. FP64 is bitwise the oracle's; FP32 is within two steps' rounding of FP64."""
import numpy as np
import pytest

from euler_kokkos_amd import native

import test_mhd3d_gpu
import test_min_grids_gpu

pytestmark = pytest.mark.gpu

P, W, O = (3, 3), (1, 1), (2, 2)
CASES = [((15, 3, 3), P + P + P), ((16, 4, 4), P + P + P), ((17, 5, 6), P + P + P), ((15, 3, 5), W + O + W),
         ((16, 4, 3), O + W + O), ((31, 7, 9), P + W + P), ((32, 9, 4), W + P + O), ((33, 8, 11), O + P + P),
         ((20, 6, 7), (3, 1, 2, 3, 3, 2)), ((48, 20, 17), P + P + W)]


@pytest.mark.parametrize("shape,bc", CASES)
@pytest.mark.parametrize("riemann", ["hlld", "hll", "llf"])
def test_fp64_bitwise(oracle, shape, bc, riemann):
    ekp = test_mhd3d_gpu.m3(*shape, bc=bc, riemann=riemann, slope_type="1" if riemann == "llf" else "2")
    R0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), True, 31)
    g, o = test_mhd3d_gpu.run_pair(oracle, ekp, R0, 3)
    print(f"case=mhd3d tiles {shape} bc={bc} {riemann}: max|diff|={np.max(np.abs(g - o)):.3e}", flush=True)
    assert np.array_equal(g, o)


@pytest.mark.parametrize("shape,bc", CASES)
def test_fp32_near_fp64(oracle, shape, bc):
    out = []
    for prec in (native.EK_FP64, native.EK_FP32):
        ekp = test_mhd3d_gpu.m3(*shape, bc=bc, precision=prec)
        R0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), True, 32)
        ctx = native.Context(ekp)
        try:
            ctx.upload(R0)
            ctx.run(2, 2, 1e30)
            out.append(ctx.download(native.EK_LAYOUT_SOA))
        finally:
            ctx.close()
    off = float(np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0]))
    print(f"case=mhd3d tiles fp32 {shape} bc={bc}: off {off:.3e}", flush=True)
    assert off < 1e-5  # two steps of a thousand-odd FP32 operations per cell
