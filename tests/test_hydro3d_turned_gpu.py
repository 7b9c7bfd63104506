"""3D hydro grids that take the 8x16 column tiles (fewer of them than of the 16x8 ones): less than a
tile, a tile, a cell more along y, ragged on every axis. FP64 is bitwise the oracle's, FP32 within
three steps' rounding of it (each step rounds a few hundred FP32 operations per cell: 1e-5 of the
norm)."""
import numpy as np
import pytest

from euler_kokkos_amd import native
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
@pytest.mark.parametrize("rs", ["hllc", "approx"])
@pytest.mark.parametrize("shape", [(7, 15, 3), (8, 16, 4), (8, 17, 5), (23, 30, 9), (24, 180, 20)])
def test_turned_tiles(oracle, shape, rs, prec):
    ekp = make_params("Hydro_Muscl_3D", *shape, riemann=rs, slope_type="2", cfl="0.5", bc=(1, 2, 3, 3, 2, 1), precision=prec)
    op = oracle.from_ek(ekp)
    U0 = oracle.blast(op, radius=0.25, center_x=0.45, center_y=0.55, center_z=0.5, density_in=1.0, density_out=1.0,
                      pressure_in=10.0, pressure_out=0.1)
    U = U0.copy()
    oracle.run(op, U, 3, 1e30)
    ctx = native.Context(ekp)
    try:
        ctx.upload(U0)
        ctx.run(3, 3, 1e30)
        g, o = oracle.interior(op, ctx.download()), oracle.interior(op, U)
    finally:
        ctx.close()
    off = float(np.linalg.norm(g - o) / np.linalg.norm(o))
    print(f"case=hydro3d {shape} {rs}: off {off:.3e}", flush=True)
    assert np.array_equal(g, o) if prec == native.EK_FP64 else off < 1e-5
