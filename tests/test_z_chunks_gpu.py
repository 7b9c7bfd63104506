"""3D hydro at the z-chunk lengths the estimate of hydro3d_z_chunk picks: two planes with a last
chunk of one, a single short chunk, long chunks with a short last one. Chunking changes where
planes are traced, never a result: FP64 is bitwise the oracle's, FP32 within three steps'
rounding of it (each step rounds a few hundred FP32 operations per cell: 1e-5 of the norm)."""
import numpy as np
import pytest

from euler_kokkos_amd import native
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
@pytest.mark.parametrize("shape,cz64,cz32", [((32, 24, 9), 2, 2), ((40, 40, 2), 2, 2), ((64, 64, 64), 4, 2),
                                             ((100, 90, 131), 15, 9), ((300, 200, 65), 22, 13)])
def test_chunk_lengths(oracle, shape, cz64, cz32, prec):
    ekp = make_params("Hydro_Muscl_3D", *shape, riemann="hllc", slope_type="2", cfl="0.5", bc=(3, 3, 1, 2, 2, 1),
                      precision=prec)
    U0 = oracle.blast(oracle.from_ek(ekp), radius=0.2, center_x=0.45, center_y=0.55, center_z=0.5,
                      density_in=1.0, density_out=1.0, pressure_in=10.0, pressure_out=0.1)
    op = oracle.from_ek(ekp)
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
    print(f"case=hydro3d {shape} (z-chunk {cz64 if prec == native.EK_FP64 else cz32}): off {off:.3e}", flush=True)
    assert np.array_equal(g, o) if prec == native.EK_FP64 else off < 1e-5
