"""2D hydro at the edges of its tiles and of the rule that picks one from the grid's size: less
than a tile, a tile, one cell more, and grids on both sides of each line. A tile changes where a
cell is computed, never its result: FP64 is bitwise the oracle's, and a job of a pool is bitwise
its single-grid run with every tile of the pool, in both precisions."""
import numpy as np
import pytest

import test_parity_gpu
from euler_kokkos_amd import native, pool, problems
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu


def params(shape, rs, prec=native.EK_FP64):
    return make_params("Hydro_Muscl_2D", *shape, riemann=rs, slope_type="2", cfl="0.5", bc=(1, 2, 3, 3, 3, 3), precision=prec)


# small tiles up to 256 blocks of 16x8 (then up to 512 where the 16x12 tiles number over 256)
@pytest.mark.parametrize("shape", [(15, 7), (16, 8), (17, 9), (33, 13), (256, 128), (257, 128), (256, 256), (257, 256)])
@pytest.mark.parametrize("rs", ["hllc", "approx"])
def test_tiles_bitwise(oracle, shape, rs):
    ekp = params(shape, rs)
    op = oracle.from_ek(ekp)
    U0 = oracle.blast(op, radius=0.25, center_x=0.4, center_y=0.55, center_z=0.5, density_in=1.0,
                      density_out=1.0, pressure_in=10.0, pressure_out=0.1)
    g, o = test_parity_gpu.run_pair(oracle, ekp, U0, 4)
    assert np.array_equal(g, o)


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_pool_tiles_equal_single_runs(prec):
    for shape in [(7, 5), (33, 17), (200, 130), (300, 290)]:
        p = params(shape, "hllc", prec)
        U = problems.blast(p, radius="0.25", center_x="0.4", center_y="0.55")
        ctx = native.Context(p)
        try:
            ctx.upload(U, native.EK_LAYOUT_SOA)
            ctx.run(5, 5, 1e30)
            ref = ctx.download(native.EK_LAYOUT_SOA)
        finally:
            ctx.close()
        P = pool.Pool(p, 64 << 20, 2)
        try:
            for choice in range(4):
                P.set_tile(choice)
                j = P.admit(p, U, 5)
                P.step(5)
                assert np.array_equal(P.download(j), ref), (shape, choice)
                P.retire(j)
        finally:
            P.close()
