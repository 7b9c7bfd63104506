"""2D MHD at the edges of its three tiles (14x6, 14x10, and 27x11 or 30x14) and of the estimate
that picks one: less than a tile, a tile, one cell more, and grids on both sides of the lines. A
tile changes where a cell is computed, never its result: FP64 is bitwise the oracle's, FP32 within
the rounding of its steps (each rounds a few hundred FP32 operations per cell: 1e-5 of the norm)."""
import numpy as np
import pytest

import test_mhd_gpu
from euler_kokkos_amd import native

pytestmark = pytest.mark.gpu


# FP64: 14x6 up to 512 blocks, then 27x11 (230x215), 14x10 (300x290, 351x340), 27x11 (700x420);
# FP32: 14x6 up to 230x215, 14x10 (300x211, 351x340), 30x14 (300x290, 700x420)
@pytest.mark.parametrize("shape", [(13, 5), (14, 6), (15, 7), (55, 23), (195, 193), (230, 215), (300, 211), (300, 290),
                                   (351, 340), (700, 420)])
@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_tiles(oracle, shape, prec):
    ekp = test_mhd_gpu.mparams(*shape, bc=(3, 3, 1, 2, 3, 3), precision=prec)
    op = oracle.from_ek(ekp)
    U0 = oracle.orszag_tang(op)
    U = U0.copy()
    oracle.mhd_run(op, U, 3, 1e30)
    ctx = native.Context(ekp)
    try:
        ctx.upload(U0)
        ctx.run(3, 3, 1e30)
        g, o = oracle.interior(op, ctx.download()), oracle.interior(op, U)
    finally:
        ctx.close()
    off = float(np.linalg.norm(g - o) / np.linalg.norm(o))
    print(f"case=mhd2d {shape} off {off:.3e}", flush=True)
    assert np.array_equal(g, o) if prec == native.EK_FP64 else off < 1e-5
