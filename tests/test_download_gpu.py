"""Downloads by one thread and by several: sizes below the first split, a split whose parts differ
by a value, and the most parts. A state that took no step comes back as it went up: FP64 bit for
bit, FP32 rounded once."""
import ctypes as C

import numpy as np
import pytest

from euler_kokkos_amd import native, pool
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu

# 4 variables: 8 KB; 2 MB (FP64), one part; 9.1 MB, two; 16.7 MB, four; 50.6 MB, the most
SHAPES = [(16, 16), (301, 207), (541, 527), (724, 723), (1531, 1033)]


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
@pytest.mark.parametrize("shape", SHAPES)
def test_state_comes_back(shape, prec):
    p = make_params("Hydro_Muscl_2D", *shape, riemann="hllc", slope_type="2", cfl="0.5", bc=(3,) * 6, precision=prec)
    U = np.random.default_rng(sum(shape)).uniform(1.0, 2.0, (4, shape[1], shape[0]))
    U[1] += 10.0
    want = U if prec == native.EK_FP64 else U.astype(np.float32).astype(np.float64)
    ctx = native.Context(p)
    try:
        ctx.upload(U, native.EK_LAYOUT_SOA)
        assert np.array_equal(ctx.download(native.EK_LAYOUT_SOA), want)
        host = native.pinned_copy(np.zeros_like(U))  # a pinned destination too
        assert ctx._L.ek_download(ctx.h, host.ctypes.data_as(C.POINTER(C.c_double)), native.EK_LAYOUT_SOA) == 0
        assert np.array_equal(host, want)
    finally:
        ctx.close()
    P = pool.Pool(p, 128 << 20, 1)
    try:
        assert np.array_equal(P.download(P.admit(p, U, 1)), want)
    finally:
        P.close()
