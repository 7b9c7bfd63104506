"""Device memory of a 3D MHD pool: of the 84 % of arena_bytes that its jobs' work areas count for, it
holds half, since an area of 78 counted reals per padded cell uses 32. What fits in the pool stays as
counted, and jobs that fill it do not share an element."""
import ctypes as C

import numpy as np
import pytest

from euler_kokkos_amd import native, pool

import test_mhd3d_gpu
import test_min_grids_gpu

pytestmark = pytest.mark.gpu


def free_bytes():
    native.lib()  # loads the library and, with it, its HIP runtime
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_held(prec):
    arena = 8 << 30
    pool.Pool(test_mhd3d_gpu.m3(8, 8, 8, precision=prec), 1 << 20, 2).close()  # what a first pool loads
    before = free_bytes()
    p = pool.Pool(test_mhd3d_gpu.m3(8, 8, 8, precision=prec), arena, 16)
    held = before - free_bytes()
    p.close()
    print(f"case=pool of {arena} bytes holds {held}", flush=True)
    assert held < 0.6 * arena


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_full_pool(oracle, prec):
    ekp = test_mhd3d_gpu.m3(13, 9, 8, precision=prec)
    R0 = [test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), True, 60 + k) for k in range(40)]
    p = pool.Pool(ekp, 12 * (19 * 15 * 14 * 78 + 13 * 9 * 8 * 16) * (8 if prec == native.EK_FP64 else 4), 64)
    ids = []
    try:
        with pytest.raises(pool.PoolFull):
            for R in R0:
                ids.append(p.admit(ekp, R, 3, layout=native.EK_LAYOUT_REFERENCE))
        assert 8 <= len(ids) <= 12
        p.step(3)
        for R, jid in zip(R0, ids):
            ctx = native.Context(ekp)
            ctx.upload(R)
            ctx.run(3, 3, 1e30)
            want = ctx.download(native.EK_LAYOUT_SOA)
            ctx.close()
            assert np.array_equal(p.download(jid), want)
    finally:
        p.close()
