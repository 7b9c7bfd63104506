"""Steps of 2D grids whose tiles have 2^32 threads and more between them, the most that one launch
takes: strips two or three cells wide, so that a tile holds few cells and the state stays small
(7 to 33 GB). The state repeats every 64 rows, and so does the result: it is bitwise the step of
the 64 rows alone, periodic."""
import ctypes as C

import numpy as np
import pytest

from euler_kokkos_amd import native, pool
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu

ROWS = 64


def strip(solver, nx, rows, period, precision):
    """Parameters of a strip of `rows` rows with the cells of the one of `period` rows."""
    p = make_params(solver, nx, rows, riemann="hlld" if solver.startswith("MHD") else "hllc", slope_type="2", cfl="0.5",
                    bc=(1, 2, 3, 3, 3, 3), precision=precision)
    p.dx, p.dy, p.ymax = 1.0 / nx, 1.0 / period, rows / period
    return p


def pattern(p, seed):
    rng = np.random.default_rng(seed)
    U = rng.uniform(-0.3, 0.3, (p.nbvar, ROWS, p.nx))
    U[0] = rng.uniform(1.0, 2.0, U[0].shape)
    U[1] = rng.uniform(3.0, 4.0, U[0].shape)
    return U.astype(np.float32).astype(np.float64)


def alone(p, U):
    ctx = native.Context(p)
    try:
        ctx.upload(U, native.EK_LAYOUT_SOA)
        ctx.run(2, 2, 1e30)
        return ctx.download(native.EK_LAYOUT_SOA)
    finally:
        ctx.close()


class Strip:
    """A device buffer of nbvar x rows x nx floats."""

    def __init__(self, p):
        native.lib()  # loads the library and, with it, its HIP runtime
        self.hip = C.CDLL("libamdhip64.so.7")
        self.hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.nbvar, self.bytes = p.nbvar, p.ny * p.nx * 4  # of one variable
        self.ptr = C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.ptr), self.nbvar * self.bytes) == 0

    def copy(self, dst, src, n, kind):
        assert self.hip.hipMemcpy(dst, src, n, kind) == 0

    def fill(self, U):
        """Every variable: its rows of U over and over, doubling what is there."""
        for v in range(self.nbvar):
            u = np.ascontiguousarray(U[v], dtype=np.float32)
            at, n = self.ptr.value + v * self.bytes, u.nbytes
            self.copy(at, u.ctypes.data, n, 1)
            while n < self.bytes:
                m = min(n, self.bytes - n)
                self.copy(at + n, at, m, 3)
                n += m

    def holds(self, U):
        part = native.pinned_empty((32768,) + U[0].shape, np.float32)
        for v in range(self.nbvar):
            for off in range(0, self.bytes, part.nbytes):
                n = min(part.nbytes, self.bytes - off)
                self.copy(part.ctypes.data, self.ptr.value + v * self.bytes + off, n, 2)
                if not (part.reshape(-1, U[v].size)[: n // 4 // U[v].size] == U[v].astype(np.float32).ravel()).all():
                    return False
        return True

    def free(self):
        assert self.hip.hipFree(self.ptr) == 0


@pytest.mark.parametrize("solver,nx,tile_rows,threads", [("Hydro_Muscl_2D", 2, 16, 512), ("MHD_Muscl_2D", 3, 10, 256)])
def test_single_grid(solver, nx, tile_rows, threads):
    rows = (2 ** 32 // threads * tile_rows // ROWS + 3) * ROWS
    small, large = (strip(solver, nx, n, ROWS, native.EK_FP32) for n in (ROWS, rows))
    U = pattern(small, 5)
    want = alone(small, U)
    print(f"case={solver} {nx}x{rows}", flush=True)
    a, b = Strip(large), Strip(large)
    try:
        a.fill(U)
        in_b = native.run_noalloc(large, a.ptr.value, b.ptr.value, 2, 2, 1e30)[3]
        assert (b if in_b else a).holds(want)
    finally:
        a.free()
        b.free()


def test_pool():
    rows = (2 ** 32 // 320 * 8 // ROWS + 3) * ROWS  # tiles of 16 x 8 cells, 320 threads
    small, large = (strip("Hydro_Muscl_2D", 2, n, ROWS, native.EK_FP32) for n in (ROWS, rows))
    U = pattern(small, 6)
    want = alone(small, U)
    print(f"case=pool 2x{rows}", flush=True)
    P = pool.Pool(small, 2 * rows * 32 + (1 << 20), 2)
    try:
        P.set_tile(1)
        jid = P.admit(large, np.broadcast_to(U[:, None], (4, rows // ROWS, ROWS, 2)).reshape(4, rows, 2), 2)
        P.step(2)
        got = P.download(jid)
        assert P.status(jid)[1:] == (2, True)
    finally:
        P.close()
    assert bool((got.reshape(4, -1, ROWS, 2) == want[:, None]).all())
