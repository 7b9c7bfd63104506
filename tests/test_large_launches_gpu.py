"""Steps of 2D grids whose tiles have 2^32 threads and more between them, the most that one launch
takes: strips two or three cells wide, so that a tile holds few cells and the state stays small
(7 to 33 GB). The state repeats every 64 rows, and so does the result: it is bitwise the step of
the 64 rows alone, periodic."""
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


@pytest.mark.parametrize("solver,nx,tile_rows,threads", [("Hydro_Muscl_2D", 2, 16, 512), ("MHD_Muscl_2D", 3, 10, 256)])
def test_single_grid(solver, nx, tile_rows, threads):
    import torch

    rows = (2 ** 32 // threads * tile_rows // ROWS + 3) * ROWS
    small, large = (strip(solver, nx, n, ROWS, native.EK_FP32) for n in (ROWS, rows))
    U = pattern(small, 5)
    want = torch.from_numpy(alone(small, U)).cuda().float()
    a = torch.from_numpy(U).cuda().float()[:, None].expand(-1, rows // ROWS, -1, -1).contiguous()
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    print(f"case={solver} {nx}x{rows} {2 * a.nbytes / 1e9:.1f} GB", flush=True)
    in_b = native.run_noalloc(large, a.data_ptr(), b.data_ptr(), 2, 2, 1e30)[3]
    for v in range(small.nbvar):
        assert bool(((b if in_b else a)[v] == want[v]).all())


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
