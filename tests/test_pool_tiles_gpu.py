"""Job pool work lists at their edges: one item, fewer items than XCDs, a list whose length is
no multiple of 8, ragged tiles, and more jobs than have CFL words of their own (the job slots
past 2048 use one word). Every checked job is bitwise its single-grid run."""
import numpy as np
import pytest

from euler_kokkos_amd import native, pool, problems
from euler_kokkos_amd.params import make_params

pytestmark = pytest.mark.gpu


def job(solver, n, k, prec):
    shape = (n, n + k % 3) + ((n - 1,) if solver.endswith("3D") else ())
    p = make_params(solver, *shape, riemann="hllc", slope_type="2", cfl="0.5", bc=(1, 2, 3, 3, 2, 1), precision=prec)
    return p, problems.blast(p, radius="0.25", center_x=repr(0.3 + 0.05 * (k % 7)), center_y="0.55", center_z="0.5")


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
@pytest.mark.parametrize("solver,edges,count", [("Hydro_Muscl_2D", (8,), 1), ("Hydro_Muscl_2D", (15, 17, 40), 5),
                                                ("Hydro_Muscl_3D", (7, 18, 33), 4), ("Hydro_Muscl_2D", (4, 9), 2051)])
def test_jobs_equal_single_runs(solver, edges, count, prec):
    jobs = [job(solver, edges[k % len(edges)], k, prec) for k in range(count)]
    P = pool.Pool(jobs[0][0], 256 << 20, count)
    try:
        ids = [P.admit(p, U, 9) for p, U in jobs]
        P.step(9)
        for k in sorted({0, 1, count // 2, count - 3, count - 1} & set(range(count))):
            p, U = jobs[k]
            ctx = native.Context(p)
            try:
                ctx.upload(U, native.EK_LAYOUT_SOA)
                t, it, _ = ctx.run(9, 9, 1e30)
                assert P.status(ids[k])[:2] == (t, it)
                assert np.array_equal(P.download(ids[k]), ctx.download(native.EK_LAYOUT_SOA))
            finally:
                ctx.close()
    finally:
        P.close()
