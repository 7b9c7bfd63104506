"""The range of values over which the FP64 step is the reference's bit for bit: densities and
pressures (and squared fields) from 1e-60 to 1e60, in every combination, and cells of very different
ones side by side; every solver, one and two steps bitwise the oracle's. And FP32 in gas so cold and
thin that products of its slopes fall below the smallest FP32 number: within three steps' rounding
of FP64 (each step rounds a few hundred FP32 operations per cell: 1e-5 of each variable's norm)."""
import numpy as np
import pytest

from euler_kokkos_amd import native
from euler_kokkos_amd.params import make_params

import test_mhd3d_gpu
import test_mhd_gpu
import test_min_grids_gpu
import test_parity_gpu

pytestmark = pytest.mark.gpu

ID, IP, IU, IV, IW, IA, IB, IC = range(8)
PATHS = {"hydro2d": ["hllc", "approx", "llf", "hll"], "hydro3d": ["hllc", "approx", "llf"],
         "mhd2d": ["hlld", "hll", "llf"], "mhd3d": ["hlld", "hll", "llf"]}
CORNERS = [(1e-60, 1e-60), (1e-60, 1e60), (1e60, 1e-60), (1e60, 1e60), (1e60, 1.0), (1.0, 1e60)]


def params(path, riemann):
    slope = "1" if riemann == "llf" else "2"
    if path == "hydro2d":
        return make_params("Hydro_Muscl_2D", 37, 30, riemann=riemann, slope_type=slope, bc=(1, 2, 3, 3, 3, 3))
    if path == "hydro3d":
        return make_params("Hydro_Muscl_3D", 19, 17, 10, riemann=riemann, slope_type=slope, bc=(3, 3, 1, 2, 2, 1))
    if path == "mhd2d":
        return test_mhd_gpu.mparams(31, 18, riemann=riemann, slope_type=slope, bc=(1, 2, 3, 3, 3, 3))
    return test_mhd3d_gpu.m3(13, 9, 8, riemann=riemann, slope_type=slope, bc=(3, 3, 1, 2, 2, 1))


def floors(ekp, rho, p):
    """Floors far below densities `rho`, pressures `p` (smallp is smallc^2 / gamma, which floors p / rho and,
    in the 3D MHD trace, p) and their sound speeds."""
    ekp.smallr, ekp.smallc = 1e-10 * rho, 1e-10 * min(p / rho, p) ** 0.5
    ekp.smallp = ekp.smallc * ekp.smallc / ekp.gamma0
    ekp.smallpp = ekp.smallr * ekp.smallp


def check(oracle, path, ekp, U0, steps, name):
    mod = {"mhd2d": test_mhd_gpu, "mhd3d": test_mhd3d_gpu}.get(path, test_parity_gpu)
    g, o = mod.run_pair(oracle, ekp, U0, steps)
    bad = int(np.count_nonzero(~((g == o) | (np.isnan(g) & np.isnan(o)))))
    print(f"case={path} {name} steps={steps}: {bad} of {g.size} differ", flush=True)
    assert bad == 0


@pytest.mark.parametrize("path,riemann", [(a, r) for a in PATHS for r in PATHS[a]])
def test_corners(oracle, path, riemann):
    for rho, p in CORNERS:
        ekp = params(path, riemann)
        floors(ekp, rho, p)
        U0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), bool(ekp.mhd), 51)
        scale = {ID: rho, IP: p, IU: (rho * p) ** 0.5, IV: (rho * p) ** 0.5, IW: (rho * p) ** 0.5}
        for v in range(U0.shape[-1]):
            U0[..., v] *= scale.get(v, p ** 0.5)
        for steps in (1, 2):
            check(oracle, path, ekp, U0, steps, f"{riemann} rho {rho:g} p {p:g}")


@pytest.mark.parametrize("path,riemann", [(a, r) for a in PATHS for r in PATHS[a]])
def test_side_by_side(oracle, path, riemann):
    ekp = params(path, riemann)
    floors(ekp, 1e-20, 1e-20)
    rng = np.random.default_rng(52)
    U0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), bool(ekp.mhd), 53)
    shape = U0.shape[:-1]
    rho, p = (10.0 ** rng.uniform(-20.0, 20.0, shape) for _ in range(2))
    for v in range(U0.shape[-1]):
        U0[..., v] *= rho if v == ID else p if v == IP else np.sqrt(rho * p) if v < IA else np.sqrt(p)
    check(oracle, path, ekp, U0, 1, f"{riemann} side by side")


@pytest.mark.parametrize("path,riemann", [("hydro2d", "hllc"), ("hydro2d", "llf"), ("hydro2d", "hll"), ("hydro3d", "hllc"),
                                          ("hydro3d", "llf")])
def test_fp32_slopes_below_the_smallest_product(oracle, path, riemann):
    ekp = params(path, riemann)
    ekp.precision = native.EK_FP64
    U0 = test_min_grids_gpu.random_state(oracle, oracle.from_ek(ekp), False, 54)
    for v in range(U0.shape[-1]):  # densities 1e-6, pressures 1e-18, speeds 1e-6
        U0[..., v] *= {ID: 1e-6, IP: 1e-18}.get(v, 1e-12)
    out = []
    for prec in (native.EK_FP64, native.EK_FP32):
        ekp.precision = prec
        ctx = native.Context(ekp)
        try:
            ctx.upload(U0.astype(np.float32).astype(np.float64))
            ctx.run(3, 3, 1e30)
            out.append(ctx.download(native.EK_LAYOUT_SOA))
        finally:
            ctx.close()
    for v in range(ekp.nbvar):
        off = np.linalg.norm(out[1][v] - out[0][v]) / np.linalg.norm(out[0][v])
        print(f"case={path} {riemann} variable {v}: off {off:.2e}", flush=True)
        assert off < 1e-5
