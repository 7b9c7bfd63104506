"""FP64 quotients and roots over the whole exponent range: the kernels share one refined
reciprocal between the divisions by one denominator, which has to give the division's own
bits also where the numerators are tiny (momenta and field components down to the smallest
denormal, in gas that is otherwise ordinary), zero, or far from 1 (other units). One and
three steps are bitwise the oracle's."""
import numpy as np
import pytest

from euler_kokkos_amd.params import make_params

import test_mhd3d_gpu
import test_mhd_gpu
import test_parity_gpu

pytestmark = pytest.mark.gpu

ID, IP, IU, IV, IW, IA, IB, IC = range(8)

# exponents of the momenta and fields: spread down to the denormals, all denormal, a shell of
# products around the underflow threshold
SPREADS = {"spread": (-1074, 0), "denormal": (-1074, -1015), "threshold": (-560, -480)}


def small(rng, shape, lo, hi):
    """+-m 2^e with e uniform in [lo, hi), one value in eight zero."""
    x = np.ldexp(rng.uniform(0.5, 1.0, shape), rng.integers(lo, hi, shape))
    return np.where(rng.random(shape) < 0.125, 0.0, np.where(rng.random(shape) < 0.5, -x, x))


def state(oracle, op, mhd, spread, seed, ordinary=0.25):
    """Density and pressure of order 1; momenta (and fields) of the given exponents, with a share
    of ordinary cells among them so that tiny and ordinary values meet at the faces."""
    rng = np.random.default_rng(seed)
    U = np.zeros(oracle.ref_shape(op))
    shape = U.shape[:-1]
    U[..., ID] = rng.uniform(0.5, 2.0, shape)
    quiet = rng.random(shape) >= ordinary
    energy = rng.uniform(0.5, 2.0, shape) / (op.gamma0 - 1.0)
    names = [IU, IV, IW][: 3 if (mhd or U.shape[-1] == 5) else 2] + ([IA, IB, IC] if mhd else [])
    for v in names:
        U[..., v] = np.where(quiet, small(rng, shape, *SPREADS[spread]), rng.uniform(-0.3, 0.3, shape))
        energy = energy + 0.5 * U[..., v] ** 2 / (U[..., ID] if v < IA else 1.0)
    U[..., IP] = np.where(quiet & (rng.random(shape) < 0.5), 2.5, energy)
    return U


def check(name, pair, steps):
    g, o = pair
    bad = int(np.count_nonzero(~((g == o) | (np.isnan(g) & np.isnan(o)))))
    print(f"case={name} steps={steps}: {bad} of {g.size} values differ", flush=True)
    assert bad == 0


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("spread", sorted(SPREADS))
@pytest.mark.parametrize("solver", ["hllc", "approx", "hll"])
def test_hydro2d(oracle, solver, spread, steps):
    ekp = make_params("Hydro_Muscl_2D", 37, 30, riemann=solver, slope_type="2", cfl="0.5", bc=(1, 2, 3, 3, 3, 3))
    U0 = state(oracle, oracle.from_ek(ekp), False, spread, 21)
    check(f"hydro2d {solver} {spread}", test_parity_gpu.run_pair(oracle, ekp, U0, steps), steps)


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("spread", sorted(SPREADS))
@pytest.mark.parametrize("solver", ["hllc", "approx"])
def test_hydro3d(oracle, solver, spread, steps):
    ekp = make_params("Hydro_Muscl_3D", 19, 17, 10, riemann=solver, slope_type="1", cfl="0.5", bc=(3, 3, 1, 2, 2, 1))
    U0 = state(oracle, oracle.from_ek(ekp), False, spread, 22)
    check(f"hydro3d {solver} {spread}", test_parity_gpu.run_pair(oracle, ekp, U0, steps), steps)


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("spread", sorted(SPREADS))
@pytest.mark.parametrize("solver", ["hlld", "hll", "llf"])
def test_mhd2d(oracle, solver, spread, steps):
    ekp = test_mhd_gpu.mparams(31, 18, riemann=solver, bc=(1, 2, 3, 3, 3, 3))
    U0 = state(oracle, oracle.from_ek(ekp), True, spread, 23)
    check(f"mhd2d {solver} {spread}", test_mhd_gpu.run_pair(oracle, ekp, U0, steps), steps)


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("spread", sorted(SPREADS))
@pytest.mark.parametrize("solver", ["hlld", "hll"])
def test_mhd3d(oracle, solver, spread, steps):
    ekp = test_mhd3d_gpu.m3(13, 9, 8, riemann=solver, bc=(3, 3, 1, 2, 2, 1))
    U0 = state(oracle, oracle.from_ek(ekp), True, spread, 24)
    check(f"mhd3d {solver} {spread}", test_mhd3d_gpu.run_pair(oracle, ekp, U0, steps), steps)


@pytest.mark.parametrize("scale", [2.0 ** -80, 2.0 ** 80])
@pytest.mark.parametrize("path", ["hydro2d", "hydro3d", "mhd2d", "mhd3d"])
def test_other_units(oracle, path, scale):
    """The same gas with density, energy and momenta in units `scale` times smaller or larger."""
    low = repr(1e-10 * min(scale, 1.0))
    if path == "hydro2d":
        ekp = make_params("Hydro_Muscl_2D", 37, 30, riemann="hllc", slope_type="2", bc=(1, 2, 3, 3, 3, 3), smallr=low)
    elif path == "hydro3d":
        ekp = make_params("Hydro_Muscl_3D", 19, 17, 10, riemann="hllc", slope_type="2", bc=(3, 3, 1, 2, 2, 1), smallr=low)
    elif path == "mhd2d":
        ekp = test_mhd_gpu.mparams(31, 18, bc=(1, 2, 3, 3, 3, 3))
    else:
        ekp = test_mhd3d_gpu.m3(13, 9, 8, bc=(3, 3, 1, 2, 2, 1))
    if ekp.mhd:
        ekp.smallr *= min(scale, 1.0)
    U0 = state(oracle, oracle.from_ek(ekp), bool(ekp.mhd), "spread", 25, ordinary=1.0)
    for v in range(U0.shape[-1]):
        U0[..., v] *= scale if v < IA else scale ** 0.5
    mod = {"mhd2d": test_mhd_gpu, "mhd3d": test_mhd3d_gpu}.get(path, test_parity_gpu)
    check(f"{path} units {scale}", mod.run_pair(oracle, ekp, U0, 3), 3)
