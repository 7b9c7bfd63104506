"""Alfven speeds |B| / sqrt(rho) where the root's mantissa is all ones and the field is a power of
two: the quotient then lies next to a rounding boundary that a reciprocal of the root which is
not the division's own lands on the wrong side of. Gas whose density is an ulp or two below a
power of four, as a background of density 1 is after a few rounded steps, with fields of one half.
FP64 is bitwise the oracle's."""
import numpy as np
import pytest

import test_mhd3d_gpu
import test_mhd_gpu

pytestmark = pytest.mark.gpu

ID, IP, IU, IV, IW, IA, IB, IC = range(8)


@pytest.mark.parametrize("rho", [1.0 - 2.0 ** -53, 1.0 - 2.0 ** -52, 4.0 - 2.0 ** -51])
@pytest.mark.parametrize("mod,ekp", [(test_mhd_gpu, lambda g: test_mhd_gpu.mparams(64, 50, gamma0=g, cfl="0.5")),
                                     (test_mhd3d_gpu, lambda g: test_mhd3d_gpu.m3(20, 18, 16, gamma0=g, cfl="0.5"))],
                         ids=["2d", "3d"])
def test_root_next_to_a_power_of_two(oracle, mod, ekp, rho):
    for gamma in ("1.666", "1.4"):
        p = ekp(gamma)
        R0 = np.zeros(oracle.ref_shape(oracle.from_ek(p)))
        rng = np.random.default_rng(7)
        R0[..., ID] = rho
        R0[..., IP] = 1.0 / (p.gamma0 - 1.0) + 0.375
        for v in (IA, IB, IC):
            R0[..., v] = np.where(rng.random(R0.shape[:-1]) < 0.5, 0.5, -0.5)
        for steps in (1, 4):
            g, o = mod.run_pair(oracle, p, R0, steps)
            print(f"case=field over root rho={rho!r} gamma={gamma} steps={steps}: {np.count_nonzero(g != o)} of {g.size} differ",
                  flush=True)
            assert np.array_equal(g, o)
