"""The z-chunk length of 3D steps: the shortest estimate among the lengths that spread the planes
evenly, chosen in a time that does not grow with the number of planes (3D MHD chooses it at every
launch)."""
import random
import time

import pytest

from euler_kokkos_amd import native

import test_mhd3d_gpu


def chosen(tiles, n, slots, a, b, lo, hi):
    """The rule, over every number of chunks."""
    best, least = min(n, hi), 1e300
    for nch in range(1, n + 1):
        cz = -(-n // nch)
        if cz > hi:
            continue
        if cz < lo:
            break
        m = tiles * -(-n // cz)
        full, rest = divmod(m, slots)
        t = (cz + a) * (full + ((b + (1.0 - b) * rest / slots) if rest else 0.0))
        if t < least:
            best, least = cz, t
    return best


@pytest.mark.parametrize("prec", [native.EK_FP64, native.EK_FP32])
def test_same_choice(prec):
    rng = random.Random(3)
    for _ in range(400):
        nx, ny, nz = rng.randint(3, 200), rng.randint(3, 200), rng.choice([rng.randint(3, 60), rng.randint(3, 900)])
        walls = rng.random() < 0.5
        p = test_mhd3d_gpu.m3(nx, ny, nz, bc=(1 if walls else 3,) * 6, precision=prec)
        faces = [n + walls for n in (nx, ny, nz)]
        tiles = -(-faces[0] // 16) * -(-faces[1] // 4)
        want = (chosen(tiles, faces[2], 768, 0.3, 0.2, 1, 40) if prec == native.EK_FP64 else
                chosen(tiles, faces[2], 1536, 0.5, 0.1, 1, 40))
        assert native.z_chunk(p)[0] == want


def test_long_columns_cost_no_more():
    p = test_mhd3d_gpu.m3(3, 3, 4000000)
    start = time.perf_counter()
    for _ in range(200):
        native.z_chunk(p)
    assert time.perf_counter() - start < 1.0  # 5 ms a call (going through 4e6 numbers of chunks takes 40)
