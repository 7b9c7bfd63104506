"""The tiles and z-chunk lengths that grids named by GPU tests are launched with: a new fit of the
launch estimates would otherwise leave those tests with other lengths than they are there for."""
import pytest

from euler_kokkos_amd import native
from euler_kokkos_amd.params import make_params

import test_marches_gpu as marches
import test_mhd3d_gpu
import test_z_chunks_gpu


@pytest.mark.parametrize("shape,fp64,fp32", marches.TURNED)
def test_turned(shape, fp64, fp32):
    assert native.z_chunk(marches.hydro(shape, "hllc", native.EK_FP64)) == fp64
    got = native.z_chunk(marches.hydro(shape, "hllc", native.EK_FP32))
    assert got == fp32 if fp32 else got[1:] == (16, 8)
    assert shape[0] % 8 and shape[1] % 16


@pytest.mark.parametrize("shape,bc,fp64,fp32", marches.MHD)
def test_mhd(shape, bc, fp64, fp32):
    for prec, planes in ((native.EK_FP64, fp64), (native.EK_FP32, fp32)):
        assert native.z_chunk(test_mhd3d_gpu.m3(*shape, bc=bc, precision=prec)) == (planes, 16, 4)
    faces = shape[2] + (bc[4:] != (3, 3))
    assert fp64 >= 3 and faces % fp64


def chunk_cases():
    """The grids and lengths of test_z_chunks_gpu's own parameters."""
    marks = [m for m in test_z_chunks_gpu.test_chunk_lengths.pytestmark if m.name == "parametrize"]
    return next(m.args[1] for m in marks if m.args[0].startswith("shape"))


@pytest.mark.parametrize("shape,cz64,cz32", chunk_cases())
def test_chunk_lengths(shape, cz64, cz32):
    for prec, planes in ((native.EK_FP64, cz64), (native.EK_FP32, cz32)):
        ekp = make_params("Hydro_Muscl_3D", *shape, riemann="hllc", slope_type="2", cfl="0.5", bc=(3, 3, 1, 2, 2, 1),
                          precision=prec)
        assert native.z_chunk(ekp)[0] == planes


def test_hook_refuses_what_has_no_z_chunks():
    with pytest.raises(native.EkError, match="dim"):
        native.z_chunk(make_params("Hydro_Muscl_2D", 32, 32, riemann="hllc", slope_type="2"))
    with pytest.raises(native.EkError, match="slope_type"):
        native.z_chunk(make_params("Hydro_Muscl_3D", 32, 32, 32, riemann="hllc", slope_type="1.5"))
