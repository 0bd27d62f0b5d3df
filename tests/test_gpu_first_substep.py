"""Substep 0 has no previous stage: its update is u + beta dt F of the current value alone. A density
whose logarithm is infinite (an empty cell, -inf) stays so: its rate does not contain the cell's own
lnrho, while a term (u - u) of a stage that is not there would turn it into NaN.
"""
import numpy as np
import pytest

from astaroth_amd import abi
from astaroth_amd.api import HostMesh, Library
from astaroth_amd.initial import mhd_fields

pytestmark = pytest.mark.gpu

DT = 1e-3
# smaller than a tile, tile remainders, and regions that take the other tiles of either precision
DIMS = [(12, 7, 5), (33, 18, 20), (350, 90, 70), (150, 33, 60)]


@pytest.mark.parametrize("form", ["filled", "images", "compensated"])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "%dx%dx%d" % d)
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_first_substep_keeps_infinite_density(double, dims, form):
    nx, ny, nz = dims
    lib = Library(double)
    info = lib.config(n=nx, ny=ny, nz=nz)
    fields = [f.astype(lib.dtype) for f in mhd_fields(nx, ny, nz, np.float64, config_id=6)]
    lnrho = fields[abi.VTX["VTXBUF_LNRHO"]]
    cells = [((3, 3, 3), -np.inf), ((nz + 2, ny + 2, nx + 2), np.inf)]  # the first and the last
    for cell, value in cells:
        lnrho[cell] = value
    with lib.device_create(0, info, autotune=False) as dev:
        dev.set_compensated_integration(form == "compensated")
        dev.load_mesh(HostMesh(lib, info, fields))
        if form == "images":
            assert lib.dll.acDeviceSetReadPeriodicImages(dev.handle, 1) == abi.AC_SUCCESS
            assert lib.dll.acDeviceIntegrateSubstepPeriodic(dev.handle, abi.STREAM_DEFAULT, 0, DT) == abi.AC_SUCCESS
        else:
            assert dev.integrate_substep(0, dt=DT) == abi.AC_SUCCESS
        dev.swap_buffers()
        out = HostMesh(lib, info)
        dev.store_mesh(out)
    for cell, value in cells:
        assert out.fields[abi.VTX["VTXBUF_LNRHO"]][cell] == value, (cell, value)
