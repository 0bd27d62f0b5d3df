"""Every tile of the ring march computes the bits of every other, plain and compensated, on boxes smaller
than a tile, at tile edges and with remainders: variant 24 names the tile, and boxes below 2^21 cells run
variant 19 in 16 x 16 tiles (variant 8 in FP64 in 16 x 16 ones wherever 32 x 8 do not take fewer rounds of
blocks, as in all of these in whole columns)."""
import numpy as np
import pytest

from astaroth_amd.api import HostMesh, Library
from astaroth_amd.initial import mhd_fields

pytestmark = pytest.mark.gpu

DIMS = [(3, 3, 3), (16, 16, 3), (17, 15, 4), (33, 18, 5), (64, 8, 3), (65, 9, 7), (32, 16, 6), (15, 33, 10), (130, 35, 9)]
DT = 1e-3


@pytest.mark.parametrize("compensated", [False, True], ids=["plain", "compensated"])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "%dx%dx%d" % d)
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_tiles_agree_bit_for_bit(double, dims, compensated):
    nx, ny, nz = dims
    lib = Library(double)
    info = lib.config(n=nx, ny=ny, nz=nz)
    fields = [f.astype(lib.dtype) for f in mhd_fields(nx, ny, nz, np.float64, config_id=6)]
    configs = [(8, 16, 16, 0), (24, 32, 8, 0), (24, 32, 8, 2)] if double else \
        [(19, 16, 16, 0), (24, 64, 8, 0), (24, 32, 16, 0), (24, 64, 8, 2), (24, 32, 16, 3)]
    results = []
    for config in configs:
        with lib.device_create(0, info, autotune=False) as dev:
            dev.set_kernel_config(*config)
            dev.set_compensated_integration(compensated)
            dev.load_mesh(HostMesh(lib, info, fields))
            for _ in range(2):
                dev.periodic_boundconds()
                for substep in range(3):  # (with filled ghosts in every configuration)
                    assert dev.integrate_substep(substep, dt=DT) == 0
                    dev.swap_buffers()
                    dev.periodic_boundconds()
            out = HostMesh(lib, info)
            dev.store_mesh(out)
        results.append(out)
    for config, out in zip(configs[1:], results[1:]):
        for q in range(8):
            assert np.any(results[0].interior(q) != fields[q][3:-3, 3:-3, 3:-3])
            assert np.array_equal(out.interior(q), results[0].interior(q)), (config, q)
