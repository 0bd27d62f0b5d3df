"""The FP32 ring march chooses its tile by rounds of resident blocks as well as by covered cells: a box
whose 16 x 16 blocks fill one round while the wide tiles just miss it, with a second, nearly empty one."""
import pytest

from astaroth_amd import abi
from astaroth_amd.api import Library

pytestmark = pytest.mark.gpu


def test_tile_goes_by_rounds_of_blocks():
    lib = Library(False)
    nx, ny, nz = 400, 80, 100  # 125 x 4 blocks of 16 x 16 on 512 slots; 65 x 4 of 32 x 16, 70 x 4 of 64 x 8 on 256
    with lib.device_create(0, lib.config(n=nx, ny=ny, nz=nz), autotune=False) as dev:
        for q in range(8):
            dev.randomize_uniform(q, -1e-3, 1e-3, q + 1)
        dev.periodic_boundconds()
        c = dev.kernel_config()
        assert (c.variant, c.tile_x, c.tile_y) == (19, 16, 16)
        own, wide = [], []
        for _ in range(5):
            own.append(dev.time_kernel_config(c, iters=50))
            wide.append(min(dev.time_kernel_config(abi.KernelConfig(24, 64, 8, depth), iters=50) for depth in (15, 25)))
    # 85 us against 104 (64 x 8 at its best depth) and 106 (32 x 16)
    assert min(own) < 0.92 * min(wide), (own, wide)
