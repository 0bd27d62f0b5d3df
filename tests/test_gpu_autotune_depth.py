"""The tuner and the default configuration: it is timed at its own z-depth beside the tiles and cuts that the
tuner tries, and another one replaces it only where that is faster, not where it is the same launch by
another name."""
import pytest

from astaroth_amd import abi
from astaroth_amd.api import Library

pytestmark = pytest.mark.gpu


def test_tuned_configuration_is_not_slower_than_the_default():
    lib = Library(True)
    # two rows: no step reads images, 16 x 16 tiles are left out of the sweep as too tall, and the default
    # cuts its columns in 32, which none of the tuner's depths does
    info = lib.config(n=256, ny=2, nz=1024)
    with lib.device_create(0, info, autotune=False) as dev:
        for q in range(8):
            dev.randomize_uniform(q, -1e-3, 1e-3, q + 1)
        dev.periodic_boundconds()
        default = dev.kernel_config()
        dev.autotune()
        tuned = dev.kernel_config()
        times = {True: [], False: []}
        for _ in range(5):
            times[True].append(dev.time_kernel_config(tuned, iters=20))
            times[False].append(dev.time_kernel_config(default, iters=20))
    # 96 us for the default, 184 for the best of the others
    assert min(times[True]) < 1.2 * min(times[False]), (times, tuned.variant, tuned.z_depth)


@pytest.mark.parametrize("n", [256, 512])
def test_tuner_keeps_the_default_over_the_same_launch(n):
    lib = Library(False)
    # variant 24 in 64 x 8 tiles is the default's own launch at these sizes, but has no image-reading form
    with lib.device_create(0, lib.config(n=n), autotune=False) as dev:
        for q in range(8):
            dev.randomize_uniform(q, -1e-3, 1e-3, q + 1)
        dev.periodic_boundconds()
        dev.autotune()
        c = dev.kernel_config()
        assert (c.variant, c.tile_x, c.tile_y) == (19, 16, 16)
        assert lib.dll.acDeviceSetReadPeriodicImages(dev.handle, 1) == abi.AC_SUCCESS
