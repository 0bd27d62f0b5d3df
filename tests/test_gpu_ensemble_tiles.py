"""The ensemble's tuner chooses among all tile shapes of the batched solve: thin boxes run in the tiles
that they fill (in 16 x 16 ones their launches take 1.2 to 3 times as long), with the bits of any other
shape."""
import numpy as np
import pytest

from astaroth_amd.api import HostMesh, Library

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,tile", [((32, 4, 64), (32, 4)), ((64, 4, 32), (32, 4)), ((16, 8, 64), (16, 8)),
                                       ((64, 64, 64), (16, 16))],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_tuned_tile_fits_the_boxes(double, dims, tile):
    lib = Library(double)
    boxes = 32 if dims == (64, 64, 64) else 1024
    infos = [lib.config(n=dims[0], ny=dims[1], nz=dims[2])] * boxes
    out = []
    for tuned in (True, False):
        with lib.ensemble_create(infos, autotune=tuned) as ens:
            c = ens.kernel_config()
            assert (c.tile_x, c.tile_y) == (tile if tuned else (16, 16))
            for b in (0, boxes - 1):
                for q in range(8):
                    ens.randomize_uniform(b, q, -1e-3, 1e-3, 100 * b + q)
            ens.periodic_boundconds()
            ens.integrate_step(1e-3)
            for b in (0, boxes - 1):
                mesh = HostMesh(lib, infos[b])
                ens.store_mesh(b, mesh)
                out.append([f.copy() for f in mesh.fields])
    for got, want in zip(out[:2], out[2:]):
        for q in range(8):
            assert np.abs(want[q]).max() > 0
            assert np.array_equal(got[q], want[q]), q
