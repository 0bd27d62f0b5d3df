"""The ring march (variant 19 in FP32, 8 in FP64; variant 24: its 64 x 8 blocks) at the sizes where a
tiled march can go wrong: boxes smaller than a tile, tile edges and remainders, columns cut into chunks
of one plane and more. Every chunk depth, block shape and ghost form (filled, or read at their periodic
images) computes the same bits, and those are the oracle's.
"""
import numpy as np
import pyoracle
import pytest

from astaroth_amd import abi
from astaroth_amd.api import HostMesh, Library, real_params_double
from astaroth_amd.initial import mhd_fields

pytestmark = pytest.mark.gpu

DIMS = [(3, 3, 3), (16, 16, 3), (17, 15, 4), (33, 18, 5), (64, 8, 3), (65, 9, 7), (15, 33, 10)]
DT = 1e-3


@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "%dx%dx%d" % d)
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_ring_march_forms(double, dims):
    nx, ny, nz = dims
    lib = Library(double)
    info = lib.config(n=nx, ny=ny, nz=nz)
    fields = mhd_fields(nx, ny, nz, np.float64, config_id=6)
    variants = [(8, 16, 16)] if double else [(19, 16, 16), (24, 64, 8)]
    results = {}
    for variant in variants:
        for depth in (0, 1, 2, 3, 5):
            for images in (0, 1):
                if images and (variant[0] == 24 or min(dims) < abi.NGHOST):
                    continue
                with lib.device_create(0, info, autotune=False) as dev:
                    dev.set_kernel_config(*variant, depth)
                    if variant[0] != 24:
                        assert lib.dll.acDeviceSetReadPeriodicImages(dev.handle, images) == abi.AC_SUCCESS
                    mesh = HostMesh(lib, info, [f.astype(lib.dtype) for f in fields])
                    dev.load_mesh(mesh)
                    for _ in range(2):
                        dev.integrate_step(DT)
                    out = mesh.copy()
                    dev.store_mesh(out)
                results[variant + (depth, images)] = [out.interior(q) for q in range(8)]
    first = next(iter(results.values()))
    for key, got in results.items():
        for q in range(8):
            assert np.array_equal(got[q], first[q]), (dims, key, q)
    ref = [f.astype(lib.dtype).astype(np.float64) for f in fields]
    pyoracle.integrate_steps_gpu_form(ref, real_params_double(info), DT, 2)
    # 6 substeps, each of which rounds a value once and adds an increment whose sums of about 20 terms
    # carry a few roundings more: 4 ulps of the field's largest value per substep
    eps = np.finfo(lib.dtype).eps
    for q in range(8):
        want = ref[q][3:-3, 3:-3, 3:-3]
        scale = max(np.abs(want).max(), np.abs(fields[q]).max())
        assert np.abs(first[q].astype(np.float64) - want).max() <= 24 * eps * scale, (dims, q)


@pytest.mark.parametrize("dims", [(3, 4, 5), (17, 15, 4), (65, 9, 7)], ids=lambda d: "%dx%dx%d" % d)
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_ring_march_compensated(double, dims):
    """The compensated build: the same bits for every chunk depth, and the oracle's values (tolerance
    as above; the compensation only takes rounding away)."""
    nx, ny, nz = dims
    lib = Library(double)
    info = lib.config(n=nx, ny=ny, nz=nz)
    fields = mhd_fields(nx, ny, nz, np.float64, config_id=6)
    results = []
    for depth in (0, 1, 3):
        with lib.device_create(0, info, autotune=False) as dev:
            dev.set_kernel_config(8 if double else 19, 16, 16, depth)
            dev.set_compensated_integration(True)
            mesh = HostMesh(lib, info, [f.astype(lib.dtype) for f in fields])
            dev.load_mesh(mesh)
            for _ in range(2):
                dev.integrate_step(DT)
            out = mesh.copy()
            dev.store_mesh(out)
        results.append([out.interior(q) for q in range(8)])
    ref = [f.astype(lib.dtype).astype(np.float64) for f in fields]
    pyoracle.integrate_steps_gpu_form(ref, real_params_double(info), DT, 2)
    eps = np.finfo(lib.dtype).eps
    for q in range(8):
        want = ref[q][3:-3, 3:-3, 3:-3]
        scale = max(np.abs(want).max(), np.abs(fields[q]).max())
        assert np.array_equal(results[1][q], results[0][q]) and np.array_equal(results[2][q], results[0][q]), (dims, q)
        assert np.abs(results[0][q].astype(np.float64) - want).max() <= 24 * eps * scale, (dims, q)


@pytest.mark.parametrize("dims", [((64, 8, 5), (128, 9, 7), (32, 16, 40), (33, 17, 12), (3, 4, 5)), ((48, 48, 9), (17, 15, 4))],
                         ids=["wide", "narrow"])
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_ring_march_batched(double, dims):
    """Boxes at the edges of the batched launch's tile shapes: the same bits as box after box (the
    march writes out every multiply-add, so a cell's value depends on no tile or z range)."""
    lib = Library(double)
    infos = [lib.config(n=nx, ny=ny, nz=nz, AC_nu_visc=1e-3 * (b + 1)) for b, (nx, ny, nz) in enumerate(dims)]
    out = {}
    for mode, depth in (("looped", None), ("batched", None), ("batched", 0), ("graph", 3)):
        with lib.ensemble_create(infos) as ens:
            if depth is not None:
                ens.set_kernel_config(16, 16, depth)
            for b, d in enumerate(dims):
                ens.load_mesh(b, HostMesh(lib, infos[b], [f.astype(lib.dtype) for f in mhd_fields(*d, np.float64, config_id=4)]))
            for _ in range(2):
                ens.integrate_step(DT, mode=mode)
            for b in range(len(dims)):
                mesh = HostMesh(lib, infos[b])
                ens.store_mesh(b, mesh)
                out.setdefault(b, []).append([mesh.interior(q).copy() for q in range(8)])
    for b, d in enumerate(dims):
        for q in range(8):
            assert np.abs(out[b][0][q]).max() > 0, (d, q)
            for other in out[b][1:]:
                assert np.array_equal(other[q], out[b][0][q]), (d, q)


@pytest.mark.parametrize("dims", [(352, 96, 63), (350, 90, 70), (450, 49, 97)], ids=lambda d: "%dx%dx%d" % d)
def test_ring_march_tiles(dims):
    """FP32 regions of 2^21 cells or more, whose tile goes by what covers them: the same bits as in
    64 x 8 tiles, with and without compensation."""
    nx, ny, nz = dims
    assert nx * ny * nz >= 2**21
    lib = Library(False)
    info = lib.config(n=nx, ny=ny, nz=nz)
    for compensated in (False, True):
        out = []
        for config in ((19, 16, 16, 0), (19, 16, 16, 11), (24, 64, 8, 0)):
            with lib.device_create(0, info, autotune=False) as dev:
                dev.set_kernel_config(*config)
                dev.set_compensated_integration(compensated)
                for q in range(8):
                    dev.randomize_uniform(q, -1e-3, 1e-3, 7 * q + 1)
                dev.integrate_step(DT)
                mesh = HostMesh(lib, info)
                dev.store_mesh(mesh)
                out.append([mesh.interior(q).copy() for q in range(8)])
        for q in range(8):
            assert np.abs(out[0][q]).max() > 0
            assert np.array_equal(out[1][q], out[0][q]) and np.array_equal(out[2][q], out[0][q]), (dims, compensated, q)


@pytest.mark.parametrize("compensated", [False, True], ids=["plain", "compensated"])
@pytest.mark.parametrize("dims", [(150, 33, 60), (145, 35, 61)], ids=lambda d: "%dx%dx%d" % d)
def test_ring_march_fp64_flat_tiles(dims, compensated):
    """FP64 regions that 32 x 8 tiles cover at less cost than 16 x 16 ones, against the oracle
    (tolerance as above)."""
    nx, ny, nz = dims
    lib = Library(True)
    info = lib.config(n=nx, ny=ny, nz=nz)
    fields = mhd_fields(nx, ny, nz, np.float64, config_id=6)
    ref = [f.copy() for f in fields]
    pyoracle.integrate_steps_gpu_form(ref, real_params_double(info), DT, 2)
    for depth in (0, 2):
        with lib.device_create(0, info, autotune=False) as dev:
            dev.set_kernel_config(8, 16, 16, depth)
            dev.set_compensated_integration(compensated)
            mesh = HostMesh(lib, info, [f.copy() for f in fields])
            dev.load_mesh(mesh)
            for _ in range(2):
                dev.integrate_step(DT)
            out = mesh.copy()
            dev.store_mesh(out)
        for q in range(8):
            want = ref[q][3:-3, 3:-3, 3:-3]
            scale = max(np.abs(want).max(), np.abs(fields[q]).max())
            assert np.abs(out.interior(q) - want).max() <= 24 * np.finfo(np.float64).eps * scale, (dims, depth, q)
