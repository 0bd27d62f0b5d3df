"""Rounding error of the default solve against 80-bit arithmetic: no larger, in any field, than that of
the lean z-march (variant 3), whose sums it takes in another order. Noise on a fine grid, where the
viscous terms are large beside the field (near the diffusive limit of the time step), on a coarse one,
and on one between them at uniform entropy, where the pressure drives the velocity.
"""
import math

import numpy as np
import pyoracle
import pytest

from astaroth_amd import abi
from astaroth_amd.api import HostMesh, Library, real_params_double

pytestmark = pytest.mark.gpu

N, DT = 40, 1e-3
GROUPS = [[abi.VTX[k] for k in names] for names in (
    ("VTXBUF_LNRHO",), ("VTXBUF_UUX", "VTXBUF_UUY", "VTXBUF_UUZ"), ("VTXBUF_AX", "VTXBUF_AY", "VTXBUF_AZ"),
    ("VTXBUF_ENTROPY",))]


@pytest.mark.parametrize("cells,steps,entropy", [(512, 2, 1e-5), (64, 2, 1e-5), (192, 3, 0.0)],
                         ids=["fine", "coarse", "pressure"])
@pytest.mark.parametrize("double", [False, True], ids=["fp32", "fp64"])
def test_default_solve_error(double, cells, steps, entropy):
    lib = Library(double)
    h = 2 * math.pi / cells
    amplitude = [1e-2] + [1e-3] * 6 + [entropy]
    info = lib.config(n=N, AC_dsx=h, AC_dsy=h, AC_dsz=h)
    default = (8, 16, 16, 0) if double else (19, 16, 16, 0)
    error = {default: np.zeros(8), (3, 16, 16, 0): np.zeros(8)}
    for seed in range(3):
        rng = np.random.default_rng(seed)
        fields = [np.pad(rng.uniform(-a, a, (N, N, N)), 3, mode="wrap").astype(lib.dtype) for a in amplitude]
        ref = [f.astype(np.longdouble) for f in fields]
        pyoracle.integrate_steps_gpu_form(ref, real_params_double(info), float(lib.real(DT).value), steps)
        for config in error:
            with lib.device_create(0, info, autotune=False) as dev:
                dev.set_kernel_config(*config)
                dev.load_mesh(HostMesh(lib, info, fields))
                for _ in range(steps):
                    dev.integrate_step(DT)
                out = HostMesh(lib, info)
                dev.store_mesh(out)
            for q in range(8):
                d = (out.interior(q).astype(np.longdouble) - ref[q][3:-3, 3:-3, 3:-3]).astype(np.float64)
                error[config][q] += np.sum(d * d)
    # 192000 values per field: a root mean square is known to 0.2 %, and two errors that are equal in
    # truth (both are mostly the last rounding of the result) may fall either way by as much
    for group in GROUPS:
        mine, lean = (math.sqrt(sum(error[c][q] for q in group)) for c in (default, (3, 16, 16, 0)))
        assert mine <= 1.005 * lean, (group, mine, lean)
