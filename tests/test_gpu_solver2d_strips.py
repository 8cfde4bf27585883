"""The 2D solver's pipelined columns at the edges of strips (64 columns),
passes (8 strips), batches (8 steps) and grids longer than a pass is wide:
fields equal the oracle's bit for bit."""
from ctypes import byref, c_int

import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_helpers import lib, _d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,nx", [
    (3, 3), (9, 65), (10, 66), (8, 129), (700, 514), (1200, 515), (5, 577),
    (63, 1025), (200, 1026), (1500, 1090), (31, 1601), (2000, 70),
])
def test_strips_match_oracle(nz, nx):
    rng = np.random.default_rng(nz * 7 + nx)
    dz, dx = 10.0, 12.0
    vel = 1000.0 * rng.uniform(1.0, 5.0, (nz - 1) * (nx - 1))
    slow = orc.cell_slowness(vel, nz, nx)
    grid = (nz, nx, 1, dz, dx, 1.0, 0.0, 0.0, 0.0)
    L, ierr = lib(), c_int(1)
    L.fteik_solver2d_initialize(nz, nx, 0.0, 0.0, dz, dx, 2, 3.0, 0.0, 0,
                                byref(ierr))
    assert ierr.value == 0
    L.fteik_solver2d_setCellVelocityModel64f(vel.size, 0, _d(vel),
                                             byref(ierr))
    assert ierr.value == 0
    # near both ends of the profile and in the middle, one at a time and
    # together (the last one's field is kept)
    zs = np.array([0.2, 0.7 * (nz - 2.2), 0.4 * nz * (nz > 4)]) * dz
    xs = np.array([0.3, nx - 2.3, 0.5 * nx * (nx > 4)]) * dx
    print("case: 2D strips", nz, nx, flush=True)
    for k in (range(3), [0], [1]):
        z, x = zs[list(k)].copy(), xs[list(k)].copy()
        L.fteik_solver2d_setSources64f(z.size, _d(z), _d(x), byref(ierr))
        assert ierr.value == 0
        if z.size > 1:
            L.fteik_solver2d_solveLSM(byref(ierr))
        else:
            L.fteik_solver2d_solveSourceLSM(1, byref(ierr))
        assert ierr.value == 0
        tt = np.zeros(nz * nx)
        L.fteik_solver2d_getTravelTimeField64f(tt.size, 0, _d(tt),
                                               byref(ierr))
        assert ierr.value == 0
        src = orc.source_locate(grid, z[-1], x[-1], slow=slow, is3d=False)
        ref = orc.solve2d(slow, nz, nx, dz, dx, src, 2, 3.0)
        np.testing.assert_array_equal(tt, ref)
    L.fteik_solver2d_free()
