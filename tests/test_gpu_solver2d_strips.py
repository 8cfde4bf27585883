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


@pytest.mark.parametrize("nz,nx", [(20, 600), (102, 520), (103, 520)])
def test_many_sources_on_wide_grids(nz, nx):
    """More sources than CUs on both sides of the line between the schedules:
    receiver times of every source equal the level schedule's, the last
    source's field the oracle's."""
    rng = np.random.default_rng(nz)
    dz, dx, nsrc, nrec = 10.0, 11.0, 260, 7
    vel = 1000.0 * rng.uniform(1.0, 5.0, (nz - 1) * (nx - 1))
    zs = rng.uniform(0, (nz - 2.1) * dz, nsrc)
    xs = rng.uniform(0, (nx - 2.1) * dx, nsrc)
    zr = rng.uniform(0, (nz - 1) * dz, nrec)
    xr = rng.uniform(0, (nx - 1) * dx, nrec)
    L, ierr = lib(), c_int(1)
    print("case: 2D many sources", nz, nx, flush=True)
    L.fteik_solver2d_initialize(nz, nx, 0.0, 0.0, dz, dx, 1, 3.0, 0.0, 0,
                                byref(ierr))
    assert ierr.value == 0
    L.fteik_solver2d_setCellVelocityModel64f(vel.size, 0, _d(vel),
                                             byref(ierr))
    L.fteik_solver2d_setReceivers64f(nrec, _d(zr), _d(xr), byref(ierr))
    assert ierr.value == 0
    L.fteik_solver2d_setSources64f(nsrc, _d(zs), _d(xs), byref(ierr))
    assert ierr.value == 0
    got = []
    for schedule in (0, 1):
        L.fteik_solver2d_setSchedule(schedule, byref(ierr))
        L.fteik_solver2d_solveLSM(byref(ierr))
        assert ierr.value == 0
        times = np.zeros((nsrc, nrec))
        L.fteik_solver2d_getTravelTimes64f(nrec, _d(times), byref(ierr))
        assert ierr.value == 0
        tt = np.zeros(nz * nx)
        L.fteik_solver2d_getTravelTimeField64f(tt.size, 0, _d(tt),
                                               byref(ierr))
        got.append((times, tt))
    L.fteik_solver2d_free()
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
    slow = orc.cell_slowness(vel, nz, nx)
    src = orc.source_locate((nz, nx, 1, dz, dx, 1.0, 0.0, 0.0, 0.0), zs[-1],
                            xs[-1], slow=slow, is3d=False)
    np.testing.assert_array_equal(
        got[0][1], orc.solve2d(slow, nz, nx, dz, dx, src, 1, 3.0))
