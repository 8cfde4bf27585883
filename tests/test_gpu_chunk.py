"""The chunked tiles of the iteration sweeps (the default until a tile shape
is chosen): fields equal the oracle's bit for bit, and the streamed tiles'
where the oracle has no such mode, at the edges of tiles (8 x 8 columns),
chunks (4 levels) and runs (4,092 levels), with and without skipping."""
from ctypes import byref, c_int

import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_helpers import lib, _d

pytestmark = pytest.mark.gpu

# nz, nx, ny, (dz, dx, dy), source in cells, iterations.  Random velocities
# in every cell bend the rays, so fields keep changing for several iterations
# in ever fewer places.
CASES = [
    (3, 3, 3, (10.0, 10.0, 10.0), (0.4, 0.9, 0.7), 3),
    (4, 9, 10, (10.0, 10.0, 10.0), (1.5, 0.0, 7.9), 4),
    (5, 17, 8, (10.0, 12.0, 9.0), (0.0, 14.5, 3.2), 6),
    (18, 16, 25, (5.0, 5.0, 5.0), (15.9, 7.9, 0.1), 9),
    (33, 41, 34, (10.0, 10.0, 10.0), (16.3, 20.0, 31.7), 12),
    (61, 26, 33, (7.0, 11.0, 13.0), (3.3, 23.9, 0.0), 12),
    (4080, 9, 17, (10.0, 10.0, 10.0), (2000.5, 3.0, 8.0), 4),
    (4100, 9, 17, (10.0, 10.0, 10.0), (4000.0, 0.0, 14.9), 4),
]


def _model(nz, nx, ny, seed):
    rng = np.random.default_rng(seed)
    return 1000.0 * rng.uniform(1.0, 6.0, (nz - 1) * (nx - 1) * (ny - 1))


def _oracle(vel, nz, nx, ny, d, src, nsweep):
    slow = orc.cell_slowness(vel, nz, nx, ny, order=0)
    s = orc.source_locate((nz, nx, ny) + d + (0.0, 0.0, 0.0), *src, slow)
    return orc.solve3d(slow, nz, nx, ny, *d, s, nsweep, 3.0, schedule=1)


def _solver(case, seed, precision=0, skipping=1, tile=None, conv=0.0):
    nz, nx, ny, d, c, nsweep = case
    L, ierr = lib(), c_int(1)
    L.fteik_solver3d_initialize(nz, nx, ny, 0.0, 0.0, 0.0, *d, nsweep, 3.0,
                                conv, 0, byref(ierr))
    assert ierr.value == 0
    L.fteik_solver3d_setPrecision(precision, byref(ierr))
    L.fteik_solver3d_setTileSkipping(skipping, byref(ierr))
    if tile is not None:
        L.fteik_solver3d_setTile(tile, tile, byref(ierr))
        assert ierr.value == 0
    vel = _model(nz, nx, ny, seed)
    src = tuple(a * b for a, b in zip(c, d))
    L.fteik_solver3d_setVelocityModel64f(vel.size, _d(vel), byref(ierr))
    assert ierr.value == 0
    s = [np.array([a]) for a in src]
    L.fteik_solver3d_setSources64f(1, *[_d(a) for a in s], byref(ierr))
    assert ierr.value == 0
    L.fteik_solver3d_solveSourceLSM(1, byref(ierr))
    assert ierr.value == 0
    tt = np.zeros(nz * nx * ny)
    L.fteik_solver3d_getTravelTimeField64f(tt.size, 0, _d(tt), byref(ierr))
    assert ierr.value == 0
    return tt, vel, src


@pytest.mark.parametrize("skipping", [1, 0])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_chunked_sweeps_match_oracle(case, skipping):
    c = CASES[case]
    print("case: chunked", c, "skipping", skipping, flush=True)
    tt, vel, src = _solver(c, 100 + case, skipping=skipping)
    np.testing.assert_array_equal(tt, _oracle(vel, *c[:4], src, c[5]))


@pytest.mark.parametrize("case", [1, 2, 4, 5])
def test_chunked_mixed_matches_streamed(case):
    c = CASES[case]
    print("case: chunked mixed", c, flush=True)
    a, _, _ = _solver(c, 200 + case, precision=1)
    b, _, _ = _solver(c, 200 + case, precision=1, tile=12)
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("cube", [True, False])
@pytest.mark.parametrize("precision", [0, 1])
def test_chunked_batch(cube, precision):
    """Uneven grids: FP64 against the oracle, mixed against the streamed
    tiles; solved twice, the second time with the tile shape chosen."""
    cases = [c[:3] + ((10.0, 10.0, 10.0) if cube else c[3],) + c[4:5]
             for c in CASES[:7]]
    nsweep = 9
    print("case: chunked batch", cube, precision, flush=True)
    L, ierr = lib(), c_int(1)
    L.fteik_batch3d_initialize(len(cases), byref(ierr))
    assert ierr.value == 0
    models = [_model(*c[:3], 300 + i) for i, c in enumerate(cases)]
    srcs = [tuple(a * b for a, b in zip(c[4], c[3])) for c in cases]
    for i, c in enumerate(cases):
        L.fteik_batch3d_setGrid(i + 1, *c[:3], 0.0, 0.0, 0.0, *c[3],
                                _d(models[i]), *srcs[i], byref(ierr))
        assert ierr.value == 0
    L.fteik_batch3d_setPrecision(precision, byref(ierr))
    fields, status = [], []
    for tile in (None, 12):
        if tile is not None:
            L.fteik_batch3d_setTile(tile, byref(ierr))
            assert ierr.value == 0
        L.fteik_batch3d_solve(nsweep, 3.0, byref(ierr))
        # 2: corrections of a mixed solve that ran out before it converged
        assert ierr.value in ((0, 2) if precision else (0,))
        status.append(ierr.value)
        got = []
        for i, c in enumerate(cases):
            tt = np.zeros(c[0] * c[1] * c[2])
            L.fteik_batch3d_getTravelTimeField64f(i + 1, tt.size, 0, _d(tt),
                                                  byref(ierr))
            assert ierr.value == 0
            got.append(tt)
        fields.append(got)
    L.fteik_batch3d_free()
    assert status[0] == status[1]
    for i, c in enumerate(cases):
        np.testing.assert_array_equal(fields[0][i], fields[1][i])
        if precision == 0:
            np.testing.assert_array_equal(
                fields[0][i], _oracle(models[i], *c[:4], srcs[i], nsweep))


def _serpentine(nz, nx, ny):
    """Fast corridors along x, joined at alternate ends, between walls of 1
    m/s: with sources at the first corridor's end the front passes a few bends
    an iteration."""
    v = np.ones((ny - 1, nx - 1, nz - 1))
    v[::2] = 5000.0
    v[1::4, -1] = 5000.0
    v[3::4, 0] = 5000.0
    return v.ravel()


SERPENTINE = (3, 10, 260)
SOURCE = (5.0, 15.0, 5.0)
D = (10.0, 10.0, 10.0)


def test_more_sweeps_than_the_record_has_numbers():
    """The change record numbers sweeps modulo 255: a field that still changes
    in every iteration from the 8th to the 40th (sweeps 57 to 320)."""
    nz, nx, ny = SERPENTINE
    vel = _serpentine(*SERPENTINE)
    print("case: serpentine", SERPENTINE, flush=True)
    L, ierr = lib(), c_int(1)
    L.fteik_solver3d_initialize(nz, nx, ny, 0.0, 0.0, 0.0, *D, 40, 3.0, 0.0,
                                0, byref(ierr))
    assert ierr.value == 0
    L.fteik_solver3d_setVelocityModel64f(vel.size, _d(vel), byref(ierr))
    assert ierr.value == 0
    s = [np.array([a]) for a in SOURCE]
    L.fteik_solver3d_setSources64f(1, *[_d(a) for a in s], byref(ierr))
    last = None
    for nsweep in (31, 32, 33, 40):
        L.fteik_solver3d_setNumberOfSweeps(nsweep, byref(ierr))
        L.fteik_solver3d_solveSourceLSM(1, byref(ierr))
        assert ierr.value == 0
        tt = np.zeros(nz * nx * ny)
        L.fteik_solver3d_getTravelTimeField64f(tt.size, 0, _d(tt),
                                               byref(ierr))
        np.testing.assert_array_equal(
            tt, _oracle(vel, nz, nx, ny, D, SOURCE, nsweep))
        assert last is None or np.any(tt != last)
        last = tt


@pytest.mark.parametrize("precision,nsweep,cube", [
    (0, 36, True), (0, 7, False), (1, 5, True)])
def test_chunked_batch_of_many_grids(precision, nsweep, cube):
    """A batch large enough for the chunked tiles (24,576 nodes per level of
    the longest sweep), of ragged grids and one whose field keeps changing:
    every field equals the streamed tiles', some the oracle's too."""
    rng = np.random.default_rng(71)
    dims = [SERPENTINE] + [tuple(int(n) for n in rng.integers(30, 65, 3))
                           for _ in range(80)]
    nodes = sum(a * b * c for a, b, c in dims)
    assert nodes >= 96 * 256 * max(map(sum, dims))
    print("case: batch of many", precision, nsweep, cube, flush=True)
    d = D if cube else (9.0, 10.0, 12.0)
    models = [_serpentine(*SERPENTINE)]
    models += [_model(*n, 400 + i) if i % 3 else np.repeat(
        np.linspace(2000.0, 5000.0, n[2] - 1), (n[0] - 1) * (n[1] - 1))
        for i, n in enumerate(dims[1:])]
    srcs = [SOURCE] + [tuple(rng.uniform(0, n - 2.1) * h for n, h in
                             zip(n, d)) for n in dims[1:]]
    L, ierr = lib(), c_int(1)
    L.fteik_batch3d_initialize(len(dims), byref(ierr))
    assert ierr.value == 0
    for i, n in enumerate(dims):
        L.fteik_batch3d_setGrid(i + 1, *n, 0.0, 0.0, 0.0, *d, _d(models[i]),
                                *srcs[i], byref(ierr))
        assert ierr.value == 0
    L.fteik_batch3d_setPrecision(precision, byref(ierr))
    fields = []
    for tile in (None, 12):
        if tile is not None:
            L.fteik_batch3d_setTile(tile, byref(ierr))
            assert ierr.value == 0
        L.fteik_batch3d_solve(nsweep, 3.0, byref(ierr))
        # 2: corrections of a mixed solve that ran out before it converged
        assert ierr.value in ((0, 2) if precision else (0,))
        got = [np.zeros(a * b * c) for a, b, c in dims]
        for i, tt in enumerate(got):
            L.fteik_batch3d_getTravelTimeField64f(i + 1, tt.size, 0, _d(tt),
                                                  byref(ierr))
            assert ierr.value == 0
        fields.append(got)
    L.fteik_batch3d_free()
    for a, b in zip(*fields):
        np.testing.assert_array_equal(a, b)
    for i in (0, 1, 2, 80) if precision == 0 else ():
        np.testing.assert_array_equal(
            fields[0][i], _oracle(models[i], *dims[i], d, srcs[i], nsweep))
