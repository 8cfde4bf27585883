"""The locator's search through the index of its tables equals the oracle's
full search bit for bit (cell, objective, origin time): table counts around
the kernels' padded sizes, grids that the 4 x 4 x 4 blocks do not divide,
missing picks and uneven weights, ties, tables without structure, and
infinities, which are searched without the index."""
import ctypes

import numpy as np
import pytest

import fteik_amd as fa
from oracle import oracle as orc
from tests.gpu_helpers import lib

pytestmark = pytest.mark.gpu


def _tables(rng, ntf, nz, nx, ny):
    """Straight-ray times with a smooth perturbation, z fastest."""
    z, x, y = (np.arange(n, dtype=float) for n in (nz, nx, ny))
    out = []
    for _ in range(ntf):
        sx, sy = rng.uniform(0, nx), rng.uniform(0, ny)
        d = np.sqrt((x[None, :, None] - sx) ** 2 + (y[:, None, None] - sy) ** 2
                    + z[None, None, :] ** 2)
        out.append((d / 5.0 * (1 + 0.1 * np.sin(d / 7.0))).ravel())
    return np.array(out).astype(np.float32)


def _check(tables, obs, searches=1):
    """obs: (obs2tf, picks, weights) per event."""
    print("case:", tables.shape, len(obs), "events", flush=True)
    ntf, ngrd = tables.shape
    L = lib()
    f = L.fteik_k_locate_index_searches
    f.restype = ctypes.c_int
    loc = fa.Locator(len(obs), ntf, ngrd)
    loc.setReferenceCompatibility(0)
    ref = orc.Locator(len(obs), ntf, ngrd)
    for k in range(ntf):
        loc.setTravelTimeField(k + 1, tables[k])
        ref.set_table(k + 1, tables[k].astype(np.float64))
    for e, (k, t, w) in enumerate(obs):
        loc.setObservation(e + 1, k, t, w)
        ref.set_observation(e + 1, k.astype(np.int32), t, w)
    ev = np.arange(1, len(obs) + 1)
    opt, t0, ob = loc.locateEvents(ev)
    for e in range(len(obs)):
        r = ref.locate(e + 1, accumulate_t0=False, pad_argmin=False)
        assert (int(opt[e]), float(t0[e]), float(ob[e])) == r, "event %d" % e
    # events out of order and one at a time
    back = loc.locateEvents(ev[::-1])
    np.testing.assert_array_equal(back[0][::-1], opt)
    np.testing.assert_array_equal(back[1][::-1], t0)
    np.testing.assert_array_equal(back[2][::-1], ob)
    assert loc.locateEvent(2) == (opt[1], t0[1], ob[1])
    assert (f() >= searches) if searches else f() == 0
    # the reference's carried-over origin times follow on the last event
    loc.setReferenceCompatibility(1)
    a = loc.locateEvent(1)
    again = orc.Locator(len(obs), ntf, ngrd)
    for k in range(ntf):
        again.set_table(k + 1, tables[k].astype(np.float64))
    for e, (k, t, w) in enumerate(obs):
        again.set_observation(e + 1, k.astype(np.int32), t, w)
    again.locate(2, accumulate_t0=True, pad_argmin=False)
    assert a == again.locate(1, accumulate_t0=True, pad_argmin=True)
    loc.finalize()


def _events(rng, tables, n, missing=0.0, noise=0.1):
    ntf, ngrd = tables.shape
    out = []
    for c in rng.integers(0, ngrd, n):
        have = rng.uniform(size=ntf) >= missing
        have[rng.integers(0, ntf)] = True
        k = np.flatnonzero(have)
        w = rng.choice((1.0, 0.5, 0.1), k.size) if missing else np.ones(k.size)
        t = tables[k, c].astype(np.float64) + rng.uniform(0, 50) \
            + rng.normal(0, noise, k.size)
        out.append(((k + 1).astype(np.int32), t, w))
    return out


@pytest.mark.parametrize("ntf,shape,missing", [
    (9, (41, 37, 33), 0.0), (13, (23, 50, 45), 0.3), (17, (40, 36, 32), 0.2),
    (33, (21, 47, 29), 0.5), (41, (31, 29, 37), 0.0), (65, (20, 41, 31), 0.1),
    (96, (17, 33, 30), 0.2),
])
def test_index_equals_full_search(ntf, shape, missing):
    rng = np.random.default_rng(ntf)
    tables = _tables(rng, ntf, *shape)
    _check(tables, _events(rng, tables, 70, missing))


@pytest.mark.parametrize("kind", ["constant", "noise", "prime", "plane"])
def test_index_on_other_tables(kind):
    """Every cell a tie (the first one wins), tables without structure (no
    block can be left out), a cell count without divisors, a 2D grid."""
    rng = np.random.default_rng(3)
    ntf = 11
    if kind == "constant":
        tables = np.full((ntf, 20000), 2.5, dtype=np.float32)
    elif kind == "noise":
        tables = rng.uniform(0, 9, (ntf, 20000)).astype(np.float32)
    elif kind == "prime":
        tables = _tables(rng, ntf, 29, 30, 23)[:, :19997]
    else:
        tables = _tables(rng, ntf, 130, 151, 1)
    tables = np.ascontiguousarray(tables)
    _check(tables, _events(rng, tables, 60, 0.2))


@pytest.mark.parametrize("scale,weight,noise,missing", [
    (1000 * 10 ** (6 / 7), 0.99e15, 1.0, 0.0), (1.0e5, 0.99e15, 0.1, 0.2),
    (1.0e6, 0.99e15, 0.1, 0.2), (10 ** (-25 / 3), 1.1e-14, 0.1, 0.2),
    (1.0e-8, 1.01e-15, 1.0, 0.0), (10 ** -7.5, 1.01e-15, 1.0, 0.0),
    (1.0e-6, 1.1e-14, 0.1, 0.2)])
def test_index_at_the_ends_of_single_precision(scale, weight, noise, missing):
    """Misfits that overflow at a block's representative but not in all of
    its cells, and misfits of a few units of the smallest denormal."""
    rng = np.random.default_rng(17)
    tables = (_tables(rng, 9, 41, 37, 33) * np.float32(scale))
    obs = [(k, t, w * weight) for k, t, w in
           _events(rng, tables, 70, missing, noise=noise * scale)]
    _check(tables, obs)


def test_index_left_out_for_infinite_times():
    rng = np.random.default_rng(8)
    tables = _tables(rng, 10, 30, 31, 32)
    tables[4, 12345] = np.inf
    _check(tables, _events(rng, tables, 60), searches=0)


@pytest.mark.parametrize("change", ["table32", "table64", "sizes"])
def test_origin_times_carry_over_from_the_old_tables(change):
    """With the reference's compatibility an event starts from the origin
    times that the event before it left, also where a table (or the number of
    tables) changed in between and the earlier event went through the
    index."""
    print("case:", change, flush=True)
    rng = np.random.default_rng(21)
    ntf, shape = 32, (120, 120, 130)      # large: one event uses the index
    tables = _tables(rng, ntf, *shape)
    ngrd = tables.shape[1]
    obs = _events(rng, tables, 2)
    k, t, w = obs[0]
    obs[0] = (k[:-1], t[:-1], w[:-1])     # no pick at the last table
    L = lib()
    f = L.fteik_k_locate_index_searches
    f.restype = ctypes.c_int
    loc = fa.Locator(2, ntf, ngrd)
    ref = orc.Locator(2, ntf, ngrd)
    for i in range(ntf):
        loc.setTravelTimeField(i + 1, tables[i])
        ref.set_table(i + 1, tables[i].astype(np.float64))
    for e, (k, t, w) in enumerate(obs):
        loc.setObservation(e + 1, k, t, w)
        ref.set_observation(e + 1, k.astype(np.int32), t, w)
    loc.setReferenceCompatibility(0)
    for _ in range(2):                    # the second builds the index
        got = loc.locateEvent(2)
    assert f() == 1
    assert got == ref.locate(2, accumulate_t0=True, pad_argmin=False)
    if change == "sizes":
        ierr = ctypes.c_int(1)
        L.locate_setNumberOfTravelTimeFields(ntf - 1, ctypes.byref(ierr))
        assert ierr.value == 0
    else:
        new = tables[0] * np.float32(1.3)
        loc.setTravelTimeField(1, new if change == "table32"
                               else new.astype(np.float64))
        ref.set_table(1, new.astype(np.float64))
    loc.setReferenceCompatibility(1)
    assert loc.locateEvent(1) == ref.locate(1, accumulate_t0=True,
                                            pad_argmin=True)
    loc.finalize()


@pytest.mark.parametrize("kind,shape", [
    ("smooth", (81, 161, 161)), ("noise", (60, 60, 70))])
def test_large_calls_equal_full_search(kind, shape):
    """8,192 events through the index against a call of 8,193, which is
    searched in full: smooth tables, whose work space takes the events in two
    batches, and tables without structure, whose batch is given up after the
    bounds and searched in full (and so are the next calls)."""
    print("case:", kind, shape, flush=True)
    rng = np.random.default_rng(31)
    ntf, n = 8, 8193
    tables = _tables(rng, ntf, *shape) if kind == "smooth" else \
        rng.uniform(0, 9, (ntf, int(np.prod(shape)))).astype(np.float32)
    f = lib().fteik_k_locate_index_searches
    f.restype = ctypes.c_int
    loc = fa.Locator(n, ntf, tables.shape[1])
    loc.setReferenceCompatibility(0)
    for k in range(ntf):
        loc.setTravelTimeField(k + 1, tables[k])
    for e, (k, t, w) in enumerate(_events(rng, tables, n, 0.1)):
        loc.setObservation(e + 1, k, t, w)
    ev = np.arange(1, n + 1)
    full = loc.locateEvents(ev)
    assert f() == 0
    for calls in (1, 2):
        got = loc.locateEvents(ev[:-1])
        assert f() == (calls if kind == "smooth" else 1)
        for a, b in zip(got, full):
            np.testing.assert_array_equal(a, b[:-1])
    loc.setReferenceCompatibility(1)
    loc.finalize()
