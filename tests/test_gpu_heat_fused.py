"""The heat step kernel tile by tile (PH_HEAT_TILE names one), with the cell's
first operation as a multiply and a subtract and as one fused multiply-add:
bit for bit against the oracle's single steps.  A run is fused when max|u|
shows that 4u cannot overflow, which is asked of runs predicted at 300 us or
more; the launch of that question, which ph_heat2d_noalloc never asks, shows
that a run was long enough."""
import ctypes
import os

import numpy as np
import oracle_api as O
import pytest

pytestmark = pytest.mark.gpu

# columns a lane, rows a wavefront, wavefronts (heat_tile.hip)
COMMON = {0: (1, 4, 8), 1: (1, 6, 8), 2: (1, 8, 8), 3: (2, 4, 8), 5: (2, 12, 8), 8: (4, 1, 1), 9: (4, 2, 1), 10: (4, 4, 1),
          11: (4, 8, 1), 12: (2, 16, 1), 13: (2, 12, 2), 14: (2, 16, 2), 15: (2, 12, 4), 16: (2, 16, 4)}
TILES = {np.float64: {**COMMON, 4: (2, 8, 8), 6: (2, 16, 8), 7: (2, 24, 8)},
         np.float32: {**COMMON, 4: (2, 8, 16), 6: (2, 12, 16), 7: (2, 16, 16)}}


def launches(ph, u0, r, steps, every):
    """Field and energies of ph.heat2d, and its launches beyond those of
    ph_heat2d_noalloc, whose field must be the same."""
    lib = ctypes.CDLL(os.path.join(ph.LIB_DIR, "libphhip.so"))
    f64 = u0.dtype == np.float64
    v, tmp = ph.NArray.from_numpy(u0), ph.NArray.empty(list(u0.shape), ph.DType.F64 if f64 else ph.DType.F32)
    e = ph.NArray.empty([steps // every + 1 if every else 1], ph.DType.F64)
    n0 = ph.launch_count()
    rc = lib.ph_heat2d_noalloc(ctypes.c_int32(2 if f64 else 1), ctypes.c_void_p(v.device_ptr), ctypes.c_void_p(tmp.device_ptr),
                               ctypes.c_int64(u0.shape[0]), ctypes.c_int64(u0.shape[1]), ctypes.c_double(r),
                               ctypes.c_int64(steps), ctypes.c_int64(every), ctypes.c_void_p(e.device_ptr if every else None))
    assert rc == 0
    n1 = ph.launch_count()
    u = ph.NArray.from_numpy(u0)
    energy = np.array(ph.heat2d(u, r, steps, every=every))
    extra = ph.launch_count() - n1 - (n1 - n0)
    got = u.to_numpy()
    assert np.array_equal(got, v.to_numpy(), equal_nan=True), (u0.shape, steps)
    return got, energy, extra


def _grids(t):
    tx, ty = 64 * t[0], t[1] * t[2]
    if t[2] == 1:  # a lone wavefront spans the rows: whole tiles, a row missing, columns missing
        return [(ty, 2 * tx + 37), (max(1, ty - 1), 2 * tx + 37), (ty, tx - 5)]
    return [(ty + ty // 2 + 1, tx + 37), (ty - 3, 2 * tx + 5), (ty + 9, tx - 5), (ty, tx)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("tile", range(17))
def test_every_tile(ph, monkeypatch, dt, tile):
    monkeypatch.setenv("PH_HEAT_TILE", str(tile))
    rng = np.random.default_rng(tile)
    for ny, nx in _grids(TILES[dt][tile]):
        u0 = (rng.standard_normal((ny, nx)) * 3).astype(dt)
        for steps, every in [(1, 0), (13, 5)]:
            u, e, extra = launches(ph, u0, 0.2, steps, every)
            ref, eref = O.heat2d(u0, 0.2, steps, every=every)
            assert extra == 0 and np.array_equal(u, ref), (ny, nx, steps)
            if every:
                assert np.all(np.abs(e - eref) <= 1e-14 * np.abs(u0).astype(np.float64).sum()), (ny, nx, steps)
        # (a small r, so that the field of a long run stays a field)
        u, _, extra = launches(ph, u0, 1e-3, 4000, 0)
        ref, _ = O.heat2d(u0, 1e-3, 4000, every=0)
        assert extra == 1 and np.array_equal(u, ref), (ny, nx)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_long_runs_that_must_not_fuse(ph, dt):
    """Values whose 4u overflows, infinities and NaN: max|u| says no and the
    separate operations run, as for r > 1/4, where it is not asked.  One step a
    pass (an energy each), so that every pass's first operation shows."""
    big = np.finfo(dt).max
    rng = np.random.default_rng(73)
    shape = (200, 700)
    cases = []
    u0 = rng.random(shape).astype(dt)
    u0[10, 20] = big * 0.9
    u0[190:194, 100] = -big * 0.6
    u0[100:106, 300:310] = big * 0.3  # 4u overflows, uN - 4u in one operation does not
    cases.append((u0, 0.2, 1))
    u1 = rng.random(shape).astype(dt)
    u1[5, 5], u1[199, 699], u1[100, 350] = np.inf, -np.inf, np.nan
    cases.append((u1, 0.2, 1))
    u2 = rng.random(shape).astype(dt)  # the last value alone, right at the limit and over it
    u2[199, 699] = np.nextafter(np.ldexp(dt(1), 1020 if dt == np.float64 else 124), dt(np.inf))
    cases.append((u2, 0.25, 1))
    cases.append((rng.random(shape).astype(dt), 0.3, 0))
    for u0, r, asked in cases:
        u, _, extra = launches(ph, u0, r, 120, 1)
        ref, _ = O.heat2d(u0, r, 120, every=1)
        assert extra == asked
        assert np.array_equal(u, ref, equal_nan=True), r
        num = ~np.isnan(ref)
        bits = np.uint64 if dt == np.float64 else np.uint32
        assert np.array_equal(u[num].view(bits), ref[num].view(bits)), r
