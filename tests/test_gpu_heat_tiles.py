"""The heat step kernel at the edges of its tiles, bit for bit against the
oracle's single steps: grids of one cell or line, exactly one tile and one
more or less (tiles are 64 or 128 columns by 32 to 256 rows), several tiles
with a ragged last one, grids low and wide or narrow and tall (one axis
shorter than a tile), and runs of one pass, of an even and of an odd number
of passes.  Energies (summed by the passes themselves) within 1e-14 of
sum |u| of the oracle's."""
import numpy as np
import oracle_api as O
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1), (1, 300), (300, 1), (2, 2), (31, 63), (32, 64), (33, 65), (48, 64), (49, 64), (64, 64), (65, 64), (64, 65),
         (127, 129), (257, 300), (37, 1500), (1500, 37), (513, 1025), (700, 1111)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("steps,every", [(1, 1), (2, 0), (7, 7), (50, 20), (113, 50)])
def test_heat_tile_edges(ph, dt, steps, every):
    rng = np.random.default_rng(11)
    for ny, nx in GRIDS:
        u0 = (rng.standard_normal((ny, nx)) * 3).astype(dt)
        u = ph.NArray.from_numpy(u0)
        e = np.array(ph.heat2d(u, 0.2, steps, every=every))
        ref, eref = O.heat2d(u0, 0.2, steps, every=every)
        assert np.array_equal(u.to_numpy(), ref), (ny, nx, steps)
        assert e.shape == np.shape(eref if every else [])
        if every:
            assert np.all(np.abs(e - eref) <= 1e-14 * np.abs(u0).astype(np.float64).sum()), (ny, nx, steps)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_heat_tiles_of_large_grids(ph, dt):
    """Grids large enough for the tallest tiles, some tiles moved inside the grid."""
    rng = np.random.default_rng(12)
    for ny, nx, steps in [(2050, 2300, 11), (4500, 4100, 13)]:
        u0 = rng.standard_normal((ny, nx)).astype(dt)
        u = ph.NArray.from_numpy(u0)
        e = np.array(ph.heat2d(u, 0.25, steps, every=steps))
        ref, eref = O.heat2d(u0, 0.25, steps, every=steps)
        assert np.array_equal(u.to_numpy(), ref), (ny, nx)
        assert np.all(np.abs(e - eref) <= 1e-14 * np.abs(u0).astype(np.float64).sum())
