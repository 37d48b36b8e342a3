"""Reductions that keep a middle axis of a view (slices(k).map(&.sum) and
(&.max)): the axes before and after it are read in place as two parts of the
columns.  Odd and even last axes (whole-vector and single loads), axes of one
element, several axes on either side, strided and reversed regions, every
element type; Int32 running totals in lexicographic order, and the sign of a
zero maximum from the first zero.  Sums of floats within 1e-12 sum |x|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [((3, 5, 7), 1), ((2, 9, 512), 1), ((40, 33, 20), 1), ((5, 300, 3), 1), ((1, 6, 50), 1), ((7, 4, 1), 1),
          ((6, 70, 1030), 1), ((130, 3, 1028), 1), ((3, 4, 5, 6), 1), ((3, 4, 5, 6), 2), ((70, 2, 9, 8), 2)]


def _others(h, k):
    return tuple(i for i in range(h.ndim) if i != k)


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int32, np.uint16])
def test_middle_axis(ph, dt):
    for n, (shape, k) in enumerate(SHAPES):
        rng = np.random.default_rng(n)
        if dt == np.int32:
            h = rng.integers(-1000, 1000, shape).astype(np.int32)
        elif dt == np.uint16:  # BFloat16 storage
            h = (rng.standard_normal(shape).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        else:
            h = rng.standard_normal(shape).astype(dt)
        x = ph.NArray.from_numpy(h)
        v = (h.astype(np.uint32) << 16).view(np.float32) if dt == np.uint16 else h
        w = v.astype(np.float64)
        s, m = np.array(x.slices_sum(k)), np.array(x.slices_max(k))
        assert np.array_equal(m, w.max(axis=_others(h, k))), (shape, k)
        tol = 0.0 if dt == np.int32 else 1e-12
        assert np.all(np.abs(s - w.sum(axis=_others(h, k))) <= tol * np.abs(w).sum(axis=_others(h, k))), (shape, k)


def test_middle_axis_of_views(ph):
    h = np.random.default_rng(3).standard_normal((9, 14, 33))
    x = ph.NArray.from_numpy(h)
    for lits, cut in [(("1..", "..", ".."), np.s_[1:]), (("..", "..2..", "3..-2"), np.s_[:, ::2, 3:-1]),
                      (("-1..0", "..", ".."), np.s_[::-1]), (("..", "..", "..2.."), np.s_[:, :, ::2]),
                      (("..", "-1..0", "-1..0"), np.s_[:, ::-1, ::-1])]:
        v, w = x.view(*lits), h[cut]
        assert np.array_equal(np.array(v.slices_max(1)), w.max(axis=(0, 2))), lits
        assert np.all(np.abs(np.array(v.slices_sum(1)) - w.sum(axis=(0, 2))) <= 1e-12 * np.abs(w).sum(axis=(0, 2))), lits
    p = x.view().permute(1, 0, 2).process(lambda e: e * 2.0 - 1.0)
    w = h.transpose(1, 0, 2) * 2.0 - 1.0
    assert np.array_equal(np.array(p.slices_max(1)), w.max(axis=(0, 2)))


def test_middle_axis_order(ph):
    top = 2**31 - 1
    h = np.zeros((2, 3, 2), np.int32)
    h[:, 1, :] = [[top, -1], [1, 0]]  # in order: top, top - 1, top
    assert ph.NArray.from_numpy(h).slices_sum(1) == [0.0, float(top), 0.0]
    h[:, 1, :] = [[top, 1], [-1, 0]]  # in order: top, overflow
    with pytest.raises(OverflowError):
        ph.NArray.from_numpy(h).slices_sum(1)
    z = np.full((3, 2, 70), -1.0)
    z[1, 0, 69], z[2, 0, 0] = -0.0, 0.0  # the first zero of slice 0 is -0.0
    z[0, 1, 5], z[2, 1, 1] = 0.0, -0.0
    m = ph.NArray.from_numpy(z).slices_max(1)
    assert np.signbit(m[0]) and not np.signbit(m[1]) and m == [0.0, 0.0]


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int32])
def test_every_row_of_a_tile_is_its_own(ph, dt):
    """Every element of a slice holds the slice's number, so a row of a tile
    that is read in another's place shows: tiles with and without missing
    rows and columns, the kept axis in the middle and in front."""
    for shape, k in [((4, 16, 512), 1), ((4, 33, 512), 1), ((8, 129, 515), 1), ((96, 1000, 515), 1), ((2, 96, 2048), 1),
                     ((33, 1030), 0), ((160, 1024), 0)]:
        j = np.arange(shape[k])
        h = np.broadcast_to(j.reshape([-1 if a == k else 1 for a in range(len(shape))]), shape)
        x = ph.NArray.from_numpy(np.ascontiguousarray(h).astype(dt))
        n = h.size // shape[k]
        assert x.slices_max(k) == [float(v) for v in j], (shape, k)
        assert x.slices_sum(k) == [float(v) for v in j * n], (shape, k)
