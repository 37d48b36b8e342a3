"""Int32 reductions whose running totals are first bounded and, where a bound
leaves Int32, followed exactly.  Small values (the bounds settle it), large
values that cancel (the exact states settle it, no overflow), totals that leave
Int32 and come back (overflow), and totals that end outside.  Sums and maxima
are whole numbers below 2^53: equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one element, under a leaf of 256 columns, its edges, over a tile of 1024, rows over one tile
SHAPES = [(1, 1), (3, 255), (17, 256), (5, 1025), (600, 40), (1100, 1500)]


def _fits(w, axis):
    """Every running total of w along axis (None: all elements in order) stays in Int32."""
    t = np.cumsum(w if axis is not None else w.reshape(-1), axis=axis or 0) if axis != 1 else np.cumsum(w, axis=1)
    return bool(t.min() >= -(2**31) and t.max() < 2**31)


def _check(x, w):
    for k in (0, 1):
        if _fits(w, 1 - k):
            assert x.slices_sum(k) == [float(v) for v in w.sum(axis=1 - k)], (w.shape, k)
        else:
            with pytest.raises(OverflowError):
                x.slices_sum(k)
        assert x.slices_max(k) == [float(v) for v in w.max(axis=1 - k)], (w.shape, k)
    if _fits(w, None):
        assert x.sum() == w.sum(), w.shape
    else:
        with pytest.raises(OverflowError):
            x.sum()
    assert x.max() == w.max(), w.shape


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["small", "cancel", "leave", "end", "negative"])
def test_int32_running_totals(ph, shape, kind):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    big = 1 << 30
    r, c = np.indices(shape)
    if kind == "small":
        w = rng.integers(-1000, 1000, shape)
    elif kind == "cancel":  # +big, -big, ... along every row and every column
        w = np.where((r + c) % 2 == 0, big, -big) + (rng.integers(0, 2, shape) if shape[0] < 600 else 0)
    elif kind == "leave":
        w = np.zeros(shape, np.int64)
        w[-1, -3:] = [2**31 - 1, 5, -7][-min(3, shape[1]):]
    elif kind == "end":
        w = np.full(shape, 2**31 - 1)
    else:
        w = np.full(shape, -(2**31))
    w = w.astype(np.int64)
    _check(ph.NArray.from_numpy(w.astype(np.int32)), w)
