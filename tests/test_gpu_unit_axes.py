"""Reductions of views in which an axis of one element stands between longer
ones: a contiguous array of rank 3 to 5 restricted to a single index of an
axis by a range.  The axes around it are then not one run of the buffer,
whatever stride the single element's axis kept.  Sums and maxima of whole
numbers in Int32 and Float64 are exact: equal to numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(3, 5, 4), (2, 5, 3, 4), (2, 3, 4, 3, 5)]


@pytest.mark.parametrize("dt", [np.int32, np.float64])
def test_single_index_of_an_axis(ph, dt):
    for n, shape in enumerate(SHAPES):
        h = np.random.default_rng(n).integers(-1000, 1000, shape).astype(dt)
        x = ph.NArray.from_numpy(h)
        picks = [{a: i} for a in range(1, len(shape)) for i in (0, shape[a] - 1)]
        for pick in picks if len(shape) < 5 else [{1: 2, 2: 1}, {1: 0, 3: 2}]:
            lits = ["%d..%d" % (pick[a], pick[a]) if a in pick else ".." for a in range(len(shape))]
            w = h[tuple(slice(pick[a], pick[a] + 1) if a in pick else slice(None) for a in range(len(shape)))]
            v = x.view(*lits)
            assert list(v.shape) == list(w.shape)
            assert v.sum() == w.sum() and v.max() == w.max(), (shape, lits)
            for k in range(len(shape)):
                others = tuple(a for a in range(len(shape)) if a != k)
                assert v.slices_sum(k) == [float(t) for t in w.sum(axis=others)], (shape, lits, k)
                assert v.slices_max(k) == [float(t) for t in w.max(axis=others)], (shape, lits, k)
