"""Copies at the edges of their vectors and tiles, bit for bit against numpy:
transposes whose sides straddle the tile sizes (32, 64, 128, 512) and the
narrow-side limits, in patches of tiles and reversed; rows that cross vectors
(trimmed borders of short, odd and long rows, reversed rows, permuted outer
axes, slabs); fills with a scattered region of any step on rows of any length.
Element sizes 1, 2, 4 and 8 bytes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NP = {"Bool": np.uint8, "BF16": np.uint16, "I32": np.int32, "F64": np.float64}


def _array(ph, dt, shape, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    if dt == "Bool":
        h = rng.integers(0, 2, n).astype(np.bool_).reshape(shape)
    elif dt == "F64":
        h = rng.standard_normal(n).reshape(shape)
    else:
        h = rng.integers(0, 60000, n).astype(NP[dt]).reshape(shape)
    return h, ph.NArray.from_numpy(h, dtype=getattr(ph.DType, dt))


@pytest.mark.parametrize("dt", ["Bool", "BF16", "I32", "F64"])
def test_transpose_tile_edges(ph, dt):
    shapes = [(8, 9), (7, 40), (16, 17), (31, 33), (32, 513), (513, 48), (49, 64), (63, 65), (127, 129), (700, 130),
              (2049, 10007)]
    for k, (a, b) in enumerate(shapes):
        h, x = _array(ph, dt, (a, b), k)
        assert np.array_equal(x.view().permute(1, 0).to_narr().to_numpy(), h.T), (a, b)
        if a < 2000:
            assert np.array_equal(x.view().reverse().permute(1, 0).to_narr().to_numpy(), h[::-1, ::-1].T), (a, b)
            z = ph.NArray.fill([b, a], ph.i32(0) if dt != "F64" else ph.f64(0.0), dtype=getattr(ph.DType, dt)).materialize()
            z.mutable_view().permute(1, 0)[[]] = x
            assert np.array_equal(z.to_numpy(), h.T), (a, b)
    for k, (shape, order) in enumerate([((5, 33, 21), (2, 0, 1)), ((9, 130, 12), (0, 2, 1)), ((64, 3, 66), (2, 1, 0)),
                                        ((17, 30, 9), (1, 2, 0)), ((2, 3, 20, 18), (1, 3, 0, 2))]):
        h, x = _array(ph, dt, shape, 40 + k)
        assert np.array_equal(x.view().permute(*order).to_narr().to_numpy(), h.transpose(order)), (shape, order)


@pytest.mark.parametrize("dt", ["BF16", "F64"])
def test_transposes_either_side_of_a_tile_size(ph, dt):
    """Below and above 700000 and 3 million elements (8-byte tiles change
    there), and 20 million and 32 tiles either way (tiles in patches)."""
    for k, (a, b) in enumerate([(836, 837), (837, 837), (701, 1001), (1731, 1733), (1733, 1733), (2049, 10007)]):
        h, x = _array(ph, dt, (a, b), k)
        assert np.array_equal(x.view().permute(1, 0).to_narr().to_numpy(), h.T), (a, b)


@pytest.mark.parametrize("dt", ["Bool", "BF16", "I32", "F64"])
def test_rows_across_vectors(ph, dt):
    for k, (rows, cols) in enumerate([(40, 9), (33, 16), (50, 35), (7, 700), (300, 31), (3, 5003)]):
        h, x = _array(ph, dt, (rows, cols), k)
        for lit, cut in [(("1..-2", "3..-2"), np.s_[1:-1, 3:-1]), (("..", "-1..0"), np.s_[:, ::-1]),
                         (("-1..0", "2.."), np.s_[::-1, 2:]), (("..2..", "1..-1"), np.s_[::2, 1:])]:
            g = x.view(*lit).to_narr()
            assert np.array_equal(g.to_numpy(), h[cut]), (rows, cols, lit)
            hz, z = _array(ph, dt, (rows, cols), 90 + k)
            z.mutable_view(*lit)[[]] = g
            hz[cut] = h[cut]
            assert np.array_equal(z.to_numpy(), hz), (rows, cols, lit)
    for k, shape in enumerate([(5, 7, 3), (6, 20, 33), (2, 3, 4, 19)]):
        h, x = _array(ph, dt, shape, 70 + k)
        order = list(range(len(shape)))
        order[0], order[1] = 1, 0
        assert np.array_equal(x.view().permute(*order).to_narr().to_numpy(), h.transpose(order)), shape


@pytest.mark.parametrize("dt", ["Bool", "BF16", "I32", "F64"])
def test_fill_scatter_any_rows(ph, dt):
    D = getattr(ph.DType, dt)
    fill = ph.f64(2.5) if dt == "F64" else ph.i32(1)
    for k, shape in enumerate([(3, 1), (5, 3), (9, 17), (33, 16), (70, 35), (11, 600), (4, 6, 7), (3, 5, 33)]):
        h0 = np.full(shape, 2.5 if dt == "F64" else 1, NP[dt] if dt != "Bool" else np.bool_)
        if dt == "BF16":
            h0[...] = 0x3F80  # 1.0
        outer = [("..", np.s_[:])] * (len(shape) - 2)
        for (rl, rc), (cl, cc) in [(("..", np.s_[:]), ("..", np.s_[:])), (("1..", np.s_[1:]), ("..-2..", np.s_[::-2])),
                                   (("-1..0", np.s_[::-1]), ("..3..", np.s_[::3])), (("..2..", np.s_[::2]), ("0..0", np.s_[0:1])),
                                   (("1..1", np.s_[1:2]), ("..-1", np.s_[:]))]:
            z = ph.NArray.fill(list(shape), ph.f32(1.0) if dt == "BF16" else fill, dtype=D)
            v = z.mutable_view(*[o[0] for o in outer], rl, cl)
            h, g = _array(ph, dt, tuple(v.shape), 100 + k)
            v[[]] = g
            want = h0.copy()
            cut = tuple(o[1] for o in outer) + (rc, cc)
            want[cut] = h.reshape(want[cut].shape)
            assert np.array_equal(z.to_numpy(), want), (shape, rl, cl)
