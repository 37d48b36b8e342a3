"""Forms of the copy kernels that small arrays of the usual kinds do not reach,
bit for bit against numpy: transposes in patches of tiles over several planes
and reversed; destinations of over 100 MB, whose stores are streamed, at every
element size; and the fill+scatter of a buffer that does not start on 16 bytes,
which keeps the 64-bit kernel."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NP = {1: np.bool_, 2: np.uint16, 4: np.int32, 8: np.float64}
DT = {1: "Bool", 2: "BF16", 4: "I32", 8: "F64"}
CODE = {1: 4, 2: 3, 4: 0, 8: 2}


def _values(es, shape, seed):
    b = np.random.default_rng(seed).integers(0, 2 if es == 1 else 250, int(np.prod(shape)), dtype=np.uint8)
    return (b.astype(NP[es]) if es != 8 else b * 0.5).reshape(shape)


def _array(ph, es, shape, seed=1):
    h = _values(es, shape, seed)
    return h, ph.NArray.from_numpy(h, dtype=getattr(ph.DType, DT[es]))


@pytest.mark.parametrize("es", [1, 2, 4, 8])
def test_patches_of_several_planes(ph, es):
    h, x = _array(ph, es, (5, 2050, 2060))
    assert np.array_equal(x.view().permute(0, 2, 1).to_narr().to_numpy(), h.transpose(0, 2, 1))
    assert np.array_equal(x.view().reverse().permute(0, 2, 1).to_narr().to_numpy(), h[::-1, ::-1, ::-1].transpose(0, 2, 1))
    z = x.clone()
    z.mutable_view().permute(0, 2, 1)[[]] = ph.NArray.from_numpy(np.ascontiguousarray(h[::-1].transpose(0, 2, 1)),
                                                                 dtype=getattr(ph.DType, DT[es]))
    assert np.array_equal(z.to_numpy(), h[::-1])


@pytest.mark.parametrize("es", [1, 2, 4, 8])
def test_streamed_stores(ph, es):
    """One run of over 100 MB, in order, in rows backwards and of an odd row
    length, and rows that start on whole vectors; rows that do not are stored
    as usual."""
    side = {1: 10496, 2: 7424, 4: 5248, 8: 3712}[es]  # side^2 es bytes: over 100 MiB, whole vectors
    h, x = _array(ph, es, (side, side))
    assert side * side * es > 100 << 20
    assert np.array_equal(x.clone().to_numpy(), h)
    assert np.array_equal(x.view().permute(1, 0).to_narr().to_numpy(), h.T)
    assert np.array_equal(x.view("-1..0", "..").to_narr().to_numpy(), h[::-1])
    assert np.array_equal(x.view("..", "-1..0").to_narr().to_numpy(), h[:, ::-1])
    for lit, cut in (("16..-17", np.s_[16:-16]), ("3..-2", np.s_[3:-1])):
        z = x.clone()
        z.mutable_view("..", lit)[[]] = x.view("-1..0", lit).to_narr()
        want = h.copy()
        want[:, cut] = h[::-1, cut]
        assert np.array_equal(z.to_numpy(), want), lit
    n = side * side // (side - 1)
    y = x.view("0..%d" % (n - 2), "0..%d" % (side - 2)).to_narr()
    assert np.array_equal(y.to_numpy(), h[:n - 1, :side - 1])


@pytest.mark.parametrize("es", [1, 2, 4, 8])
def test_fill_scatter_off_16_bytes(ph, es):
    from test_gpu_alias_deep import _desc
    lib = ctypes.CDLL(os.path.join(ph.LIB_DIR, "libphhip.so"))
    i64 = lambda *v: (ctypes.c_int64 * len(v))(*v)  # noqa: E731
    for k, (rows, cols) in enumerate([(1, 1), (5, 3), (33, 35), (9, 700), (70, 16)]):
        for (r0, rs), (c0, cs) in [((0, 1), (0, 1)), ((rows - 1, -1), (0, 2)), ((0, 2), (cols - 1, -3))]:
            nr = (rows - 1) // abs(rs) + 1
            nc = (cols - 1) // abs(cs) + 1
            hs, src = _array(ph, es, (nr, nc), 10 + k)
            hb, buf = _array(ph, es, (rows * cols + 24,), 20 + k)
            fill = np.full(1, 1, NP[es]) if es != 8 else np.full(1, 2.5)
            for off in (1, 3):  # elements
                if off * es % 16 == 0:
                    continue
                rc = lib.ph_fill_scatter(ctypes.c_void_p(buf.device_ptr + off * es), ctypes.c_int32(CODE[es]), i64(rows, cols),
                                         ctypes.c_int32(2), i64(r0, c0), i64(rs, cs), i64(nr, nc), (ctypes.c_int32 * 2)(0, 1),
                                         ctypes.c_void_p(src.device_ptr), ctypes.byref(_desc(CODE[es], nr * nc, [nr, nc])),
                                         ctypes.c_void_p(fill.ctypes.data))
                assert rc == 0
                want = np.full((rows, cols), fill[0])
                want[np.ix_(r0 + rs * np.arange(nr), c0 + cs * np.arange(nc))] = hs
                hb[off:off + rows * cols] = want.reshape(-1)
                got = np.zeros(rows * cols + 24, NP[es])
                assert lib.ph_d2h(ctypes.c_void_p(got.ctypes.data), ctypes.c_void_p(buf.device_ptr),
                                  ctypes.c_size_t(got.nbytes)) == 0
                assert np.array_equal(got, hb), (rows, cols, rs, cs, off)
