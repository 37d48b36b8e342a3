"""ph_d2h called through the C-ABI with what its small copies must not take:
null pointers and a range past the buffer's end are errors of the call (they
never reach a kernel); device memory as the destination and buffers of
another owner are copied by the runtime.  Small and large sizes, and offsets
that leave the range inside its buffer."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PH_E_HIP = -10


@pytest.fixture(scope="module")
def lib(ph):
    lib = ctypes.CDLL(os.path.join(ph.LIB_DIR, "libphhip.so"))
    for f in (lib.ph_d2h, lib.ph_h2d):
        f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    lib.ph_alloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    lib.ph_free.argtypes = [ctypes.c_void_p]
    return lib


@pytest.mark.parametrize("n", [8, 1000, 65536, 65544, 300000])
def test_ranges(lib, n):
    p = ctypes.c_void_p()
    assert lib.ph_alloc(ctypes.byref(p), n) == 0
    h = np.random.default_rng(n).integers(0, 256, n).astype(np.uint8)
    assert lib.ph_h2d(p, h.ctypes.data, n) == 0
    for o, m in [(0, n), (1, n - 1), (n - 1, 1), (n // 2, n - n // 2), (3, 4)]:
        g = np.zeros(m + 8, np.uint8)
        assert lib.ph_d2h(g.ctypes.data, p.value + o, m) == 0
        assert np.array_equal(g[:m], h[o:o + m]) and not g[m:].any()
    g = np.full(n + 16, 7, np.uint8)
    for o, m in [(0, n + 1), (n - 1, 2), (n // 2, n)]:  # past the end: refused, nothing written
        assert lib.ph_d2h(g.ctypes.data, p.value + o, m) == PH_E_HIP
    for dst, src in [(None, p), (g.ctypes.data, None)]:
        assert lib.ph_d2h(dst, src, n) == PH_E_HIP
    assert (g == 7).all()
    assert lib.ph_d2h(g.ctypes.data, p, n) == 0 and np.array_equal(g[:n], h)  # later calls work
    assert lib.ph_free(p) == 0


@pytest.mark.parametrize("n", [40, 1 << 17])
def test_other_memory(lib, n):
    """Buffers that the HIP runtime gave someone else, on either side."""
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(m.split()[-1] for m in f if "libamdhip64.so" in m))
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    h = np.random.default_rng(n).integers(0, 256, n).astype(np.uint8)
    g = np.zeros(n, np.uint8)
    p, t = ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.ph_alloc(ctypes.byref(p), n) == 0 and hip.hipMalloc(ctypes.byref(t), n) == 0
    assert lib.ph_h2d(p, h.ctypes.data, n) == 0
    assert lib.ph_d2h(t, p, n) == 0  # into device memory
    assert lib.ph_d2h(g.ctypes.data, t, n) == 0 and np.array_equal(g, h)
    assert lib.ph_free(p) == 0 and hip.hipFree(t) == 0
