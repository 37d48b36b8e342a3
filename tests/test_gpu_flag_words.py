"""Element flags (Int32 overflow, division by zero, negative exponents) across
calls: a call that raises is followed by one that does not and must not see
the old flag, every bit alone and together, in maps, in-place maps and sums,
on one element and on many workgroups that all raise.  Small and large
read-backs through the same page."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 300, 1 << 20])
def test_flags_do_not_outlive_their_call(ph, n):
    big = ph.NArray.fill([n], ph.i32(2**31 - 1))
    one = ph.NArray.fill([n], ph.i32(1))
    zero = ph.NArray.fill([n], ph.i32(0))
    neg = ph.NArray.fill([n], ph.i32(-1))
    for _ in range(3):
        with pytest.raises(OverflowError):
            big + one
        assert np.array_equal((one + one).to_numpy(), np.full(n, 2, np.int32))
        with pytest.raises(ZeroDivisionError):
            one // zero
        assert np.array_equal((big - one).to_numpy(), np.full(n, 2**31 - 2, np.int32))
        with pytest.raises(ValueError):
            one ** neg
        assert np.array_equal((one ** one).to_numpy(), np.ones(n, np.int32))
    h = np.ones(n, np.int32)
    h[n // 2] = 2**31 - 1
    x = ph.NArray.from_numpy(h)
    if n > 1:
        with pytest.raises(OverflowError):
            x.sum()
    with pytest.raises(OverflowError):
        x + one  # a single element of a single workgroup
    assert one.sum() == n


@pytest.mark.parametrize("n", [1, 7, 8191, 8192, 8193, 100000])
def test_read_back_sizes(ph, n):
    for dt in (np.float64, np.int32, np.uint16, np.bool_):
        h = (np.arange(n) % 251).astype(dt)
        assert np.array_equal(ph.NArray.from_numpy(h).to_numpy(), h)
