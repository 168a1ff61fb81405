"""The comparison that the numerics tests rest on."""
import numpy as np
import pytest

from _helpers import assert_close


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1.1])
def test_assert_close_refuses(bad):
    a = np.ones((2, 3))
    a[1, 1] = bad
    with pytest.raises(AssertionError):
        assert_close(a, np.ones((2, 3)), 1e-3, 1e-3)
    with pytest.raises(AssertionError):
        assert_close(np.ones((2, 3)), a, 1e-3, 1e-3)


def test_assert_close_takes_equal_specials():
    a = np.array([1.0, np.inf, -np.inf, np.nan])
    assert_close(a, a.copy(), 1e-3, 1e-3)
