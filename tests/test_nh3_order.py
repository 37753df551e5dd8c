"""kernels.nh3_order names every column of a request once, whatever its frequencies are: the device
array of the reordered frequencies is read at every column."""
import numpy as np
import pytest

from radiobear_amd import kernels


@pytest.mark.parametrize('f', [[40.0, np.nan, 10.0], [np.nan], [np.inf, 30.0, -np.inf, 30.1], [5.0, 1.0]])
def test_every_column_once(f):
    order, low = kernels.nh3_order(f)
    assert sorted(order) == list(range(len(f)))
    assert all(f[i] <= 30.0 for i in order[:low]) and not any(f[i] <= 30.0 for i in order[low:])
    assert list(order[:low]) == sorted(order[:low]) and list(order[low:]) == sorted(order[low:])
