"""Host inputs that cross to the device in one copy are accepted and refused as they are one by one."""
import numpy as np
import pytest
import torch

from radiobear_amd import kernels


@pytest.fixture
def on_host(monkeypatch):
    monkeypatch.setattr(kernels, 'device', lambda: torch.device('cpu'))


@pytest.mark.parametrize('x', [None, [1.0, None], np.array([1.0, 'a'], dtype=object), np.array(['1.5', '2']),
                               np.ones(3, dtype=np.longdouble), np.ones(3, dtype='>f8'), [1.0 + 0.0j],
                               [[1.0, 2.0], [3.0, 4.0]], np.arange(6, dtype=np.int32)[::2], np.float32(2.5), 3,
                               np.arange(12.0).reshape(3, 4).T, np.ones((0, 3)), [True, False],
                               np.ones(2, dtype=np.uint8), torch.arange(4)], ids=str)
def test_all_as_one(on_host, x):
    other = np.linspace(0.0, 1.0, 70)
    try:
        want = kernels.as_device(x)
    except Exception as e:
        with pytest.raises(type(e)):
            kernels.as_device_all(other, x)
        return
    a, b, c = kernels.as_device_all(other, x, [5.0])
    assert b.shape == want.shape and b.dtype == want.dtype and torch.equal(b, want)
    assert b.is_contiguous() and np.array_equal(a.numpy(), other) and c.tolist() == [5.0]


def test_odd_impact_parameters_are_a_value_error():
    pl = kernels.planet_desc(1.0, 0.9)
    with pytest.raises(ValueError):
        kernels.raypaths(pl, [1.0, 0.9], [1.0, 1.0], [0.1, 0.2, 0.3])
