"""Alpha.scale_table: one factor for every layer is what the per-layer list of it gives."""
import numpy as np
import pytest

from radiobear_amd import config
from radiobear_amd.alpha import Alpha


@pytest.mark.parametrize('scale,value', [(False, 1.0), (True, 1.0), (None, 1.0), (2, 2.0), (0.5, 0.5),
                                         (np.float32(1.5), 1.5), ('3.0', 3.0), ('x', 1.0)])
@pytest.mark.parametrize('nl', [1, 7])
def test_one_factor(scale, value, nl):
    a = Alpha(config=config.planetConfig('jupiter', configFile=None), verbose=False)
    got = a.scale_table(scale, nl)
    assert got.dtype == np.float64 and np.array_equal(got, a.scale_table([value] * nl, nl))
