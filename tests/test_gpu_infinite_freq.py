"""An infinite or absurdly large frequency spoils its own column of the absorption table and no other, on the
series path (whose tiles take their columns' frequency range) as with the direct sums.  Tolerances as
between those two on finite requests (16 terms at their pole ratios): 1e-6 FP32, 1e-11 FP64."""
import numpy as np
import pytest

from radiobear_amd import synth

pytestmark = pytest.mark.gpu
C = synth.GAS_ROWS
SELECT = {'h2': 'h2_jj_ddb', 'h2o': 'h2o_bk', 'h2s': 'h2s_ddb', 'nh3': 'nh3_hs_sjs', 'ph3': 'ph3_jh'}


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


@pytest.mark.parametrize('prec,tol', [('fp32', 1e-6), ('fp64', 1e-11)])
@pytest.mark.parametrize('tile_k', [1, 2, 4])
@pytest.mark.parametrize('bad', [np.inf, 1e20, 1e39, 1e150])
def test_other_columns_are_finite(K, raw_lines, bad, tile_k, prec, tol):
    atm = synth.jupiter_like(21)
    cat = K.jupiter_catalog(raw_lines, h2o=synth.h2o_lines(300, 3))
    f = np.geomspace(31.0, 200.0, 140)
    f[[77, 139]] = bad
    ok = f < 1e15
    direct, series = (K.alpha(cat, K.absorbers_struct(SELECT), atm.P, atm.T, K.mix_table(atm.gas, C), f, prec,
                              launch={'alpha_k': tile_k, 'alpha_series': m}).double().cpu().numpy() for m in (1, 2))
    assert np.all(np.isfinite(direct[:, ok]))
    assert np.all(np.isfinite(series[:, ok]))
    assert np.max(np.abs(series[:, ok] - direct[:, ok]) / np.abs(direct[:, ok])) < tol
