"""Near lines summed at Chebyshev nodes of column intervals where they are well away from them:
the series path against the direct sums over every line at the shapes that decide which interval
and which leaf a line takes.  Tolerances: the nodes leave 8e-9 (FP32, 16 nodes) or 7e-17 (FP64, 32
nodes) of a line's value, below the far-line series' own bounds, so 1e-6 and 1e-11 as for those
(16 terms at their pole ratios).  0.01-5000 GHz is an FP64 case only: the water lines' base cancels
around 723 GHz, and the direct FP32 sums are themselves 1.05e-6 from FP64 there."""
import numpy as np
import pytest

from radiobear_amd import synth

pytestmark = pytest.mark.gpu
C = synth.GAS_ROWS
SELECT = {'h2': 'h2_jj_ddb', 'h2o': 'h2o_bk', 'h2s': 'h2s_ddb', 'nh3': 'nh3_hs_sjs', 'ph3': 'ph3_jh'}
TOL = {'fp32': 1e-6, 'fp64': 1e-11}


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


def request(kind):
    """frequencies (GHz): leaves of one column, of no columns, of no width, of one line's width, and
    tiles on both sides of and across the 30 GHz switch of the inversion coefficients"""
    if kind == 'channels':       # a narrow band about an inversion line: leaves far narrower than a line
        return 23.6945 + 1e-4 * np.arange(193)
    if kind == 'equal':          # intervals of no width
        return np.repeat([22.2, 23.7, 183.31], 64)
    if kind == 'switch':         # the switch inside a leaf, one column past it, and between tiles
        return np.concatenate([np.linspace(5.0, 30.0, 97), np.linspace(30.0001, 60.0, 160)])
    if kind == 'one past':       # a last tile of one column
        return np.geomspace(0.6, 300.0, 257)
    if kind == 'linear':
        return np.linspace(1.0, 50.0, 129)
    if kind == 'wide':
        return np.geomspace(0.01, 5000.0, 96)
    rng = np.random.default_rng(8)
    return rng.permutation(np.geomspace(0.5, 100.0, 150))


@pytest.mark.parametrize('prec', ['fp32', 'fp64'])
@pytest.mark.parametrize('tile_k', [1, 2, 4])
@pytest.mark.parametrize('kind', ['channels', 'equal', 'switch', 'one past', 'linear', 'wide', 'shuffled'])
def test_near_tree_matches_direct(K, raw_lines, kind, tile_k, prec):
    if kind == 'wide' and prec == 'fp32':
        pytest.skip('the direct FP32 sums are 1.05e-6 from FP64 where the base cancels')
    atm = synth.jupiter_like(29)
    cat = K.jupiter_catalog(raw_lines, h2o=synth.h2o_lines(400, 3))
    f = request(kind)
    got = [K.alpha(cat, K.absorbers_struct(SELECT), atm.P, atm.T, K.mix_table(atm.gas, C), f, prec,
                   launch={'alpha_k': tile_k, 'alpha_series': m}).double().cpu().numpy() for m in (1, 2)]
    assert np.all(np.isfinite(got[1]))
    assert float(np.max(np.abs(got[1] - got[0]) / np.abs(got[0]))) < TOL[prec]
