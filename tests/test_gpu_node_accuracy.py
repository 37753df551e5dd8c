"""Accuracy of the series path's near lines beside the direct sums, one line at a time and as tables.

One narrow line beside an interval of columns, at distances on both sides of the ellipse from which it
is taken at the interval's nodes.  FP32: a term at a column carries at most ten roundings of its
denominator (FP32 distances at a quarter of x + |Ds| or more) and six more, 16 x 2^-24 = 9.6e-7, and
one at the nodes less.  FP64: the nodes leave 1.1e-15 and round their f to 2^-53, which moves the line
by up to 2.6e-15 in the narrowest interval here and, over the interpolation, three times that; the
direct sum's own roundings are 2e-15: 1.2e-14.

Tables: lines at nodes and far lines carry no FP32 rounding, so a table is no further from FP64 than
the direct FP32 sums: in the largest error up to one unit in the last place of the result, and in the
mean square.  0.01-5000 GHz has the widest intervals; there the water lines' base cancels around 723
GHz, where an entry's relative error is whatever its cancellation makes of a rounding, so the largest
error is bounded against the sums before the cancellation: 1e-6 of |alpha| + |base| f^2, the base from
the water row at 5000 GHz, where the lines themselves are 2 % of it."""
import numpy as np
import pytest

from radiobear_amd import synth

pytestmark = pytest.mark.gpu
C = synth.GAS_ROWS
SELECT = {'h2': 'h2_jj_ddb', 'h2o': 'h2o_bk', 'h2s': 'h2s_ddb', 'nh3': 'nh3_hs_sjs', 'ph3': 'ph3_jh'}
TOL = {'fp32': 16 * 2.0 ** -24, 'fp64': 1.2e-14}


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


def table(K, cat, select, atm, f, prec, **launch):
    return K.alpha(cat, K.absorbers_struct(select), atm.P, atm.T, K.mix_table(atm.gas, C), f, prec,
                   launch=launch).double().cpu().numpy()


@pytest.mark.parametrize('prec', ['fp32', 'fp64'])
@pytest.mark.parametrize('form', ['gross', 'ben-reuven'])
def test_one_line_beside_an_interval(K, raw_lines, form, prec):
    from radiobear_amd import _lib
    atm = synth.jupiter_like(9, pmax=0.02)   # narrow lines
    cat = K.jupiter_catalog(raw_lines)
    lo = 20.0
    for hi in (40.0, 32.0, 24.0):
        f, r = np.linspace(lo, hi, 64), 0.5 * (hi - lo)
        for t in (0.757, 0.85, 0.93, 0.945, 1.1, 1.21, 1.225, 1.4, 1.8):   # in half widths from the interval's end
            for f0 in (lo - t * r, hi + t * r):
                one = {'f0': [f0], 'I0': [1e-20], 'E': [50.0]}
                if form == 'gross':
                    cat.set_lines(_lib.LINES_H2S, dict(one, GH2S=[6.0]))
                    select = {'h2s': 'h2s_ddb'}
                else:
                    cat.set_lines(_lib.LINES_PH3, dict(one, WgtI0=[1.0], WgtFGB=[1.0], WgtSB=[1.0]))
                    select = {'ph3': 'ph3_jh'}
                want = table(K, cat, select, atm, f, 'fp64', alpha_series=1, alpha_k=1)
                got = table(K, cat, select, atm, f, prec, alpha_series=2, alpha_k=1)
                assert np.all(want > 0.0)
                assert float(np.max(np.abs(got - want) / want)) < TOL[prec], (hi, t, f0)


@pytest.mark.parametrize('tile_k', [1, 2, 4])
@pytest.mark.parametrize('wide', [False, True])
def test_tables_no_further_than_direct(K, raw_lines, wide, tile_k):
    from radiobear_amd import _lib
    f = np.geomspace(0.01, 5000.0, 96) if wide else np.geomspace(0.3, 300.0, 201)
    atm = synth.jupiter_like(60)
    cat = K.jupiter_catalog(raw_lines, h2o=synth.h2o_lines(400, 3))
    want, rows = K.alpha(cat, K.absorbers_struct(SELECT), atm.P, atm.T, K.mix_table(atm.gas, C), f, 'fp64',
                         by_constituent=True, launch={'alpha_series': 1, 'alpha_k': 1})
    want = want.cpu().numpy()
    direct, series = (np.abs(table(K, cat, SELECT, atm, f, 'fp32', alpha_series=m, alpha_k=tile_k) - want)
                      for m in (1, 2))
    if wide:
        water = rows[_lib.CONSTITUENTS.index('h2o')].cpu().numpy()
        assert np.all(series < 1e-6 * (np.abs(want) + np.abs(water[:, -1:]) * (f / f[-1]) ** 2))
    else:
        assert np.max(series / want) < np.max(direct / want) + 2.0 ** -23
    assert np.mean((series / want) ** 2) <= np.mean((direct / want) ** 2)
