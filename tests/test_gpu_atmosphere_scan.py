"""rbx_atmosphere_batch where its chunked scan can go wrong: one and two layers, chunk edges (256
layers), several atmospheres, given z, and a p_ref no layer comes near.  z against the serial sum
from the deepest layer in long double: a sum of n positive terms, each within a few ulps, so
(n + 8) 2^-53 relative; R within that of z plus an ulp of req."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REQ, GM = 71492.0, 126686538.0
AMU = np.array([2.016, 4.003, 16.04, 17.030, 18.015, 34.076, 33.997, 0.0])


def serial_z(P, T, mix):
    P, T = P.astype(np.longdouble), T.astype(np.longdouble)
    H = 8.314462 * T / ((AMU[:, None] * mix).sum(0) * (GM / REQ ** 2)) / 1000.0
    dz = 0.5 * (H[:-1] + H[1:]) * np.log(P[1:] / P[:-1])
    return np.append(np.cumsum(dz[::-1])[::-1], 0.0)


@pytest.mark.parametrize('sizes', [[1], [2, 1, 3], [256, 257], [258, 512], [513, 64, 1000]])
@pytest.mark.parametrize('p_ref', [1.0, 5.0e7])
def test_scan_matches_serial_sum(sizes, p_ref):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels as K
    rng = np.random.default_rng(len(sizes) * 1000 + sizes[0])
    P = np.concatenate([np.logspace(-3, 2, n) for n in sizes])
    T = rng.uniform(100.0, 900.0, len(P))
    mix = rng.uniform(1e-6, 1e-3, (8, len(P)))
    mix[0], mix[1] = 0.86, 0.136
    off = np.concatenate([[0], np.cumsum(sizes)])
    Z, R, N = (t.cpu().numpy() for t in K.atmosphere_batch(P, T, mix, off, REQ, GM, p_ref))
    given = rng.uniform(0.0, 500.0, len(P))
    Zg, Rg, _ = (t.cpu().numpy() for t in K.atmosphere_batch(P, T, mix, off, REQ, GM, p_ref, Z=given))
    assert np.array_equal(Zg, given)
    for a in range(len(sizes)):
        s = slice(off[a], off[a + 1])
        want = serial_z(P[s], T[s], mix[:, s])
        tol = (sizes[a] + 8) * 2.0 ** -53 * want
        assert np.all(np.abs(Z[s] - want) <= tol)
        d = np.abs(P[s] - p_ref)
        iref = int(np.argmin(d)) if d.min() < 1e6 else 0
        assert np.all(np.abs(R[s] - (REQ + want - want[iref])) <= tol + tol[iref] + 2 * np.spacing(2 * REQ))
        assert np.array_equal(Rg[s], REQ + given[s] - given[s][iref])
    assert np.all(N > 1.0)
