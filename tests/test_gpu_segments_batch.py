"""Rays of several atmospheres laid end to end, with their steps split over threads (few rays) against
the serial walk: layer counts of one step, one over a run and several runs a thread, in rows padded to
the deepest, rays in no order of their atmospheres and given an order of their own; and a NaN half
step past the cut in every table type, point rays and discs.

Both are FP64 sums of at most n = 300 terms of one sign in another order: n 2.2e-16 (1 + tau e^-tau)
< 1e-12 relative; the FP32 walk's weights and sums carry at most 10 roundings of 2^-24: < 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KINDS = [('float64', 'fp64', 1e-12), ('float32', 'fp32', 1e-6)]


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


@pytest.mark.parametrize('disc', [False, True])
@pytest.mark.parametrize('dtype,precision,tol', KINDS)
@pytest.mark.parametrize('nf', [1, 17])
@pytest.mark.parametrize('ordered', [False, True])
def test_batch_against_walk(K, nf, dtype, precision, tol, disc, ordered):
    import torch
    rng = np.random.default_rng(nf)
    counts = [65, 2, 300, 3]
    off = np.concatenate([[0], np.cumsum(counts)])
    alpha = 10.0 ** rng.uniform(-8.0, -6.0, (off[-1], nf))
    T = rng.uniform(110.0, 600.0, off[-1])
    atm = np.array([2, 0, 3, 2, 1, 1, 0, 2, 3, 2, 0])
    hds = rng.uniform(0.5, 1.5, (len(atm), max(counts) - 1)) * 1.0e5
    ns = np.array([counts[a] - 1 for a in atm], dtype=np.int32)
    ns[[3, 6]] = [-1, 40]
    order = rng.permutation(len(atm)) if ordered else None
    args = (torch.as_tensor(alpha, device='cuda').to(getattr(torch, dtype)), T, off, atm,
            torch.as_tensor(hds, device='cuda'), torch.as_tensor(ns, device='cuda'))
    kw = dict(order=order, disc=disc, precision=precision, tau_cut=30.0)
    split = K.integrate_batch(*args, **kw)
    walk = K.integrate_batch(*args, launch={'int_unroll': 4}, **kw)
    assert torch.isfinite(walk).all()
    torch.testing.assert_close(split, walk, rtol=tol, atol=0.0)


@pytest.mark.parametrize('disc', [False, True])
@pytest.mark.parametrize('dtype,precision,tol', KINDS)
def test_nan_past_the_cut(K, dtype, precision, tol, disc):
    import torch
    nl, nf, nray = 300, 20, 5
    tab = torch.full((nl, nf), 1.0e-6, device='cuda', dtype=getattr(torch, dtype))
    hds = torch.full((nray, nl - 1), 5.0e5, device='cuda', dtype=torch.float64)   # tau grows by 1 a step
    T = np.linspace(110.0, 600.0, nl)
    ns = torch.full((nray,), nl - 1, device='cuda', dtype=torch.int32)
    hds[2, 290] = float('nan')
    Tb = K.integrate(tab, T, hds, ns, disc=disc, precision=precision, tau_cut=20.0)
    assert torch.isnan(Tb[2]).all() and torch.isfinite(Tb[[0, 1, 3, 4]]).all()
    T[280] = np.nan                               # in every ray's path
    assert torch.isnan(K.integrate(tab, T, hds, ns, disc=disc, precision=precision, tau_cut=20.0)).all()
