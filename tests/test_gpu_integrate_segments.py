"""Requests of few (ray, 64 frequencies) wavefronts: each ray's path points are split into runs,
one per thread.  Compared with the serial walk (a launch shape that names the unroll keeps it)
at run boundaries: fewer points than runs, one point over, columns past a block's, rays of no,
one and few steps, batches and NaN half steps.

Both are FP64 sums of at most n = 1300 terms of one sign in another order, tau included, and a
weight moves by its tau's rounding: n * 2.2e-16 * (1 + tau e^-tau) relative in all < 1e-12.  The
FP32 walk's weights and sums carry 2^-24 roundings, at most 2 (1 + tau e^-tau) + 8 of them in a
sum of 8: < 1e-6 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


def request(nl, nf, nray, seed):
    rng = np.random.default_rng(seed)
    alpha = 10.0 ** (np.linspace(-10.0, -5.0, nl)[:, None] + rng.uniform(-1.0, 1.0, (nl, nf)))
    hds = rng.uniform(0.5, 1.5, (nray, nl - 1)) * 2.0e7 / nl
    ns = np.full(nray, nl - 1, dtype=np.int32)
    ns[1:4] = [-1, 1, min(3, nl - 1)][:max(0, min(3, nray - 1))]
    return alpha, np.linspace(110.0, 600.0, nl), hds, ns


@pytest.mark.parametrize('disc', [False, True])
@pytest.mark.parametrize('dtype,precision,tol', [('float64', 'fp64', 1e-12), ('float32', 'fp32', 1e-6)])
@pytest.mark.parametrize('nl,nf,nray', [(2, 1, 1), (3, 5, 2), (64, 16, 5), (66, 17, 40), (257, 4, 1), (259, 3, 7),
                                        (1300, 65, 9),
                                        (90, 33, 170)])
def test_segments_against_walk(K, nl, nf, nray, dtype, precision, tol, disc):
    import torch
    alpha, T, hds, ns = request(nl, nf, nray, nl + nf)
    tab = torch.as_tensor(alpha, device='cuda').to(getattr(torch, dtype))
    hg, ng = torch.as_tensor(hds, device='cuda'), torch.as_tensor(ns, device='cuda')
    cut = 40.0
    walk, iw0 = K.integrate(tab, T, hg, ng, disc=disc, precision=precision, tau_cut=cut, with_intW=True,
                            launch={'int_unroll': 4})
    seg, iw1 = K.integrate(tab, T, hg, ng, disc=disc, precision=precision, tau_cut=cut, with_intW=True)
    torch.testing.assert_close(seg, walk, rtol=tol, atol=0.0)
    torch.testing.assert_close(iw1, iw0, rtol=tol, atol=1e-300)


def test_nan_step_past_the_cut(K):
    import torch
    alpha, T, hds, ns = request(300, 6, 3, 1)
    ns[:] = 299
    hds[1, 290] = np.nan
    args = (torch.as_tensor(alpha * 1e3, device='cuda'), T, torch.as_tensor(hds, device='cuda'),
            torch.as_tensor(ns, device='cuda'))
    seg = K.integrate(*args, precision='fp64', tau_cut=20.0)
    assert torch.isnan(seg[1]).all() and torch.isfinite(seg[[0, 2]]).all()
