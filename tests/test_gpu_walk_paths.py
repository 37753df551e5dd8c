"""The serial walk of the brightness integration, which large images and maps take: requests of few
rays split a ray's steps over threads instead, so small cases reach the walk only by a launch shape
that names its unroll or block order, or by enough rays.  The properties the walk has to keep (the
frequency order's bit-identity, the factor table as another source of the same numbers, no tau cut
for a ray whose path holds a NaN) are held here on the walk itself, and the factor table is shown to
be read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALK = [{'int_unroll': 8}, {'int_unroll': 4, 'int_map': 1}, {'int_map': 2}]


@pytest.fixture(scope='module')
def K():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels
    return kernels


def request(nl, nf, nray, dtype, seed=5):
    """Columns over three decades of opacity, paths of several lengths, one ray off the planet."""
    import torch
    rng = np.random.default_rng(seed)
    alpha = 10.0 ** rng.uniform(-8.0, -5.0, nf) * np.exp(rng.uniform(-0.3, 0.3, (nl, nf)))
    hds = rng.uniform(2.0e5, 6.0e5, (nray, nl))
    ns = rng.integers(nl // 2, nl + 1, nray).astype(np.int32)
    ns[nray // 2] = -1
    tab = torch.as_tensor(alpha, device='cuda').to(getattr(torch, dtype))
    return tab, np.linspace(110.0, 650.0, nl), torch.as_tensor(hds, device='cuda'), torch.as_tensor(ns, device='cuda')


def factors(K, T, nl, hds, ns):
    import torch
    from radiobear_amd import _lib
    nray, ld = hds.shape
    fac = torch.full((nray, ld, 4), 7.0, dtype=torch.float32, device='cuda')
    _lib.check(_lib.lib().rbx_integrate_factors(K._ptr(T), nl, K._ptr(hds), ld, K._ptr(ns), nray, K._ptr(fac),
                                                K._stream()))
    return fac


def by_cols(K, tab, cols, T, hds, ns, disc, precision, cut, fac, launch):
    import torch
    from radiobear_amd import _lib
    nl, nf = tab.shape
    nray, ld = hds.shape
    aprec = _lib.FP32 if tab.dtype == torch.float32 else _lib.FP64
    Tb, iw = (torch.full((nray, nf), np.nan, dtype=torch.float64, device='cuda') for _ in range(2))
    _lib.check(_lib.lib().rbx_integrate_cols(K._ptr(tab), aprec, K._ptr(cols), K._ptr(T), nl, nf, K._ptr(hds), ld,
                                             K._ptr(ns), nray, 1 if disc else 0, _lib.PRECISIONS[precision],
                                             float(cut), K._ptr(Tb), K._ptr(iw), K._ptr(fac),
                                             _lib.launch_ref(launch), K._stream()))
    return Tb, iw


@pytest.mark.parametrize('launch', WALK, ids=str)
@pytest.mark.parametrize('precision,dtype,disc', [('fp64', 'float64', False), ('fp32', 'float32', False),
                                                  ('fp64', 'float32', True), ('fp32', 'float32', True)])
def test_identity_order(K, precision, dtype, disc, launch):
    import torch
    tab, T, hds, ns = request(120, 200, 7, dtype)
    T = K.as_device(T)
    ident = torch.arange(200, dtype=torch.int32, device='cuda')
    fac = factors(K, T, 120, hds, ns)
    on = ns.cpu().numpy() >= 0
    for cut in (0.0, 25.0):
        Tb0, iw0 = K.integrate(tab, T, hds, ns, disc=disc, precision=precision, tau_cut=cut, with_intW=True,
                               launch=launch)
        for f in (None, fac):
            Tb1, iw1 = by_cols(K, tab, ident, T, hds, ns, disc, precision, cut, f, launch)
            assert torch.equal(Tb0[on], Tb1[on]) and torch.equal(iw0[on], iw1[on])


@pytest.mark.parametrize('launch', WALK, ids=str)
def test_factor_table_is_read(K, launch):
    """A table with the temperature factors doubled gives Tb doubled."""
    import torch
    tab, T, hds, ns = request(90, 150, 6, 'float32')
    T = K.as_device(T)
    ident = torch.arange(150, dtype=torch.int32, device='cuda')
    fac = factors(K, T, 90, hds, ns)
    Tb0, _ = by_cols(K, tab, ident, T, hds, ns, False, 'fp32', 20.0, fac, launch)
    fac[..., 3] *= 2.0
    Tb1, _ = by_cols(K, tab, ident, T, hds, ns, False, 'fp32', 20.0, fac, launch)
    warm = Tb0 > 50.0
    assert warm.sum() > 300
    assert torch.equal(Tb1[warm], 2.0 * Tb0[warm])


@pytest.mark.parametrize('nray,launch', [(4, WALK[0]), (4, WALK[1]), (4, WALK[2]), (80, None)], ids=str)
@pytest.mark.parametrize('precision', ['fp64', 'fp32', 'fp32 factors'])
def test_nan_past_the_cut(K, precision, nray, launch):
    """A NaN half step past the depth where every column is opaque keeps the ray's Tb NaN.  80 rays
    of 130 columns take the walk by themselves."""
    import torch
    rng = np.random.default_rng(4)
    nl, nf = 200, 130
    prec = precision[:4]
    tab = torch.as_tensor(1.0e-6 * np.exp(rng.uniform(-0.5, 0.5, (nl, nf))), device='cuda')
    tab = tab.float() if prec == 'fp32' else tab
    T = K.as_device(np.linspace(120.0, 600.0, nl))
    h = np.full((nray, nl), 5.0e5)                 # tau grows by about 1 a step
    h[1, 120] = np.nan
    hds, ns = torch.as_tensor(h, device='cuda'), torch.full((nray,), nl, dtype=torch.int32, device='cuda')
    cut = 20.0 if prec == 'fp32' else 40.0
    if precision == 'fp32 factors':
        ident = torch.arange(nf, dtype=torch.int32, device='cuda')
        Tb, _ = by_cols(K, tab, ident, T, hds, ns, False, prec, cut, factors(K, T, nl, hds, ns), launch)
    else:
        Tb = K.integrate(tab, T, hds, ns, precision=prec, tau_cut=cut, launch=launch)
    assert torch.isnan(Tb[1]).all()
    assert torch.isfinite(Tb[[r for r in range(nray) if r != 1]]).all()


@pytest.mark.parametrize('launch', WALK, ids=str)
@pytest.mark.parametrize('precision,dtype', [('fp64', 'float64'), ('fp32', 'float32')])
def test_ordered(K, precision, dtype, launch):
    """The frequency order changes nothing with a cut no column reaches, and with one that binds only
    what the cut leaves out (< 2 T_max e^-cut)."""
    tab, T, hds, ns = request(160, 700, 11, dtype, 23)
    on = ns.cpu().numpy() >= 0

    def Tb(cut, ordered):
        return K.integrate(tab, T, hds, ns, precision=precision, tau_cut=cut, ordered=ordered,
                           launch=launch).cpu().numpy()[on]
    assert np.array_equal(Tb(1.0e30, False), Tb(1.0e30, True))
    full = Tb(0.0, False)
    for cut in (20.0, 40.0):
        bound = 1e-9 + 2.0 * T.max() * np.exp(-cut)
        assert np.max(np.abs(Tb(cut, True) - full)) < bound
        assert np.max(np.abs(Tb(cut, True) - Tb(cut, False))) < 2.0 * bound
