"""Rays at a top shell of no radius (NaN, infinite or 0, as an atmosphere rebuilt from a NaN
temperature has) are off the planet: nsteps -1, as no trial point of raypath.py:60-110 lies below it.
By the split walk (limb 'shape') and by a thread's own (limb 'sec', and many rays)."""
import numpy as np
import pytest

from radiobear_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('limb,nray', [('shape', 5), ('shape', 32769), ('sec', 5)])
@pytest.mark.parametrize('top', [np.nan, np.inf, 0.0])
def test_off_planet(top, limb, nray):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels as K
    atm = synth.jupiter_like(40)
    pl = K.planet_desc(atm.Req, atm.Rpol, limb=limb)
    b = synth.random_disc_rays(nray, 3)
    assert (K.raypaths(pl, atm.R, atm.N, b)[1] > 0).any()
    R = np.array(atm.R)
    R[0] = top
    ns = K.raypaths(pl, R, atm.N, b)[1]
    assert (ns == -1).all()


@pytest.mark.parametrize('limb', ['shape', 'sec'])
@pytest.mark.parametrize('k', [1, 2, 17, 39])
def test_infinite_shell_part_way_down(k, limb):
    """An infinite radius at shell k turns outwards there: paths end above it (raypath.py:212-216)."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels as K
    atm = synth.jupiter_like(40)
    pl = K.planet_desc(atm.Req, atm.Rpol, limb=limb)
    R = np.array(atm.R)
    R[k] = np.inf
    b = synth.random_disc_rays(32769, 3, rmax=0.9)
    walk, ns = K.raypaths(pl, R, atm.N, b)
    assert (ns == k - 1).all()
    ds, m = K.raypaths(pl, R, atm.N, b[:40])
    assert torch.equal(m, ns[:40])
    torch.testing.assert_close(ds[:, :k - 1], walk[:40, :k - 1], rtol=1e-9, atol=0.0)
