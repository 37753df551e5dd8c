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
