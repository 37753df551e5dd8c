"""rbx_raypaths against the oracle's step-by-step geometry where the straight-line form of the
path can go wrong: two and three shells, rays in the equator plane (the 1e-6 rad latitude), rays
at and past the limb (missed shells, reflections, off-planet), tilted views, the sphere and the
'sec' limb.  ds: <= 1e-9 relative, as the recorded reference paths; path lengths and NaN steps
exact."""
import numpy as np
import pytest

from oracle import geometry
from radiobear_amd import synth

pytestmark = pytest.mark.gpu

RAYS = np.array([[0.0, 0.0], [0.3, 0.0], [0.0, 0.4], [-0.5, 0.2], [0.6, -0.6], [0.1, 0.92], [0.97, 0.05],
                 [0.995, 0.0], [0.0, 0.934], [0.0, 0.94], [0.7, 0.71], [0.999999, 0.0], [1.0, 0.0], [0.3, 1.2]])


@pytest.mark.parametrize('nl', [2, 3, 65])
@pytest.mark.parametrize('gtype,orientation,limb', [('ellipse', (0.0, 0.0), 'shape'), ('ellipse', (25.0, -31.0), 'shape'),
                                                    ('sphere', (10.0, 3.0), 'shape'), ('ellipse', (0.0, 12.0), 'sec')])
def test_paths_match_oracle(nl, gtype, orientation, limb):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from radiobear_amd import kernels as K
    atm = synth.jupiter_like(nl)
    pl = K.planet_desc(atm.Req, atm.Rpol, orientation, gtype, limb)
    ds, ns = (t.cpu().numpy() for t in K.raypaths(pl, atm.R, atm.N, RAYS, units='km'))
    half = K.raypaths(pl, atm.R, atm.N, RAYS)[0].cpu().numpy()
    for i, b in enumerate(RAYS):
        ref = geometry.compute_ds(atm.R, atm.N, b, atm.Req, atm.Rpol, orientation, gtype, limb)
        if ref.ds is None:
            assert ns[i] == -1
            continue
        n = len(ref.ds)
        assert ns[i] == n
        want = np.array(ref.ds)
        assert np.array_equal(np.isnan(ds[i, :n]), np.isnan(want))
        ok = ~np.isnan(want)
        assert np.all(np.abs(ds[i, :n][ok] - want[ok]) <= 1e-9 * np.abs(want[ok]))
        assert np.all(np.abs(half[i, :n][ok] - 5.0e4 * want[ok]) <= 1e-9 * 5.0e4 * np.abs(want[ok]))
