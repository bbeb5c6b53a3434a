"""Auto-correlations summed once per beam row, at the edges of the kernel's 16-channel groups and
16-component steps, against the oracle in FP64."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, NoBeam, SkyModeller
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_tile_forms import sky

pytestmark = pytest.mark.gpu


# 2000 components of one row split into slices, the last of them shorter; dead: tiles with a row of
# their own. The FP64 sums of n terms differ by their order: n 1.1e-16, below 1e-12.
@pytest.mark.parametrize("nt,nchan,ncomp,dead", [(2, 1, 1, None), (5, 15, 16, None), (9, 17, 17, 0), (17, 33, 129, 3),
                                                 (3, 16, 2000, 0), (20, 47, 301, 20)])
def test_autos_vs_oracle(nt, nchan, ncomp, dead):
    rng = np.random.default_rng(ncomp)
    xyzs, freqs = synthetic.tiles(rng, nt, 500.0), 170e6 + 80e3 * np.arange(nchan)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    for t in range(dead or 0):
        delays[nt - 1 - t, t % 16] = 32
    srclist = sky(rng, ncomp, False)
    beam = NoBeam() if dead is None else AnalyticBeam(delays, gains)
    m = SkyModeller(beam, srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    v32, v64 = np.zeros((nchan, nt, 8), np.float32), np.zeros((nchan, nt, 8))
    m.model_timestep_autos_with(0.1, synthetic.MWA_LAT_RAD, v32, v64)
    kw = {} if dead is None else {"beam": "analytic", "delays": delays, "gains": gains}
    o32, o64 = orc.model_autos(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.1, synthetic.MWA_LAT_RAD, **kw), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(v64, o64) <= 1e-12
    assert rel_err(v32, o64) <= 1e-7
