"""Pairs of a tile with its own beam and one of the shared beam, in FP64, at the edges of the kernel's
row and column groups, channel chunks, component stages and component slices; against the oracle at
the parity bound 1e-12 of max|V|."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, SkyModeller
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_tile_forms import sky

pytestmark = pytest.mark.gpu


def check(nt, dead, freqs, srclist):
    rng = np.random.default_rng(nt)
    xyzs = synthetic.tiles(rng, nt, 1000.0)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    for k, t in enumerate(rng.permutation(nt)[:dead]):  # baselines in both orders
        delays[t, k % 16] = 32
    m = SkyModeller(AnalyticBeam(delays, gains), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                    synthetic.MWA_LAT_RAD)
    vis, _, vis64 = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    o32, o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD,
                                          beam="analytic", delays=delays, gains=gains), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(vis64, o64) <= 1e-12
    assert rel_err(vis, o32) <= 2e-7  # one FP32 rounding on each side


@pytest.mark.parametrize("gaussian", [False, True], ids=["point", "gaussian"])
@pytest.mark.parametrize("nt,dead,nchan,ncomp", [(3, 1, 1, 1), (11, 2, 7, 3), (19, 3, 8, 4), (37, 5, 9, 15),
                                                 (40, 8, 17, 16), (43, 9, 3, 17), (58, 26, 10, 37), (12, 3, 5, 1601)])
def test_rows_by_columns_vs_oracle(nt, dead, nchan, ncomp, gaussian):
    check(nt, dead, 167e6 + 40e3 * np.arange(nchan), sky(np.random.default_rng(ncomp), ncomp, gaussian))


# Wide and descending steps take the general envelope ratios; flagged channels shorten the chunks.
@pytest.mark.parametrize("freqs", [80e6 + 1.28e6 * np.arange(19), (167e6 + 40e3 * np.arange(19))[::-1].copy(),
                                   (167e6 + 40e3 * np.arange(32))[[2, 3, 4, 5, 6, 7, 17, 18, 19, 28]]],
                         ids=["wide", "descending", "flagged"])
def test_channel_steps_vs_oracle(freqs):
    check(21, 4, freqs, sky(np.random.default_rng(5), 9, True, 0.05))
