"""Shapelets with per-tile beams in FP64: baselines of two shared-beam tiles, of one, and of none, in both
orders, with and without the per-class coherency table, against the oracle at 1e-12 of max|V|."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, PowerLaw, Shapelet, Source, SourceComponent, SourceList
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_shapelet_forms import AXES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [-1, 0], ids=["class-table", "no-table"])
@pytest.mark.parametrize("nt,dead,nchan,ncomp,df", [(2, 1, 1, 1, 40e3), (5, 2, 33, 17, 40e3), (6, 5, 65, 9, 1.28e6),
                                                    (7, 3, 129, 35, 10e3), (9, 4, 70, 18, 160e3), (4, 2, 97, 9, 80e3),
                                                    (4, 2, 96, 9, 80e3)])
def test_per_tile_beams_vs_oracle(nt, dead, nchan, ncomp, df, limit):
    rng = np.random.default_rng(nt)
    ra, dec = synthetic.cap_positions(rng, ncomp, 10.0)
    comps = []
    for k in range(ncomp):
        cf = [(int(rng.integers(0, 14)), int(rng.integers(0, 14)), float(rng.normal())) for _ in range(6)]
        ax = AXES[k % 9]
        comps.append(SourceComponent(float(ra[k]), float(dec[k]), Shapelet(ax, 0.7 * ax, 0.3 * k, cf),
                                     PowerLaw(-0.8, FluxDensity(150e6, 1.0 + k, 0.1, -0.2, 0.3))))
    srclist = SourceList([("s", Source(comps))])
    xyzs, freqs = synthetic.tiles(rng, nt, 1500.0), 100e6 + df * np.arange(nchan)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    for k, t in enumerate(rng.permutation(nt)[:dead]):
        delays[t, k] = 32
    _lib.call("sm_set_class_table_limit", limit)
    try:
        m = SkyModeller(AnalyticBeam(delays, gains), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                        synthetic.MWA_LAT_RAD)
        vis, _, vis64 = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    finally:
        _lib.call("sm_set_class_table_limit", -1)
    o32, o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD,
                                          beam="analytic", delays=delays, gains=gains), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(vis64, o64) <= 1e-12
    assert rel_err(vis, o32) <= 2e-7  # one FP32 rounding on each side
