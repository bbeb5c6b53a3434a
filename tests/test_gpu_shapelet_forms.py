"""The shared-beam shapelet kernel's forms (channel slots, baselines per wave) and its segments (runs
of channels within one cell of the basis table), against the oracle at the parity bound 1e-12 of
max|V|."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import synthetic
from mwa_hyperdrive_amd.modeller import NoBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, PowerLaw, Shapelet, Source, SourceComponent, SourceList
from oracle import oracle as orc
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def check(nt, freqs, axes, ncoeff, radius=1500.0):
    rng = np.random.default_rng(nt)
    ra, dec = synthetic.cap_positions(rng, len(axes), 10.0)
    comps = []
    for k, ax in enumerate(axes):
        cf = [(int(rng.integers(0, 14)), int(rng.integers(0, 14)), float(rng.normal()))
              for _ in range(ncoeff)]
        comps.append(SourceComponent(float(ra[k]), float(dec[k]), Shapelet(ax, 0.7 * ax, 0.3 * k, cf),
                                     PowerLaw(-0.8, FluxDensity(150e6, 1.0 + k, 0.1, -0.2, 0.3))))
    srclist = SourceList([("s", Source(comps))])
    xyzs = synthetic.tiles(rng, nt, radius)
    m = SkyModeller(NoBeam(), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    vis, _, vis64 = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    o32, o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(vis64, o64) <= 1e-12
    assert rel_err(vis, o32) <= 2e-7  # one FP32 rounding on each side


# 1.3 km, 45 cells to 0.01 degrees of axis at 167 MHz: the smallest stay in a cell, the largest leave
# the table on the long baselines and pass 64 segments, so batches of all kinds alternate.
AXES = [1e-5, 3e-4, 2e-3, 0.02, 1e-4, 0.2, 5e-3, 1e-3, 0.05]


@pytest.mark.parametrize("df", [10e3, 80e3, 160e3, 1.28e6])
@pytest.mark.parametrize("nt,nchan,ncomp", [(2, 1, 1), (3, 31, 33), (5, 33, 17), (4, 64, 9), (3, 65, 16), (4, 129, 32),
                                            (2, 384, 3)])
def test_forms_vs_oracle(nt, nchan, ncomp, df):
    check(nt, 100e6 + df * np.arange(nchan), [AXES[k % 9] for k in range(ncomp)], 7)


@pytest.mark.parametrize("ncoeff", [1, 4, 5, 140])
def test_coefficient_counts_vs_oracle(ncoeff):
    axes = [3e-4, 1e-3, 2e-3]
    check(4, 167e6 + 40e3 * np.arange(70), axes, ncoeff)


@pytest.mark.parametrize("freqs", [(80e6 + 1.28e6 * np.arange(70))[::-1].copy(), np.array([180e6, 90e6, 200e6]),
                                   np.delete(167e6 + 80e3 * np.arange(128), [0, 1, 16, 30, 31, 32, 33, 77])],
                         ids=["wide-descending", "scattered", "gaps"])
def test_channel_orders_vs_oracle(freqs):
    check(5, freqs, AXES, 6)
