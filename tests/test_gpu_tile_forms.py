"""The FP64 tile-pair kernel's forms (channel width, rows per block, component split) at the edges
of their tiles, against the oracle at the parity bound 1e-12 of max|V|."""

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import NoBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import (CurvedPowerLaw, FluxDensity, Gaussian, Point, PowerLaw, Source,
                                        SourceComponent, SourceList)
from oracle import oracle as orc
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def sky(rng, n, gaussian, axis=1e-3):
    ra, dec = synthetic.cap_positions(rng, n, 10.0)
    comps = []
    for k in range(n):
        fd = FluxDensity(150e6, float(rng.lognormal()), *(0.1 * rng.normal(size=3)).tolist())
        ft = PowerLaw(-0.8, fd) if k % 2 else CurvedPowerLaw(-0.7, fd, 0.1)
        ct = Gaussian(axis * float(rng.uniform(0.1, 1)), 0.1 * axis, float(rng.uniform(0, 3))) if gaussian else Point()
        comps.append(SourceComponent(float(ra[k]), float(dec[k]), ct, ft))
    return SourceList([("s", Source(comps))])


def check(nt, freqs, srclist, radius=1000.0):
    rng = np.random.default_rng(nt)
    xyzs = synthetic.tiles(rng, nt, radius)
    m = SkyModeller(NoBeam(), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    vis, _, vis64 = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    o32, o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(vis64, o64) <= 1e-12
    assert rel_err(vis, o32) <= 2e-7  # one FP32 rounding on each side


# Few blocks take the component-split forms (4 channels wide below one round of the 8-wide), 128 tiles
# by 64 channels and more the 16-channel form; 65 and 79 channels leave its last chunk 1 and 15.
@pytest.mark.parametrize("gaussian", [False, True], ids=["point", "gaussian"])
@pytest.mark.parametrize("nt,nchan,ncomp", [(2, 1, 1), (15, 3, 4), (16, 8, 5), (17, 9, 33), (33, 17, 31), (49, 31, 65),
                                            (128, 65, 3), (128, 79, 37), (113, 96, 34)])
def test_forms_vs_oracle(nt, nchan, ncomp, gaussian):
    check(nt, 167e6 + 40e3 * np.arange(nchan), sky(np.random.default_rng(ncomp), ncomp, gaussian))


# Steps above a thousandth of the frequency take the general second ratio; wide Gaussians on
# long baselines underflow; channels may descend.
@pytest.mark.parametrize("freqs", [80e6 + 1.28e6 * np.arange(21), (80e6 + 1.28e6 * np.arange(21))[::-1].copy(),
                                   (167e6 + 40e3 * np.arange(21))[::-1].copy(), np.array([180e6, 90e6, 200e6])],
                         ids=["wide", "wide-descending", "descending", "scattered"])
@pytest.mark.parametrize("axis", [1e-3, 0.2])
def test_gaussian_envelopes_vs_oracle(freqs, axis):
    check(21, freqs, sky(np.random.default_rng(5), 9, True, axis))


def test_envelope_forms_agree_with_the_baseline_kernel():
    """The 16-channel form, narrow and wide steps, against the baseline-per-lane kernel."""
    for df in (40e3, 1.28e6):
        rng = np.random.default_rng(3)
        xyzs, freqs = synthetic.tiles(rng, 128, 1500.0), 100e6 + df * np.arange(64)
        m = SkyModeller(NoBeam(), sky(rng, 40, True, 5e-3), 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                        synthetic.MWA_LAT_RAD)
        got = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)[2]
        _lib.call("sm_set_direct_variant", 1)
        try:
            want = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)[2]
        finally:
            _lib.call("sm_set_direct_variant", 0)
        assert rel_err(got, want) <= 1e-12


# Few blocks of many components take slices of the components (at least 128 each), the last one
# shorter or of a ragged stage.
@pytest.mark.parametrize("gaussian", [False, True], ids=["point", "gaussian"])
@pytest.mark.parametrize("nt,nchan,ncomp", [(2, 1, 257), (17, 9, 1500), (33, 17, 1025), (49, 2, 2099), (65, 28, 700)])
def test_component_slices_vs_oracle(nt, nchan, ncomp, gaussian):
    check(nt, 167e6 + 40e3 * np.arange(nchan), sky(np.random.default_rng(ncomp), ncomp, gaussian))
