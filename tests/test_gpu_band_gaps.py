"""Bands with gaps: a run of two or three channels across a gap of the band is as accurate as any other.

One component, so that each visibility is a phasor times a real amplitude, on tiles within 3 km. Per
channel, the rms difference to the oracle is held to 2.5 times the rms error E of a direct FP64
evaluation of these phases (numpy, against 80-bit floats): the oracle is such an evaluation, the
kernels' phase is the difference of two tiles' (each of about that error), sqrt(1 + 2) = 1.7 in all."""

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, NoBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, Gaussian, Point, PowerLaw, Source, SourceComponent, SourceList
from oracle import oracle as orc
from tests.test_gpu_tile_pair_forms import WIDTH, form_of

pytestmark = pytest.mark.gpu
C_M_S = 299792458.0


def direct_error(uvws, ra, dec, freqs):
    """E per channel: FP64 against 80-bit floats for the same UVWs and direction cosines."""
    ra0, dec0 = synthetic.PHASE_CENTRE
    d = ra - ra0
    l = math.cos(dec) * math.sin(d)
    m = math.sin(dec) * math.cos(dec0) - math.cos(dec) * math.sin(dec0) * math.cos(d)
    n = math.sin(dec) * math.sin(dec0) + math.cos(dec) * math.cos(dec0) * math.cos(d) - 1.0
    lmn = 2.0 * math.pi * np.array([l, m, n])
    theta = uvws[:, 0] * lmn[0] + uvws[:, 1] * lmn[1] + uvws[:, 2] * lmn[2]
    wide = np.longdouble
    exact = sum(uvws[:, k].astype(wide) * wide(lmn[k]) for k in range(3))
    out = []
    for f in freqs:
        a, b = theta * (f / C_M_S), exact * wide(f) / wide(C_M_S)
        z = np.exp(1j * a) - (np.cos(b).astype(np.float64) + 1j * np.sin(b).astype(np.float64))
        out.append(np.sqrt((np.abs(z) ** 2).mean()))
    return np.array(out)


TWO = np.array([75e6, 300e6])
THREE = np.array([80e6, 180e6, 280e6])
TENS = np.concatenate([100e6 + 40e3 * np.arange(9), 150e6 + 40e3 * np.arange(17), 230e6 + 40e3 * np.arange(9)])
LONG = np.concatenate([100e6 + 40e3 * np.arange(353), 280e6 + 40e3 * np.arange(353)])  # 16-channel runs and a pair


# faint: components of no weight, with which the sizes take the channel width (None: row tiles by the
# tiles of the shared beam, 8 channels wide).
@pytest.mark.parametrize("freqs,nt,faint,gaussian,width", [
    (TWO, 40, 0, False, 4), (TWO, 128, 0, False, None), (THREE, 40, 0, False, 4), (THREE, 128, 0, True, None),
    (TENS, 128, 40, False, 8), (TENS, 128, 0, False, None), (LONG, 128, 40, True, 16), (LONG, 128, 40, False, 8)],
    ids=["two", "two-rows", "three", "three-rows", "tens", "tens-rows", "long", "long-points"])
def test_channels_on_both_sides_of_a_gap(freqs, nt, faint, gaussian, width):
    rng = np.random.default_rng(7)
    ra, dec = 0.21, synthetic.PHASE_CENTRE[1] + 0.12
    comps = [SourceComponent(ra, dec, Gaussian(1e-9, 1e-9, 0.0) if gaussian else Point(),
                             PowerLaw(-0.8, FluxDensity(150e6, w, 0.0, 0.0, 0.0)))
             for w in [1.0] + [1e-30] * faint]
    srclist = SourceList([("s", Source(comps))])
    xyzs = synthetic.tiles(rng, nt, 3000.0)
    kw, beam = {}, NoBeam()
    if width is None:
        delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
        for k in range(12):
            delays[(k * 37) % nt, k % 3] = 32
        kw, beam = {"beam": "analytic", "delays": delays, "gains": gains}, AnalyticBeam(delays, gains)
    else:
        assert WIDTH[form_of(gaussian, nt, freqs, len(comps))[0]] == width
    m = SkyModeller(beam, srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    _, uvws, got = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    want = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD, **kw),
                              SourceList([("s", Source(comps[:1]))]))[1]
    nbl = nt * (nt - 1) // 2
    got, want = (np.asarray(v).reshape(len(freqs), nbl, 4, 2)[:, :, 0] for v in (got, want))
    diff = np.sqrt(((got - want) ** 2).sum(-1) / (want ** 2).sum(-1))
    if width is None:  # pairs of a row tile and one of the shared beam
        dead = (delays == 32).any(axis=1)
        i, j = np.triu_indices(nt, 1)
        diff = diff[:, dead[i] != dead[j]]
    error = direct_error(np.asarray(uvws), ra, dec, freqs)
    rms = np.sqrt((diff ** 2).mean(axis=1))
    assert (rms <= 2.5 * error).all()
