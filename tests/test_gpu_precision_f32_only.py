"""The precision path asked for FP32 visibilities alone, which takes FP64 kernels for some types and
sizes: both sides of those lines, against the oracle at the path's bound, and against its own FP32
visibilities where FP64 ones are asked for too."""

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, NoBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, PowerLaw, Shapelet, Source, SourceComponent, SourceList
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_tile_forms import sky

pytestmark = pytest.mark.gpu


def shapelets(rng, n):
    ra, dec = synthetic.cap_positions(rng, n, 10.0)
    comps = []
    for k in range(n):
        cf = [(int(rng.integers(0, 8)), int(rng.integers(0, 8)), float(rng.normal())) for _ in range(6)]
        comps.append(SourceComponent(float(ra[k]), float(dec[k]), Shapelet(1e-3, 5e-4, 0.3 * k, cf),
                                     PowerLaw(-0.8, FluxDensity(150e6, 1.0 + k, 0.1, -0.2, 0.3))))
    return SourceList([("s", Source(comps))])


# 33 tiles: 6 tile-group pairs, so 252 and 258 blocks of 6 channels at 252 and 253 channels. Steps of 160 kHz
# over 64 and 65 channels lie on both sides of the shapelets' line. dead: tiles with their own beams.
@pytest.mark.parametrize("kind,nt,nchan,df,dead", [("gaussian", 9, 13, 40e3, 0), ("gaussian", 40, 252, 40e3, 0),
                                                   ("gaussian", 40, 253, 40e3, 0), ("gaussian", 12, 13, 40e3, 4),
                                                   ("shapelet", 5, 33, 40e3, 0), ("shapelet", 5, 64, 160e3, 0),
                                                   ("shapelet", 5, 65, 160e3, 0), ("shapelet", 6, 33, 40e3, 3)])
def test_f32_visibilities_alone(kind, nt, nchan, df, dead):
    rng = np.random.default_rng(nt)
    srclist = sky(rng, 21, True) if kind == "gaussian" else shapelets(rng, 7)
    xyzs, freqs = synthetic.tiles(rng, nt, 1000.0), 100e6 + df * np.arange(nchan)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    for t in range(dead):
        delays[2 * t, t] = 32
    m = SkyModeller(AnalyticBeam(delays, gains) if dead else NoBeam(), srclist, 0, xyzs, freqs, [],
                    synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    shape = (nchan, nt * (nt - 1) // 2, 8)

    def run(with_f64):
        v32 = torch.zeros(shape, dtype=torch.float32, device="cuda")
        v64 = torch.zeros(shape, dtype=torch.float64, device="cuda") if with_f64 else None
        _lib.call("sm_model_timestep_factored", m._h, 0.2, synthetic.MWA_LAT_RAD, 0, C.c_void_p(v32.data_ptr()),
                  C.c_void_p(v64.data_ptr()) if with_f64 else None)
        torch.cuda.synchronize()
        return v32.cpu().numpy()

    kw = {"beam": "analytic", "delays": delays, "gains": gains} if dead else {}
    o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD, **kw), srclist)[1]
    assert np.abs(o64).max() > 0
    alone, both = run(False), run(True)
    assert rel_err(alone, o64) <= 1e-6
    assert rel_err(both, o64) <= 1e-6
    assert rel_err(alone, both) <= 2e-6
