"""FP32 visibilities asked for alone carry the bits of those asked for beside FP64 ones, on the row-by-column
kernel (one launch and in slices of the components, ragged chunks) and on every form of the shapelet
kernels. The tile-pair kernel's forms are compared alike in test_gpu_tile_pair_forms."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, PowerLaw, Shapelet, Source, SourceComponent, SourceList
from tests.test_gpu_tile_forms import sky
from tests.test_shapelet_rule import edges_per_hz, form_of

pytestmark = pytest.mark.gpu


def both_ways(srclist, xyzs, freqs, dead):
    """FP32 visibilities alone and beside FP64 ones; `dead` tiles have their own beams."""
    nt = len(xyzs)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    rows = np.zeros(nt, bool)
    for k in range(dead):
        delays[2 * k, k] = 32
        rows[2 * k] = True
    m = SkyModeller(AnalyticBeam(delays, gains), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                    synthetic.MWA_LAT_RAD)
    out = []
    for with_f64 in (False, True):
        v32 = torch.zeros((len(freqs), nt * (nt - 1) // 2, 8), dtype=torch.float32, device="cuda")
        m.model_timestep_with_device(0.2, synthetic.MWA_LAT_RAD, v32,
                                     torch.zeros_like(v32, dtype=torch.float64) if with_f64 else None)
        torch.cuda.synchronize()
        out.append(v32.cpu().numpy())
    return out, rows


@pytest.mark.parametrize("gaussian", [False, True], ids=["point", "gaussian"])
@pytest.mark.parametrize("nt,nchan,ncomp", [(92, 17, 9), (40, 7, 3001)], ids=["whole", "slices"])
def test_rows_by_columns(nt, nchan, ncomp, gaussian):
    rng = np.random.default_rng(nt)
    (alone, both), rows = both_ways(sky(rng, ncomp, gaussian), synthetic.tiles(rng, nt, 1000.0),
                                    100e6 + 40e3 * np.arange(nchan), 6)
    i, j = np.triu_indices(nt, 1)
    sel = rows[i] != rows[j]
    assert np.abs(alone[:, sel]).max() > 0
    assert np.array_equal(alone[:, sel], both[:, sel])


@pytest.mark.parametrize("dead,nchan,df,axis,form", [
    (0, 129, 20e3, 1e-3, 0), (0, 64, 320e3, 1e-3, 1), (0, 31, 40e3, 1e-3, 2), (3, 129, 20e3, 2e-4, 0),
    (3, 64, 160e3, 6e-4, 1), (3, 65, 80e3, 5e-4, 2), (3, 31, 640e3, 1e-3, 3)])
def test_shapelets(dead, nchan, df, axis, form):
    rng = np.random.default_rng(nchan)
    ra, dec = synthetic.cap_positions(rng, 40, 10.0)
    comps = [SourceComponent(float(ra[k]), float(dec[k]), Shapelet(axis, 0.6 * axis, 0.3 * k, [
        (int(rng.integers(0, 11)), int(rng.integers(0, 11)), float(rng.normal())) for _ in range(12)]),
        PowerLaw(-0.8, FluxDensity(150e6, 1.0 + k, 0.1, -0.2, 0.3))) for k in range(40)]
    xyzs = synthetic.tiles(rng, 9, 1500.0)
    xyz = np.asarray(xyzs)
    rms = np.sqrt(2.0 * ((xyz - xyz.mean(axis=0)) ** 2).sum(axis=1).mean())
    assert form_of(dead > 0, nchan, df, edges_per_hz(rms, 1.6 * axis), 40) == form
    (alone, both), _ = both_ways(SourceList([("s", Source(comps))]), xyzs, 100e6 + df * np.arange(nchan), dead)
    assert np.abs(alone).max() > 0
    assert np.array_equal(alone, both)
