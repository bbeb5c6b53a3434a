"""The precision path asked for FP32 visibilities alone, on either side of the lines where an FP64 kernel
stands in for Gaussians: above them the visibilities are bit for bit those beside FP64 ones (FP32
arithmetic both), below them they differ, within the path's bounds."""

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, NoBeam, SkyModeller
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_precision_f32_only import shapelets
from tests.test_gpu_tile_forms import sky
from tests.test_gpu_tile_pair_forms import form_of

pytestmark = pytest.mark.gpu


def run(m, shape, with_f64):
    v32 = torch.zeros(shape, dtype=torch.float32, device="cuda")
    v64 = torch.zeros(shape, dtype=torch.float64, device="cuda") if with_f64 else None
    _lib.call("sm_model_timestep_factored", m._h, 0.2, synthetic.MWA_LAT_RAD, 0, C.c_void_p(v32.data_ptr()),
              C.c_void_p(v64.data_ptr()) if with_f64 else None)
    torch.cuda.synchronize()
    return v32.cpu().numpy()


# 40 tiles: 5 tile-group pairs; 252 channels of 6 are 210 FP32 blocks, 768 channels 640.
@pytest.mark.parametrize("nchan,fp64", [(252, True), (768, False)])
def test_tile_pairs(nchan, fp64):
    rng = np.random.default_rng(40)
    xyzs, freqs = synthetic.tiles(rng, 40, 1000.0), 100e6 + 40e3 * np.arange(nchan)
    srclist = sky(rng, 21, True)
    assert (form_of(2, 40, freqs, 21)[0] >= 0) == fp64
    m = SkyModeller(NoBeam(), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0, synthetic.MWA_LAT_RAD)
    shape = (nchan, 780, 8)
    alone, both = run(m, shape, False), run(m, shape, True)
    assert np.array_equal(alone, both) == (not fp64)
    o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD), srclist)[1]
    assert np.abs(o64).max() > 0
    assert rel_err(alone, o64) <= 1e-6
    assert rel_err(alone, both) <= 2e-6


# 12 rows in 3 groups by 80 columns in 2: 6 blocks per 6 channels, so 696 and 702 blocks. Row-by-column
# visibilities alone: those of a tile with a dead dipole and one without.
@pytest.mark.parametrize("nchan,fp64", [(696, True), (697, False)])
def test_rows_by_columns(nchan, fp64):
    rng = np.random.default_rng(92)
    nt, dead = 92, 12
    xyzs, freqs = synthetic.tiles(rng, nt, 1000.0), 100e6 + 40e3 * np.arange(nchan)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    rows = np.zeros(nt, bool)
    for k in range(dead):
        delays[7 * k, k] = 32
        rows[7 * k] = True
    m = SkyModeller(AnalyticBeam(delays, gains), sky(rng, 9, True), 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                    synthetic.MWA_LAT_RAD)
    i, j = np.triu_indices(nt, 1)
    sel = rows[i] != rows[j]
    shape = (nchan, nt * (nt - 1) // 2, 8)
    alone, both = run(m, shape, False)[:, sel], run(m, shape, True)[:, sel]
    assert np.array_equal(alone, both) == (not fp64)
    m.model_timestep_with_device(0.2, synthetic.MWA_LAT_RAD, torch.zeros(shape, dtype=torch.float32, device="cuda"),
                                 v64 := torch.zeros(shape, dtype=torch.float64, device="cuda"))
    want = v64.cpu().numpy()[:, sel]
    assert np.abs(want).max() > 0
    assert rel_err(alone, want) <= 1e-6
    assert rel_err(alone, both) <= 2e-6


# 3160 baselines: 6 groups of 64 channels are below the line of few components, 7 above it.
@pytest.mark.parametrize("nchan,ncomp,fp64", [(384, 3, True), (385, 3, False), (385, 1, False), (385, 4, True)])
def test_few_shapelets(nchan, ncomp, fp64):
    rng = np.random.default_rng(nchan + ncomp)
    xyzs, freqs = synthetic.tiles(rng, 80, 1000.0), 100e6 + 40e3 * np.arange(nchan)
    m = SkyModeller(NoBeam(), shapelets(rng, ncomp), 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                    synthetic.MWA_LAT_RAD)
    shape = (nchan, 3160, 8)
    alone, both = run(m, shape, False), run(m, shape, True)
    assert np.array_equal(alone, both) == (not fp64)
    v64 = torch.zeros(shape, dtype=torch.float64, device="cuda")
    m.model_timestep_with_device(0.2, synthetic.MWA_LAT_RAD, torch.zeros_like(v64, dtype=torch.float32), v64)
    want = v64.cpu().numpy()
    assert np.abs(want).max() > 0
    assert rel_err(alone, want) <= 1e-6
    assert rel_err(both, want) <= 1e-6
