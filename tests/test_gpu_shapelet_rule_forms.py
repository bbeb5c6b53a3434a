"""Shapelets in FP64 on every form that the table edges crossed select, at full and ragged channel groups,
against the oracle at 1e-12 of max|V|: through a modeller, whose rule takes the array and the components'
sizes, and (per-tile beams) through the drop-in, which samples them on the device."""

import ctypes as C
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, SkyModeller
from mwa_hyperdrive_amd.srclist import FluxDensity, PowerLaw, Shapelet, Source, SourceComponent, SourceList
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_abi import Buckets, addresses, dt, make_sky, p
from tests.test_shapelet_rule import edges_per_hz, form_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dead,nchan,df,axis,form", [
    (0, 129, 20e3, 1e-3, 0), (0, 128, 40e3, 5e-4, 0), (0, 63, 160e3, 2e-3, 1), (0, 64, 320e3, 1e-3, 1),
    (0, 31, 40e3, 1e-3, 2), (0, 33, 1.28e6, 5e-3, 1), (3, 129, 20e3, 2e-4, 0), (3, 64, 160e3, 6e-4, 1),
    (3, 65, 80e3, 5e-4, 2), (3, 24, 80e3, 1e-3, 2), (3, 12, 1.28e6, 1e-3, 3), (3, 31, 640e3, 1e-3, 3),
    (3, 64, 160e3, 3e-3, 3), (3, 97, 160e3, 3e-3, 3)])
def test_form_vs_oracle(dead, nchan, df, axis, form):
    rng = np.random.default_rng(nchan)
    nt = 9
    ra, dec = synthetic.cap_positions(rng, 40, 10.0)
    comps = [SourceComponent(float(ra[k]), float(dec[k]), Shapelet(axis, 0.6 * axis, 0.3 * k, [
        (int(rng.integers(0, 11)), int(rng.integers(0, 11)), float(rng.normal())) for _ in range(12)]),
        PowerLaw(-0.8, FluxDensity(150e6, 1.0 + k, 0.1, -0.2, 0.3))) for k in range(40)]
    srclist = SourceList([("s", Source(comps))])
    xyzs, freqs = synthetic.tiles(rng, nt, 1500.0), 100e6 + df * np.arange(nchan)
    xyz = np.asarray(xyzs)
    rms = np.sqrt(2.0 * ((xyz - xyz.mean(axis=0)) ** 2).sum(axis=1).mean())
    assert form_of(dead > 0, nchan, df, edges_per_hz(rms, 1.6 * axis), 40) == form
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    for k in range(dead):
        delays[2 * k, k] = 32
    m = SkyModeller(AnalyticBeam(delays, gains), srclist, 0, xyzs, freqs, [], synthetic.PHASE_CENTRE, 0.0,
                    synthetic.MWA_LAT_RAD)
    vis, _, vis64 = m.model_timestep(0.2, synthetic.MWA_LAT_RAD, want_f64=True)
    o32, o64 = orc.model_timestep(orc.Obs(xyzs, freqs, synthetic.PHASE_CENTRE, 0.2, synthetic.MWA_LAT_RAD,
                                          beam="analytic", delays=delays, gains=gains), srclist)
    assert np.abs(o64).max() > 0
    assert rel_err(vis64, o64) <= 1e-12
    assert rel_err(vis, o32) <= 2e-7  # one FP32 rounding on each side


@pytest.mark.parametrize("nchan,df", [(20, 640e3), (65, 40e3)])
def test_dropin_with_per_tile_beams_vs_oracle(nchan, df):
    """Sizes at which the drop-in samples the edges: 12 components on 4560 baselines, above 1 MHz."""
    rng = np.random.default_rng(nchan)
    nt, lst, pc, freqs = 96, 0.3, synthetic.PHASE_CENTRE, 100e6 + df * np.arange(nchan)
    xyzs = synthetic.tiles(rng, nt, 1500.0)
    b = Buckets(make_sky(rng, 4, freqs, "shapelet"), freqs, pc, xyzs, lst)
    delays, gains = np.zeros((nt, 16), np.uint32), np.ones((nt, 32))
    delays[3, 5] = delays[70, 0] = 32
    n_u, tile_map = orc.unique_tiles(nt, [], delays, gains)
    az_za = [orc.azel(lst - c.ra, c.dec, synthetic.MWA_LAT_RAD) for c in b.order]
    jones = dt(np.array([[[orc.analytic_beam(az, math.pi / 2 - el, f, delays[t], gains[t]) for az, el in az_za]
                          for f in freqs] for t in [list(tile_map).index(u) for u in range(n_u)]]))
    nbl = nt * (nt - 1) // 2
    uvw = dt(orc.cross_uvws(xyzs, lst - pc[0], pc[1]))
    a, keep = addresses(freqs, nbl, nchan, tile_map, np.arange(nchan, dtype=np.int32), np.arange(nt),
                        dt(orc.shapelet_basis_table()))
    args = []
    for name in ("pl", "cpl", "list"):
        fields = ["lmn", "fds"] + (["sis"] if name != "list" else []) + (["qs"] if name == "cpl" else [])
        args += [b.n[name]] + [b.g(name + "_" + f) for f in fields + ["gps", "uvs", "coeffs", "ncoeffs"]]
    vis = torch.zeros((nchan, nbl, 8), dtype=torch.float32, device="cuda")
    vis64 = torch.zeros((nchan, nbl, 8), dtype=torch.float64, device="cuda")
    _lib.call("sm_model_shapelets_f64", C.byref(_lib.Shapelets(*args)), C.byref(a), p(uvw), p(jones), p(vis), p(vis64))
    torch.cuda.synchronize()
    o64 = orc.model_timestep(orc.Obs(xyzs, freqs, pc, lst, synthetic.MWA_LAT_RAD, beam="analytic", delays=delays,
                                     gains=gains), SourceList([("s", Source(b.order))]), mask=4)[1]
    assert np.abs(o64).max() > 0
    assert rel_err(vis64.cpu().numpy(), o64) <= 1e-12
