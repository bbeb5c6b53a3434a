"""Every form of the FP64 tile-pair kernel, unsliced and with slices of the components, at the first
and the last remainder of its channel chunk and ragged component counts, over all tiles and over those
of a beam class (tile map): against the baseline-per-lane kernel at the parity bound 1e-12 of max|V|,
and with FP32 visibilities alone against those beside FP64 ones, bit for bit. Few components, whose
FP32 visibilities alone the vector kernel forms, at both ends of its range.

The sizes are the cheapest of a grid that take the form, by the kernel's own rule."""

import ctypes as C
import functools

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import _lib, synthetic
from mwa_hyperdrive_amd.modeller import AnalyticBeam, NoBeam, SkyModeller
from oracle import oracle as orc
from tests.helpers import rel_err
from tests.test_gpu_abi import Buckets, addresses, dt, make_sky, p
from tests.test_gpu_tile_forms import sky

WIDTH = (16, 8, 8, 8, 4)  # channels of forms 0 .. 4
TILES = (2, 16, 17, 33, 49, 64, 65, 96, 113, 128, 161, 200, 256)
COMPS = (31, 34, 101, 257, 513, 1025, 2051)


def band(nchan, step):  # a step of 160 kHz is wide: more than a thousandth of the frequency
    return 100e6 + step * np.arange(nchan)


def form_of(kind, nt, freqs, ncomp, want_f64=None):
    form, slices = C.c_int32(), C.c_int32()
    freqs = np.ascontiguousarray(freqs)
    want_f64 = kind != 2 if want_f64 is None else want_f64
    _lib.call("sm_tiles_form", int(kind), int(want_f64), nt, len(freqs), freqs.ctypes.data_as(C.c_void_p), ncomp,
              C.byref(form), C.byref(slices))
    return form.value, slices.value


@functools.lru_cache(maxsize=None)
def cheapest(gaussian, form, sliced, rem):
    """(tiles, channels, components) of the least work that take the form with `rem` channels in the
    last chunk."""
    best = None
    for nt in TILES:
        for m in (0, 1, 2, 3, 4, 6, 8, 12, 16, 24, 36, 48):
            nchan = m * WIDTH[form] + rem
            for n in COMPS:
                work = nt * (nt - 1) * nchan * n
                if (best is None or work < best[0]) and (n >= 256 or not sliced):
                    got = form_of(gaussian, nt, band(nchan, 40e3), n)
                    if got[0] == form and (got[1] > 1) == sliced:
                        best = (work, nt, nchan, n)
    return best and best[1:]


FORMS = [(f, False) for f in range(5)] + [(f, True) for f in range(3)]


@pytest.mark.parametrize("gaussian", [False, True], ids=["point", "gaussian"])
@pytest.mark.parametrize("form,sliced", FORMS)
def test_every_form_has_a_size(form, sliced, gaussian):
    for rem in (1, WIDTH[form] - 1):
        assert cheapest(gaussian, form, sliced, rem) is not None


def modeller(nt, dead, ncomp, gaussian, freqs, seed):
    """nt tiles of one beam (no beam without dead dipoles) and `dead` tiles of other beams."""
    rng = np.random.default_rng(seed)
    total = nt + dead
    delays, gains = np.zeros((total, 16), np.uint32), np.ones((total, 32))
    for k in range(dead):
        delays[k * (total // 3), k] = 32
    return SkyModeller(AnalyticBeam(delays, gains) if dead else NoBeam(), sky(rng, ncomp, gaussian, 5e-3), 0,
                       synthetic.tiles(rng, total, 1500.0), freqs, [], synthetic.PHASE_CENTRE, 0.0,
                       synthetic.MWA_LAT_RAD), (len(freqs), total * (total - 1) // 2, 8)


def run(m, shape, with_f64):
    v32 = torch.zeros(shape, dtype=torch.float32, device="cuda")
    v64 = torch.zeros(shape, dtype=torch.float64, device="cuda") if with_f64 else None
    m.model_timestep_with_device(0.2, synthetic.MWA_LAT_RAD, v32, v64)
    torch.cuda.synchronize()
    return v32, v64


def baseline_kernel(m, shape):
    _lib.call("sm_set_direct_variant", 1)
    try:
        return [v.cpu().numpy() for v in run(m, shape, True)]
    finally:
        _lib.call("sm_set_direct_variant", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("mapped", [False, True], ids=["all", "class"])
@pytest.mark.parametrize("kind,step", [("point", 40e3), ("gaussian", 40e3), ("gaussian", 160e3)])
@pytest.mark.parametrize("last", [False, True], ids=["rem1", "rem-1"])
@pytest.mark.parametrize("form,sliced", FORMS)
def test_form_vs_baseline_kernel(form, sliced, last, kind, step, mapped):
    gaussian = kind == "gaussian"
    nt, nchan, ncomp = cheapest(gaussian, form, sliced, WIDTH[form] - 1 if last else 1)
    freqs = band(nchan, step)
    assert form_of(gaussian, nt, freqs, ncomp) == form_of(gaussian, nt, band(nchan, 40e3), ncomp)
    m, shape = modeller(nt, 3 if mapped else 0, ncomp, gaussian, freqs, nt + form)
    v32, v64 = run(m, shape, True)
    alone, _ = run(m, shape, False)
    if mapped:  # pairs of two tiles outside the class sum by atomics, in any order
        assert rel_err(alone.cpu().numpy(), v32.cpu().numpy()) <= 2e-7
    else:
        assert torch.equal(alone, v32)
    w32, w64 = baseline_kernel(m, shape)
    assert np.abs(w64).max() > 0
    assert rel_err(v64.cpu().numpy(), w64) <= 1e-12
    assert rel_err(v32.cpu().numpy(), w32) <= 2e-7  # one FP32 rounding on each side


# 5 pairs of tile groups of 40 tiles, 32 of 117, in chunks of 8 (points) and 6 channels (Gaussians).
@pytest.mark.gpu
@pytest.mark.parametrize("mapped", [False, True], ids=["all", "class"])
@pytest.mark.parametrize("gaussian,nt,nchan,ncomp,few", [
    (False, 40, 633, 1, True), (False, 40, 632, 1, False), (False, 40, 633, 20, True), (False, 40, 633, 21, False),
    (False, 117, 145, 28, True), (False, 117, 145, 29, False), (False, 117, 144, 28, False),
    (True, 40, 475, 1, True), (True, 40, 474, 1, False), (True, 117, 95, 18, True), (True, 117, 95, 19, False)])
def test_few_components_vs_baseline_kernel(gaussian, nt, nchan, ncomp, few, mapped):
    freqs = band(nchan, 40e3)
    assert (form_of(gaussian, nt, freqs, ncomp, want_f64=False)[0] == 5) == few
    assert form_of(gaussian, nt, freqs, ncomp)[0] != 5
    m, shape = modeller(nt, 3 if mapped else 0, ncomp, gaussian, freqs, nt + ncomp)
    w32, w64 = baseline_kernel(m, shape)
    alone = run(m, shape, False)[0].cpu().numpy()
    assert np.abs(w64).max() > 0
    assert rel_err(alone, w32) <= 2e-7  # one FP32 rounding on each side


# The drop-ins have fixed chunks instead of tables of them.
@pytest.mark.gpu
@pytest.mark.parametrize("kind,nchan", [("point", 634), ("gaussian", 476)])
def test_few_components_of_dropins_vs_baseline_kernel(kind, nchan):
    rng = np.random.default_rng(nchan)
    nt, lst, pc, freqs = 40, 0.3, synthetic.PHASE_CENTRE, band(nchan, 40e3)
    assert form_of(kind == "gaussian", nt, freqs, 3, want_f64=False)[0] == 5
    xyzs = synthetic.tiles(rng, nt, 1000.0)
    b = Buckets(make_sky(rng, 1, freqs, kind), freqs, pc, xyzs, lst)
    uvw = dt(orc.cross_uvws(xyzs, lst - pc[0], pc[1]))
    a, keep = addresses(freqs, len(uvw), 1, np.zeros(nt), np.zeros(nchan), np.arange(nt))
    args = []
    for name in ("pl", "cpl", "list"):
        fields = ["lmn", "fds"] + (["sis"] if name != "list" else []) + (["qs"] if name == "cpl" else [])
        args += [b.n[name]] + [b.g(name + "_" + f) for f in fields + ([] if kind == "point" else ["gps"])]
    comps = (_lib.Points if kind == "point" else _lib.Gaussians)(*args)

    def call():
        vis = torch.zeros((nchan, len(uvw), 8), dtype=torch.float32, device="cuda")
        _lib.call("sm_model_%ss_f64" % kind, C.byref(comps), C.byref(a), p(uvw), None, p(vis), None)
        torch.cuda.synchronize()
        return vis.cpu().numpy()

    alone = call()
    _lib.call("sm_set_direct_variant", 1)
    try:
        want = call()
    finally:
        _lib.call("sm_set_direct_variant", 0)
    assert np.abs(want).max() > 0
    assert rel_err(alone, want) <= 2e-7  # one FP32 rounding on each side
