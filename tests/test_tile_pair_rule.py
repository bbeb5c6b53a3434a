"""The rules that pick the FP64 tile-pair kernel's form, and on the precision path the FP32 or the FP64
kernel, against measured times (us, 40 kHz channels, MI355X): what they pick is within 10% of the
fastest measured."""

import pytest

from mwa_hyperdrive_amd import _lib  # noqa: F401  (the library must be there)
from tests.test_gpu_tile_pair_forms import band, form_of

# (tiles, channels, components): {form: {slices: us}}, points and Gaussians.
POINTS = {
    (32, 64, 100): {0: {1: 38.5}, 1: {1: 38.9}, 2: {1: 26.2}, 3: {1: 19.1}, 4: {1: 15.7}},
    (64, 192, 2000): {0: {1: 527.8, 2: 441.5, 4: 362.3}, 1: {1: 532.4, 2: 463.6, 4: 364.4},
                      2: {1: 511.0, 2: 388.2, 4: 379.2}, 3: {1: 514.9}, 4: {1: 623.1}},
    (128, 24, 100): {0: {1: 38.1}, 1: {1: 39.6}, 2: {1: 28.5}, 3: {1: 34.5}, 4: {1: 31.1}},
    (128, 192, 2000): {0: {1: 1254.7, 2: 1271.2, 4: 1339.0}, 1: {1: 1286.7, 2: 1299.7, 4: 1384.8},
                       2: {1: 1340.7, 2: 1374.7, 4: 1421.9}, 3: {1: 1963.5}, 4: {1: 2235.4}},
    (128, 384, 2000): {0: {1: 2371.6, 2: 2526.1, 4: 2672.0}, 1: {1: 2427.0, 2: 2601.1, 4: 2771.1},
                       2: {1: 2607.0, 2: 2710.5, 4: 2829.5}, 3: {1: 3883.5}, 4: {1: 4417.6}},
    (256, 18, 100): {0: {1: 59.1}, 1: {1: 58.9}, 2: {1: 48.7}, 3: {1: 87.9}, 4: {1: 79.3}},
}
GAUSSIANS = {
    (32, 64, 100): {0: {1: 52.7}, 1: {1: 56.0}, 2: {1: 34.7}, 3: {1: 24.2}, 4: {1: 19.6}},
    (64, 192, 2000): {0: {1: 840.1, 2: 693.7, 4: 545.9}, 1: {1: 894.6, 2: 775.7, 4: 595.1},
                      2: {1: 816.7, 2: 635.8, 4: 622.3}, 3: {1: 777.8}, 4: {1: 1193.5}},
    (128, 24, 100): {0: {1: 53.3}, 1: {1: 56.9}, 2: {1: 37.1}, 3: {1: 44.7}, 4: {1: 49.7}},
    (128, 192, 500): {0: {1: 515.1, 2: 553.3, 3: 639.8}, 1: {1: 561.5, 2: 604.9, 3: 690.7},
                      2: {1: 591.9, 2: 637.0, 3: 712.1}, 3: {1: 805.2}, 4: {1: 1241.8}},
    (128, 384, 2000): {0: {1: 3696.1, 2: 3886.9, 4: 4087.8}, 1: {1: 4112.5, 2: 4349.8, 4: 4488.3},
                       2: {1: 4462.1, 2: 4622.2, 4: 4744.8}, 3: {1: 5911.1}, 4: {1: 9230.4}},
    (256, 48, 500): {0: {1: 526.5, 2: 554.4, 3: 634.5}, 1: {1: 563.2, 2: 603.2, 3: 683.1},
                     2: {1: 585.7, 2: 627.6, 3: 702.2}, 3: {1: 801.1}, 4: {1: 1227.8}},
}


@pytest.mark.parametrize("size", POINTS)
def test_points(size):
    check(False, size, POINTS[size])


@pytest.mark.parametrize("size", GAUSSIANS)
def test_gaussians(size):
    check(True, size, GAUSSIANS[size])


def check(gaussian, size, measured):
    nt, nchan, ncomp = size
    form, slices = form_of(gaussian, nt, band(nchan, 40e3), ncomp)
    times = measured[form]
    # A slice count between two measured ones is held to the slower of the two.
    below, above = max(s for s in times if s <= slices), min((s for s in times if s >= slices), default=None)
    assert above is not None, f"{slices} slices of form {form}: more than the most measured"
    assert max(times[below], times[above]) <= 1.1 * min(t for v in measured.values() for t in v.values())


@pytest.mark.parametrize("size", [(1000, 768, 200000), (1000, 192, 200000), (512, 48, 100000), (256, 192, 50000),
                                  (256, 48, 10000), (128, 96, 10000)])
@pytest.mark.parametrize("kind", [0, 1])
def test_slices_stay_within_their_workspace(kind, size):
    nt, nchan, ncomp = size
    _, slices = form_of(kind, nt, band(nchan, 40e3), ncomp)
    assert slices == 1 or slices * nchan * nt * (nt - 1) // 2 * 64 <= 4 << 30


# (tiles, channels, components): timesteps of Gaussians alone on the FP32 and on the FP64 kernel.
PRECISION = {
    (64, 192, 200): (159.0, 148.1), (64, 192, 5000): (2713.2, 1426.1), (64, 384, 200): (185.3, 211.9),
    (101, 96, 200): (170.2, 195.3), (101, 96, 5000): (2661.9, 2072.8), (128, 48, 1000): (564.5, 368.7),
    (128, 72, 200): (183.0, 206.9), (128, 72, 1000): (619.0, 555.0), (128, 132, 200): (218.6, 291.6),
    (128, 132, 5000): (3193.1, 3668.5), (200, 48, 1000): (699.7, 804.7), (256, 18, 200): (197.2, 222.0),
    (256, 18, 1000): (627.6, 719.7), (256, 36, 1000): (774.5, 1090.3), (256, 36, 5000): (3244.7, 4540.8),
    (32, 768, 1000): (604.6, 375.4), (230, 48, 10000): (10809, 8253), (230, 96, 10000): (15647, 17893),
    (230, 384, 10000): (54030, 64570), (128, 400, 10000): (18424, 19590), (180, 300, 6000): (16588, 19700),
    (60, 768, 20000): (25728, 19357), (256, 768, 2000): (23302, 28549),
}


@pytest.mark.parametrize("size", PRECISION)
def test_precision_path_gaussians(size):
    nt, nchan, ncomp = size
    fp32 = form_of(2, nt, band(nchan, 40e3), ncomp)[0] < 0
    assert PRECISION[size][0 if fp32 else 1] <= 1.1 * min(PRECISION[size])
