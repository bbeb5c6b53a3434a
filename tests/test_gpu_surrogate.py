"""Beam surrogate on the GPU: samples, gradients, Adam, FP32 / FP16 forward passes, training
and the exact-beam fallback, each checked against the CPU oracles (oracle/surrogate_oracle.py
for the network, orc_analytic_beam_jones for the exact beam)."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mwa_hyperdrive_amd import surrogate as sg
from mwa_hyperdrive_amd.modeller import analytic_beam_device
from oracle import oracle as orc
from oracle import surrogate_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [sg.POINTING, sg.INDEPENDENT])
def test_samples_match_oracle_beam_and_features(mode):
    x, y, raw = sg.samples(11, 1000, 300, want_raw=True, mode=mode)
    raw = raw.cpu().numpy()
    np.testing.assert_allclose(x.cpu().numpy(), so.features(raw), rtol=1e-6, atol=1e-7)
    exact = np.array([orc.analytic_beam(r[0], r[1], r[2], r[3:19].astype(np.uint32), r[19:51]) for r in raw])
    np.testing.assert_allclose(y.cpu().numpy(), exact, rtol=1e-6, atol=1e-7)
    # The distribution the generator promises.
    assert (raw[:, 1] >= 0).all() and (raw[:, 1] <= np.pi / 2).all()
    assert (raw[:, 2] >= 167e6).all() and (raw[:, 2] <= 197e6).all()
    delays = raw[:, 3:19]
    assert set(np.unique(delays)) <= set(range(32))
    if mode == sg.POINTING:
        # Pointing delays: smallest 0, linear in the dipole position to within rounding.
        assert (delays.min(axis=1) == 0).all()
        d = np.arange(16)
        xy = np.stack([(d % 4 - 1.5) * 1.1, (1.5 - d // 4) * 1.1, np.ones(16)], 1)
        for row in delays[:50]:
            if row.max() >= 31:
                continue
            coef, *_ = np.linalg.lstsq(xy, row, rcond=None)
            assert np.abs(xy @ coef - row).max() <= 1.0
    # Same (seed, index) -> same sample, whatever the batch it is drawn in.
    x2, _ = sg.samples(11, 1100, 5, mode=mode)
    np.testing.assert_array_equal(x2.cpu().numpy(), x.cpu().numpy()[100:105])


def test_gradients_match_oracle():
    s = sg.BeamSurrogate(seed=5)
    p = s.get_params().astype(np.float64)
    x, y = sg.samples(3, 0, 512)
    loss, g = s.gradients(x, y)
    ref_loss, ref_g = so.loss_and_grads(p, x.cpu().numpy(), y.cpu().numpy())
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    offs = np.cumsum([0] + [o * i + o for o, i in so.DIMS])
    for li in range(len(so.DIMS)):
        a, b = g[offs[li]:offs[li + 1]], ref_g[offs[li]:offs[li + 1]]
        err = np.abs(a - b).max() / np.abs(b).max()
        print(f"layer {li}: max grad err {err:.2e} of max |grad|")
        assert err <= 1e-4


def test_adam_step_matches_oracle():
    s = sg.BeamSurrogate(seed=6)
    p0 = s.get_params().astype(np.float64)
    x, y = sg.samples(4, 0, 256)
    _, g = s.gradients(x, y)
    s.train_step(x, y, 1e-3)
    p1 = s.get_params().astype(np.float64)
    ref, _, _ = so.adam_step(p0, g.astype(np.float64), np.zeros_like(p0), np.zeros_like(p0), 1, 1e-3)
    np.testing.assert_allclose(p1, ref, rtol=1e-6, atol=1e-7)


def test_forward_fp32_and_fp16_vs_oracle():
    s = sg.BeamSurrogate(seed=8)
    p = s.get_params().astype(np.float64)
    x, _ = sg.samples(9, 0, 1000)
    ref, _ = so.forward(p, x.cpu().numpy())
    scale = np.abs(ref).max()
    y32 = s.forward(x, fp16=False).cpu().numpy()
    y16 = s.forward(x, fp16=True).cpu().numpy()
    e32 = np.abs(y32 - ref).max() / scale
    e16 = np.abs(y16 - ref).max() / scale
    print(f"forward vs oracle: fp32 {e32:.2e}, fp16 {e16:.2e} of max |y|")
    assert e32 <= 1e-5
    assert e16 <= 1e-2


@pytest.mark.parametrize("hidden,depth", [(96, 2), (320, 6)])
def test_shaped_network_vs_oracle(hidden, depth):
    """Other widths and depths: parameter count, gradients and the FP32 forward against the
    oracle over the same shape; the fused FP16 forward is for 4 x 256 only."""
    s = sg.BeamSurrogate(seed=12, hidden=hidden, depth=depth)
    shape = so.dims(hidden, depth)
    assert s.num_params() == so.num_params(shape)
    p = s.get_params().astype(np.float64)
    x, y = sg.samples(13, 0, 384)
    loss, g = s.gradients(x, y)
    ref_loss, ref_g = so.loss_and_grads(p, x.cpu().numpy(), y.cpu().numpy(), shape)
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    assert np.abs(g - ref_g).max() <= 1e-4 * np.abs(ref_g).max()
    ref, _ = so.forward(p, x.cpu().numpy(), shape)
    y32 = s.forward(x, fp16=False).cpu().numpy()
    assert np.abs(y32 - ref).max() <= 1e-5 * np.abs(ref).max()
    with pytest.raises(Exception, match="4 x 256"):
        s.forward(x, fp16=True)


def test_training_reduces_error_and_fallback_is_exact():
    s = sg.BeamSurrogate(seed=1)
    xh, yh = sg.samples(99, 0, 20000)  # held out: another seed
    def err():
        d = s.forward(xh) - yh
        return d.pow(2).mean().sqrt().item(), d.abs().max().item()
    rms0, max0 = err()
    target_rms = yh.pow(2).mean().sqrt().item()
    info = s.train(n_samples=1 << 19, epochs=12, batch=2048, lr=2e-3)
    rms1, after = err()
    print(f"held-out |J err| (pointing delays): target rms {target_rms:.3e}; untrained rms {rms0:.3e} "
          f"max {max0:.3e} -> trained rms {rms1:.3e} max {after:.3e} ({info['steps']} steps, "
          f"{info['seconds']:.1f} s)")
    assert rms1 < 0.7 * min(rms0, target_rms)
    # Fallback: threshold 0 sends every tile to the exact beam; a huge threshold keeps all.
    rng = np.random.default_rng(2)
    delays = np.zeros((3, 16), np.uint32)
    delays[1] = rng.integers(0, 32, 16)
    gains = np.ones((3, 32))
    gains[2, 4] = 0.0
    freqs = np.array([170e6, 180e6, 190e6])
    az = torch.tensor(rng.uniform(0, 2 * np.pi, 700), device="cuda")
    za = torch.tensor(np.arccos(rng.uniform(0, 1, 700)), device="cuda")
    exact = analytic_beam_device(delays, gains, freqs, az, za)
    j0, nfb0 = s.beam(delays, gains, freqs, az, za, threshold=0.0)
    assert nfb0 == 3
    assert torch.equal(j0, exact)
    j1, nfb1 = s.beam(delays, gains, freqs, az, za, threshold=1e30)
    assert nfb1 == 0
    d = (j1 - exact).abs().max().item()
    print(f"surrogate beam max |J err| on 3 tiles: {d:.3e}")
    assert d < 10 * after + 1e-2


def test_modeller_with_surrogate_beam():
    """A C2-like mixed sky through the SkyModeller with the surrogate beam: threshold 0 gives
    the analytic-beam visibilities bit for bit (every tile falls back); an infinite threshold
    uses the network on every tile (no fallback), and the visibility error against the FP64
    oracle is bounded by the network's Jones error on the sky's own directions: each term
    J_p S J_q^H moves by at most ||S|| (2 ||J|| d + d^2) (Frobenius norms, d = max ||J_sur -
    J_exact||), phasors and Gaussian envelopes having modulus <= 1 (shapelets: sum |c_k|)."""
    from mwa_hyperdrive_amd import synthetic
    from mwa_hyperdrive_amd.modeller import AnalyticBeam, SkyModeller
    from tests.helpers import oracle_model, rel_err

    obs = synthetic.shrink(synthetic.config(2, scale=200 / 8000), tiles_n=24, chans=8, timesteps=1)
    beam = AnalyticBeam(obs.delays, obs.gains)
    m = SkyModeller(beam, obs.srclist, 0, obs.xyzs, obs.freqs, [], obs.phase_centre, 0.0, obs.latitude)
    ref32, _, ref64 = m.model_timestep(float(obs.lsts[0]), obs.latitude, want_f64=True)
    s = sg.BeamSurrogate(seed=1)
    s.train(n_samples=1 << 16, epochs=4, batch=4096, lr=2e-3)
    m.set_beam_surrogate(s, 0.0)
    v32, _, v64 = m.model_timestep(float(obs.lsts[0]), obs.latitude, want_f64=True)
    nfb = m.set_beam_surrogate(s, 1e30)
    assert nfb >= 1
    np.testing.assert_array_equal(v32, ref32)
    w32, _, w64 = m.model_timestep(float(obs.lsts[0]), obs.latitude, want_f64=True)
    assert m.set_beam_surrogate(None, 0.0) == 0  # the network served every tile
    o32, o64 = oracle_model(obs, 0)
    assert rel_err(ref64, o64) <= 1e-12
    # The network's Jones error on the directions and channels this sky uses.
    from oracle import oracle as orc
    from mwa_hyperdrive_amd.srclist import flat_components
    comps = flat_components(obs.srclist)
    lst = float(obs.lsts[0])
    azel = [orc.azel(lst - c.ra, c.dec, obs.latitude) for c in comps]
    az = torch.tensor([a for a, _ in azel], dtype=torch.float64, device="cuda")
    za = torch.tensor([np.pi / 2 - e for _, e in azel], dtype=torch.float64, device="cuda")
    d0, g0 = obs.delays[:1], obs.gains[:1]
    exact = analytic_beam_device(d0, g0, obs.freqs, az, za)
    sur, nfb = s.beam(d0, g0, obs.freqs, az, za, threshold=1e30)
    assert nfb == 0
    d = (sur - exact).pow(2).sum(-1).sqrt().max().item()
    jmax = exact.pow(2).sum(-1).sqrt().max().item()
    # ||S||_F = sqrt(2 (I^2 + Q^2 + U^2 + V^2)); a shapelet envelope is at most sum |c_k| (the
    # basis functions e^{-x^2/2} H_n(x) / sqrt(2^n n!) are bounded by 1, Cramer's inequality).
    from mwa_hyperdrive_amd.srclist import Shapelet
    ssum = 0.0
    for c in comps:
        w = sum(abs(v) for _, _, v in c.comp_type.coeffs) if isinstance(c.comp_type, Shapelet) else 1.0
        ssum += w * max(np.sqrt(2 * sum(x * x for x in orc.estimate_at_freq(c, f)[1:])) for f in obs.freqs)
    scale = np.abs(o64[..., 0::2] + 1j * o64[..., 1::2]).max()
    bound = ssum * (2 * jmax * d + d * d) / scale
    err = rel_err(w64, o64)
    print(f"surrogate-beam sky: rel vis err vs oracle {err:.3e} with the network on every tile (bound "
          f"{bound:.3e} from max |dJ| {d:.3e}); exact beam {rel_err(ref64, o64):.3e}")
    assert np.isfinite(w64).all()
    assert 0.0 < err <= bound


# The weight gradients' batch slices: below one slice, one row over, ragged last slices and empty
# ones; widths of one and several 64-wide tiles. A component of an FP32 sum of n products is within
# about sqrt(n) 6e-8 of its largest, well below 1e-4 of the layer's largest gradient.
@pytest.mark.parametrize("hidden,n", [(256, 1), (256, 127), (256, 129), (256, 4097), (65, 1000), (7, 8193)])
def test_gradient_slices_vs_fp64(hidden, n):
    s = sg.BeamSurrogate(seed=5, hidden=hidden, depth=2)
    flat = torch.tensor(s.get_params(), dtype=torch.float64, requires_grad=True)
    x, y = sg.samples(3, 0, n)
    loss, g = s.gradients(x, y)
    h, o, dims = x.cpu().double(), 0, [53, hidden, hidden, 8]
    edges = [0]
    for i, (a, b) in enumerate(zip(dims, dims[1:])):
        w = flat[o:o + a * b].reshape(b, a)
        h = h @ w.T + flat[o + a * b:o + a * b + b]
        h = torch.nn.functional.silu(h) if i < 2 else h
        edges += [o + a * b, o + a * b + b]
        o += a * b + b
    ref = ((h - y.cpu().double()) ** 2).mean()
    ref.backward()
    assert abs(loss - ref.item()) <= 1e-5 * ref.item()
    want = flat.grad.numpy()
    for lo, hi in zip(edges, edges[1:]):
        assert np.abs(g[lo:hi] - want[lo:hi]).max() <= 1e-4 * np.abs(want[lo:hi]).max()
