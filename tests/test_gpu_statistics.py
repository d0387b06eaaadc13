"""Statistical parity with noise and stochastic pulses on: mean and variance of outputs and of the
weight change over 64 seeds must agree between the GPU path and the CPU oracle within 3 sigma, plus
size-independent properties at the full benchmark size (1024 x 1024, batch 256)."""
import numpy as np
import pytest
import torch

from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles
from helpers import build_pair, config2, config2_data, constant_step, io_params, make_meta, noise_free_io, soft_bounds

pytestmark = pytest.mark.gpu

N_SEEDS = 64


def cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def compare_moments(a, b, what, variance_slack=0.01):
    """a, b: [seeds, ...] samples of the same quantity from two implementations.

    Per element: z = (mean_a - mean_b) / sqrt((var_a + var_b) / n) must exceed 3 no more often than chance
    allows; pooled over all elements the mean of z must vanish within 4 standard errors and the summed
    variances must agree within 3 sigma of the summed-variance estimator (+ variance_slack of the larger sum: 1 % where
    the variance is dominated by the random pulse trains, none where only the cycle-to-cycle noise is random)."""
    n = a.shape[0]
    a = a.reshape(n, -1).astype(np.float64)
    b = b.reshape(n, -1).astype(np.float64)
    ma, mb = a.mean(0), b.mean(0)
    va, vb = a.var(0, ddof=1), b.var(0, ddof=1)
    live = (va + vb) > 0
    assert live.mean() > 0.5, what
    z = (ma[live] - mb[live]) / np.sqrt((va[live] + vb[live]) / n)
    frac = np.mean(np.abs(z) > 3.0)
    assert frac < 0.012, (what, "fraction of elements beyond 3 sigma", frac)  # 0.27 % for a Gaussian, t-tails allowed for
    assert abs(z.mean()) < 4.0 / np.sqrt(z.size) + 0.01, (what, "pooled mean shift (in sigma)", z.mean())
    # elements whose mean differs although neither implementation shows any variance would be a deterministic bug
    dead = ~live
    assert np.allclose(ma[dead], mb[dead], atol=1e-5), what
    # variance: pooled ratio; the estimator's own spread from the per-element fourth moments
    sa, sb = va[live].sum(), vb[live].sum()
    m4a = ((a[:, live] - ma[live]) ** 4).mean(0)
    m4b = ((b[:, live] - mb[live]) ** 4).mean(0)
    sd = np.sqrt(((m4a - va[live] ** 2).clip(0) + (m4b - vb[live] ** 2).clip(0)).sum() / n)
    assert abs(sa - sb) < 3.0 * sd + variance_slack * max(sa, sb), (what, "pooled variance", sa, sb, sd)
    ratio = np.log(va[live & (va > 0) & (vb > 0)] / vb[live & (va > 0) & (vb > 0)])
    assert np.mean(np.abs(ratio) > 1.5) < 0.02, (what, "per-element variance ratio tails")


def test_forward_backward_output_moments_over_64_seeds(gpu_device):
    rng = np.random.default_rng(0)
    x_size, d_size, batch = 768, 128, 32
    f_io = io_params(out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax,
                     bound_management=dv.BoundManagementType.Iterative)
    b_io = io_params(out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax)
    meta = make_meta(f_io, b_io)
    dev = soft_bounds(construction_seed=123, enforce_consistency=True)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    w = rng.uniform(-0.6, 0.6, (d_size, x_size)).astype(np.float32)
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    gpu = tiles.CudaAnalogTile(host)
    x = rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)
    d = (0.05 * rng.standard_normal((batch, d_size))).astype(np.float32)
    xg, dg = cuda(x), cuda(d)
    yg, yo, bg, bo, rg, ro = [], [], [], [], [], []
    for s in range(N_SEEDS):
        gpu.set_seed(1000 + s)
        orc.set_seed(1 + s)
        yg.append(gpu.forward(xg, False, False, False, False, False).cpu().numpy())
        rg.append(gpu.get_bm_rounds(batch).numpy())
        yo.append(orc.forward(x))
        ro.append(orc.bm_rounds(batch))
        bg.append(gpu.backward(dg, False, False, False, False).cpu().numpy())
        bo.append(orc.backward(d))
    assert np.mean(ro) > 1.5  # bound management is exercised
    assert abs(np.mean(rg) - np.mean(ro)) < 0.05
    compare_moments(np.stack(yg), np.stack(yo), "forward outputs")
    compare_moments(np.stack(bg), np.stack(bo), "backward outputs")
    # two GPU calls with the same seed give the same numbers, another seed does not
    gpu.set_seed(5)
    y1 = gpu.forward(xg, False, False, False, False, False).cpu().numpy()
    gpu.set_seed(5)
    y2 = gpu.forward(xg, False, False, False, False, False).cpu().numpy()
    gpu.set_seed(6)
    y3 = gpu.forward(xg, False, False, False, False, False).cpu().numpy()
    assert np.array_equal(y1, y2) and not np.array_equal(y1, y3)


@pytest.mark.parametrize("device,um", [("soft", True), ("constant", False), ("constant", True)])
def test_update_weight_change_moments_over_64_seeds(gpu_device, device, um):
    rng = np.random.default_rng(1)
    x_size, d_size, batch = 128, 96, 24
    meta = make_meta(desired_bl=31, update_management=um, update_bl_management=um)
    kw = dict(dw_min=0.001, dw_min_dtod=0.3, dw_min_std=0.3, up_down_dtod=0.01, w_max_dtod=0.3, w_min_dtod=0.3,
              construction_seed=123, enforce_consistency=True)
    dev = soft_bounds(**kw) if device == "soft" else constant_step(**kw)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    w = rng.uniform(-0.6, 0.6, (d_size, x_size)).astype(np.float32)
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    w0 = orc.get_weights()
    x = rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)
    d = (0.05 * rng.standard_normal((batch, d_size))).astype(np.float32)
    xg, dg = cuda(x), cuda(d)
    dwg, dwo = [], []
    for s in range(N_SEEDS):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_seed(77 + s)
        gpu.set_learning_rate(0.01)
        gpu.update(xg, dg, False, False, False, False)
        dwg.append(gpu.get_weights().numpy() - w0)
        orc.set_weights(w)
        orc.set_seed(1 + s)
        orc.set_learning_rate(0.01)
        orc.update(x, d)
        dwo.append(orc.get_weights() - w0)
    dwg, dwo = np.stack(dwg), np.stack(dwo)
    assert np.abs(dwo).mean() > 5e-4
    compare_moments(dwg, dwo, f"weight change {device} um={um}")
    # the mean step follows -lr * d^T x (scaled by the device's own step sizes) as much as the oracle's does
    sgd = -(d.T @ x)
    c_gpu = np.corrcoef(dwg.mean(0).ravel(), sgd.ravel())[0, 1]
    c_orc = np.corrcoef(dwo.mean(0).ravel(), sgd.ravel())[0, 1]
    assert c_gpu > 0.15 and abs(c_gpu - c_orc) < 0.05, (c_gpu, c_orc)


def test_full_size_update_noise_free_matches_oracle_through_the_pulse_words(gpu_device):
    """Benchmark configuration 2 at full size, cycle-to-cycle noise off: the GPU's pulse words drive the
    oracle's device model to the same 1M weights (1e-5)."""
    meta, dev = config2(ctoc=False)
    host, orc, _ = build_pair(meta, dev, 1024, 1024, gpu=False)
    w, x, d = config2_data()
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    gpu = tiles.CudaAnalogTile(host)
    gpu.set_seed(3)
    gpu.set_learning_rate(0.01)
    orc.set_learning_rate(0.01)
    gpu.update(cuda(x), cuda(d), False, False, False, False)
    xw, dw, bl = (t.numpy() for t in gpu.get_update_words(256))
    bl_orc, a_orc, b_orc = orc.update_bl_ab(x, d)
    assert np.array_equal(bl, bl_orc)
    a_gpu, b_gpu = (t.numpy() for t in gpu.get_update_ab(256))
    assert np.array_equal(a_gpu, a_orc) and np.array_equal(b_gpu, b_orc)
    orc.update_with_words(xw, dw, bl)
    wg = gpu.get_weights().numpy()
    assert np.abs(wg - orc.get_weights()).max() <= 1e-5
    # expected number of coincidences per cross-point and call: lr * E|x| * E|d| * B / dw_min = 51 (+- statistics)
    pulses_x = np.zeros((256, 1024), np.int64)
    xs = (xw.astype(np.int64) & 0xFFFFFFFF) >> 1
    ds = (dw.astype(np.int64) & 0xFFFFFFFF) >> 1
    coinc = 0.0
    for k in range(31):
        coinc += (((xs >> k) & 1).sum(1) * ((ds >> k) & 1).sum(1)).sum()
    del pulses_x
    assert coinc / (1024 * 1024) == pytest.approx(0.01 * np.abs(x).mean() * np.abs(d).mean() * 256 / 0.001, rel=0.05)


def test_full_size_update_cycle_noise_is_zero_mean_with_the_expected_spread(gpu_device):
    """Same call with cycle-to-cycle noise on (std 0.3): against the noise-free result for the *same* pulse
    words the difference must be zero-mean, and its variance must be the sum over the applied pulses of
    (0.3 * step)^2 with step = scale * (1 - w / bound), evaluated at the start weights (+- 10 %)."""
    meta, dev = config2(ctoc=True)
    meta0, dev0 = config2(ctoc=False)
    host, _, _ = build_pair(meta, dev, 1024, 1024, gpu=False)
    _, orc0, _ = build_pair(meta0, dev0, 1024, 1024, gpu=False)
    w, x, d = config2_data()
    host.set_weights(torch.from_numpy(w))
    orc0.set_weights(w)
    w0 = orc0.get_weights()
    gpu = tiles.CudaAnalogTile(host)
    gpu.set_seed(11)
    gpu.set_learning_rate(0.01)
    orc0.set_learning_rate(0.01)
    gpu.update(cuda(x), cuda(d), False, False, False, False)
    xw, dw, bl = (t.numpy() for t in gpu.get_update_words(256))
    orc0.update_with_words(xw, dw, bl)
    e = (gpu.get_weights().numpy() - orc0.get_weights()).astype(np.float64)
    hid = orc0.get_hidden().astype(np.float64)
    w_max, w_min, up, down = hid[0], hid[1], hid[2], hid[3]
    # up / down pulse counts per cross-point from the words
    xs = xw.astype(np.int64) & 0xFFFFFFFF
    ds = dw.astype(np.int64) & 0xFFFFFFFF
    n_up = np.zeros((1024, 1024))
    n_down = np.zeros((1024, 1024))
    for b in range(256):
        xb, db = xs[b], ds[b]
        sx, sd = (xb & 1), (db & 1)
        cnt = np.zeros((1024, 1024))
        for k in range(1, int(bl[b]) + 1):
            cnt += np.outer((db >> k) & 1, (xb >> k) & 1)
        same = np.equal.outer(sd, sx)
        n_down += np.where(same, cnt, 0)
        n_up += np.where(same, 0, cnt)
    step_up = up * (1 - w0 / w_max)
    step_down = down * (1 - w0 / w_min)
    var_pred = 0.09 * (n_up * step_up**2 + n_down * step_down**2)
    # away from the hard bounds, and no devices with a tiny range (their steps are huge and get clipped)
    inner = (w0 > w_min + 0.05) & (w0 < w_max - 0.05) & (var_pred > 0) & (w_max > 0.3) & (w_min < -0.3)
    assert inner.mean() > 0.6
    assert abs(e[inner].mean()) < 4 * e[inner].std() / np.sqrt(inner.sum())
    # the first-order prediction ignores that later steps damp earlier noise by (1 - scale / bound) each
    # (a simulation of the recursion gives 0.85 - 0.93 of it for these parameters)
    assert 0.75 < e[inner].var() / var_pred[inner].mean() < 1.0
    zz = e[inner] / np.sqrt(var_pred[inner])
    assert 0.85 < zz.std() < 1.0
    assert np.mean(np.abs(zz) > 3) < 0.01


@pytest.mark.parametrize("device", ["soft", "constant"])
def test_cycle_to_cycle_noise_alone_matches_the_oracle_for_fixed_pulse_words(gpu_device, device):
    """Same packed pulse words on both sides, only the cycle-to-cycle noise is random: mean and variance
    of the weights over 64 seeds, GPU against oracle."""
    rng = np.random.default_rng(4)
    x_size, d_size, batch = 96, 64, 32
    meta = make_meta(desired_bl=31, update_management=False, update_bl_management=False)
    kw = dict(dw_min=0.001, dw_min_dtod=0.3, dw_min_std=0.3, construction_seed=5, enforce_consistency=True)
    dev = soft_bounds(**kw) if device == "soft" else constant_step(**kw)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    orc.use_gauss_table(False)
    w = rng.uniform(-0.5, 0.5, (d_size, x_size)).astype(np.float32)
    host.set_weights(torch.from_numpy(w))
    # random words with about a quarter of the 31 pulse bits set
    xw = (rng.integers(0, 2**32, (batch, x_size), dtype=np.uint64) & rng.integers(0, 2**32, (batch, x_size), dtype=np.uint64)).astype(np.uint32)
    dw = (rng.integers(0, 2**32, (batch, d_size), dtype=np.uint64) & rng.integers(0, 2**32, (batch, d_size), dtype=np.uint64)).astype(np.uint32)
    bl = np.full(batch, 31, np.int32)
    xg, dg = cuda(xw.view(np.int32)), cuda(dw.view(np.int32))
    wg, wo = [], []
    for s in range(N_SEEDS):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_seed(500 + s)
        gpu.set_learning_rate(0.01)
        gpu.update_with_words(xg, dg)
        wg.append(gpu.get_weights().numpy())
        orc.set_weights(w)
        orc.set_seed(1 + s)
        orc.set_learning_rate(0.01)
        orc.update_with_words(xw, dw, bl)
        wo.append(orc.get_weights())
    wg, wo = np.stack(wg), np.stack(wo)
    assert wo.std(0).mean() > 1e-3
    compare_moments(wg, wo, f"cycle-to-cycle noise {device}")


def short_words(rng, batch, size, slots):
    """Packed pulse words with bit lines of `slots` pulses: every pulse bit set with probability 1/2, random signs."""
    pulses = rng.integers(0, 2**slots, (batch, size), dtype=np.uint64) << np.uint64(1)
    return (pulses | rng.integers(0, 2, (batch, size), dtype=np.uint64)).astype(np.uint32)


@pytest.mark.parametrize("device,shape,slots", [
    ("soft", (200, 96), 3), ("constant", (200, 96), 3),        # one column per lane
    ("soft", (512, 256), 3), ("constant", (512, 256), 7),      # two
    ("soft", (1024, 512), 3), ("soft", (1024, 512), 7), ("constant", (1024, 512), 3),   # four
])
def test_short_bit_lines_take_the_table_noise_and_match_the_oracle(gpu_device, device, shape, slots):
    """Pulse words with at most 3 / 7 pulses per line run the pulse loop of the usual update call, whose cycle-to-cycle
    factors come from the quantile table and the per-lane stream.  Same words on both sides, only that noise is random:
    mean and variance of every weight over 64 seeds against the oracle's exact normals, without slack on the pooled
    variance."""
    rng = np.random.default_rng(14)
    x_size, d_size = shape
    batch = 40
    meta = make_meta(desired_bl=31, update_management=False, update_bl_management=False)
    kw = dict(dw_min=0.001, dw_min_dtod=0.3, dw_min_std=0.3, construction_seed=5, enforce_consistency=True)
    dev = soft_bounds(**kw) if device == "soft" else constant_step(**kw)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    orc.use_gauss_table(False)
    w = rng.uniform(-0.5, 0.5, (d_size, x_size)).astype(np.float32)
    host.set_weights(torch.from_numpy(w))
    xw, dw = short_words(rng, batch, x_size, slots), short_words(rng, batch, d_size, slots)
    bl = np.full(batch, slots, np.int32)
    xg, dg = cuda(xw.view(np.int32)), cuda(dw.view(np.int32))
    n_seeds = N_SEEDS if x_size < 1024 else 32                      # half a million weights: fewer seeds suffice
    wg, wo = [], []
    for s in range(n_seeds):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_seed(900 + s)
        gpu.set_learning_rate(0.01)
        gpu.update_with_words(xg, dg)
        wg.append(gpu.get_weights().numpy())
        orc.set_weights(w)
        orc.set_seed(1 + s)
        orc.set_learning_rate(0.01)
        orc.update_with_words(xw, dw, bl)
        wo.append(orc.get_weights())
    wg, wo = np.stack(wg), np.stack(wo)
    assert wo.std(0).mean() > 3e-4
    compare_moments(wg, wo, f"table noise {device} {shape} {slots}", variance_slack=0.0)


@pytest.mark.parametrize("x_size,d_size", [(200, 2048), (512, 1024), (1024, 512)])
def test_noise_factors_of_the_pulse_loop_one_pulse_at_a_time(gpu_device, x_size, d_size):
    """One pulse per cross-point, nothing random but its cycle-to-cycle factor: xi = (dW / step - 1) / std must have
    mean 0, variance 1 and the kurtosis of the 256-level quantile table (2.92), and must be uncorrelated between the two
    consecutive pulses of a cross-point, between neighbouring rows and between columns at every distance at which one
    lane, or one draw of a lane's generator, could serve both (1, 64, 128, 192, 256, 512, 768): each within 4 standard
    errors over a million pairs."""
    std = 0.3
    meta = make_meta(desired_bl=31, update_management=False, update_bl_management=False)
    dev = constant_step(dw_min=0.001, dw_min_dtod=0.0, dw_min_std=std, up_down=0.0, up_down_dtod=0.0, w_max=1.0, w_min=-1.0,
                        w_max_dtod=0.0, w_min_dtod=0.0, construction_seed=5)
    host, _orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    host.set_weights(torch.zeros(d_size, x_size))
    names = host.get_hidden_parameter_names()
    step_down = host.get_hidden_parameters()[names.index("dwmin_down")].numpy().astype(np.float64)

    def words(batch, size):                      # slot 1 fires in every sample, positive sign
        return cuda(np.full((batch, size), 2, np.uint32).view(np.int32))

    first, second = [], []
    n_runs = 3
    for s in range(n_runs):
        one, two = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
        for t in (one, two):
            t.set_seed(40 + s)
            t.set_learning_rate(0.01)
        one.update_with_words(words(1, x_size), words(1, d_size))
        two.update_with_words(words(2, x_size), words(2, d_size))
        w1, w2 = one.get_weights().numpy().astype(np.float64), two.get_weights().numpy().astype(np.float64)
        first.append((-w1 / step_down - 1.0) / std)             # equal signs and a positive learning rate: a step down
        second.append((-(w2 - w1) / step_down - 1.0) / std)
    first, second = np.stack(first), np.stack(second)
    for xi in (first, second):
        n = xi.size
        assert n >= 1_000_000
        assert abs(xi.mean()) < 4.0 / np.sqrt(n)
        assert abs(xi.var() - 1.0) < 0.01
        kurt = np.mean((xi - xi.mean()) ** 4) / xi.var() ** 2
        assert abs(kurt - 2.92) < 0.05, kurt
        assert np.abs(xi).max() < 3.0                            # the table ends at 2.9 sigma

    def corr(a, b):
        a, b = a.ravel() - a.mean(), b.ravel() - b.mean()
        return float((a * b).mean() / np.sqrt((a * a).mean() * (b * b).mean())), a.size

    checks = [("consecutive pulses", first, second), ("rows", first[:, :-1, :], first[:, 1:, :])]
    for lag in (1, 64, 128, 192, 256, 512, 768):
        if lag < x_size:
            checks.append((f"columns {lag} apart", first[:, :, :-lag], first[:, :, lag:]))
    for what, a, b in checks:
        c, n = corr(a, b)
        assert abs(c) < 4.0 / np.sqrt(n), (what, c, n)
    # the factors of a lane's consecutive draws: squares too (a shared scale would show there first)
    c, n = corr(first ** 2, second ** 2)
    assert abs(c) < 4.0 / np.sqrt(n), ("squares of consecutive pulses", c, n)


def test_stochastic_rounding_and_input_noise_moments(gpu_device):
    """DAC / ADC stochastic rounding and input noise are random per element: moments over 64 seeds."""
    rng = np.random.default_rng(7)
    x_size, d_size, batch = 128, 64, 16
    f_io = io_params(out_noise=0.02, inp_noise=0.05, inp_sto_round=True, out_sto_round=True, inp_res=1 / 16.0,
                     out_res=1 / 32.0, noise_management=dv.NoiseManagementType.AbsMax)
    meta = make_meta(f_io, io_params(out_noise=0.0))
    dev = soft_bounds(construction_seed=3, enforce_consistency=True)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    orc.use_gauss_table(False)
    w = rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(np.float32)
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    gpu = tiles.CudaAnalogTile(host)
    x = rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)
    xg = cuda(x)
    yg, yo = [], []
    for s in range(N_SEEDS):
        gpu.set_seed(300 + s)
        orc.set_seed(1 + s)
        yg.append(gpu.forward(xg, False, False, False, False, False).cpu().numpy())
        yo.append(orc.forward(x))
    yg, yo = np.stack(yg), np.stack(yo)
    assert yo.std(0).mean() > 0.1  # coarse ADC: the rounding noise dominates
    compare_moments(yg, yo, "stochastic rounding + input noise")
    # unbiasedness of stochastic rounding: the seed-mean approaches the unquantized product
    ideal = x @ w.T
    assert np.abs(yg.mean(0) - ideal).mean() < 0.12


def test_discretized_pulse_probabilities_moments(gpu_device):
    """update.res > 0 with stochastic rounding of the pulse probabilities."""
    rng = np.random.default_rng(9)
    x_size, d_size, batch = 64, 48, 16
    meta = make_meta(desired_bl=31, update_management=False, update_bl_management=False, res=1 / 8.0, sto_round=True)
    dev = constant_step(dw_min=0.001, dw_min_dtod=0.1, dw_min_std=0.0, construction_seed=2, enforce_consistency=True)
    host, orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    w0 = orc.get_weights()
    x = rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)
    d = (0.5 * rng.standard_normal((batch, d_size))).astype(np.float32)
    xg, dg = cuda(x), cuda(d)
    dwg, dwo = [], []
    for s in range(N_SEEDS):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_seed(40 + s)
        gpu.set_learning_rate(0.01)
        gpu.update(xg, dg, False, False, False, False)
        dwg.append(gpu.get_weights().numpy() - w0)
        orc.set_weights(w0)
        orc.set_seed(1 + s)
        orc.set_learning_rate(0.01)
        orc.update(x, d)
        dwo.append(orc.get_weights() - w0)
    compare_moments(np.stack(dwg), np.stack(dwo), "discretized pulse probabilities")


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., 2011) on arrays of counters."""
    m = np.uint64(0xFFFFFFFF)
    c = [np.broadcast_to(np.asarray(v, np.uint64), np.broadcast(c0, c1).shape) for v in (c0, c1, c2, c3)]
    for r in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        a, b = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF), np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ a, p1 & m, (p0 >> np.uint64(32)) ^ c[3] ^ b, p0 & m]
    return c


@pytest.mark.parametrize("batch,d_size", [(1024, 1024), (5, 4096)])
def test_output_noise_against_64_bits(gpu_device, batch, d_size):
    """Normal numbers of the ADC stage: with no weights and a spread of one they are the outputs.  The hardware's logarithm,
    square root, sine and cosine are off by about an ulp each, of a radius of at most sqrt(2 ln 2^24) = 5.8: 2e-6 is three of
    its ulps and a half.  Root mean square 6.1e-8 over all pairs; a correctly rounded root of -2 ln u and an angle in radians
    had 1.3e-7."""
    seed = 0x1234567890ABCDEF
    io = io_params(inp_res=-1.0, out_res=-1.0, out_noise=1.0, out_bound=1000.0)
    dev = constant_step(construction_seed=1, w_max_dtod=0.0, w_min_dtod=0.0)     # (no bound below zero cuts a weight)
    host, _orc, _ = build_pair(make_meta(io, noise_free_io()), dev, 8, d_size, gpu=False)
    host.set_weights(torch.zeros(d_size, 8))
    assert not host.get_weights().any()
    tile = tiles.CudaAnalogTile(host)
    tile.set_seed(seed)
    y = tile.forward(torch.ones(batch, 8, device="cuda"), False).cpu().numpy().astype(np.float64)
    b, o4 = np.meshgrid(np.arange(batch, dtype=np.uint64), np.arange(d_size // 4, dtype=np.uint64), indexing="ij")
    r = _philox(o4, b, 0, 1, seed & 0xFFFFFFFF, seed >> 32)
    want = np.empty((batch, d_size // 4, 4))
    for pair in range(2):
        u = ((r[2 * pair] >> np.uint64(8)).astype(np.float64) + 1.0) / 2.0 ** 24
        turns = (r[2 * pair + 1] >> np.uint64(8)).astype(np.float64) / 2.0 ** 24
        radius = np.sqrt(-2.0 * np.log(u))
        want[..., 2 * pair] = radius * np.cos(2.0 * np.pi * turns)
        want[..., 2 * pair + 1] = radius * np.sin(2.0 * np.pi * turns)
    off = y - want.reshape(batch, d_size)
    assert np.abs(off).max() <= 2e-6
    assert np.sqrt((off ** 2).mean()) <= 1e-7
