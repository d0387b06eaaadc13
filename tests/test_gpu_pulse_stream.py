"""The pulse loop of long batches on tiles of few rows runs as a pipeline of waves (k_update_pulsed_stream).  A group call
runs the plain pulse loop on the same pulse trains and noise streams, so both leave the same weights, bit for bit."""
import numpy as np
import pytest
import torch

from aihwkit_amd.rpu_base import devices as dv
from helpers import constant_step, make_meta, soft_bounds

pytestmark = pytest.mark.gpu


def _tile(x_size, d_size, dev):
    from aihwkit_amd.rpu_base import tiles
    meta = make_meta(desired_bl=31)
    host = meta.create_array(x_size, d_size, dev)
    host.set_weights(torch.from_numpy(np.random.default_rng(3).uniform(-0.4, 0.4, (d_size, x_size)).astype(np.float32)))
    tile = tiles.CudaAnalogTile(host)
    tile.set_seed(17)
    return tile


def _additive(dw_min_std):
    """A linear-step device whose noise is added to the step: a step without its factor still has the slope term."""
    dev = dv.LinearStepResistiveDeviceParameter()
    for name, value in dict(gamma_up=0.4, gamma_down=0.2, mult_noise=False, dw_min_std=dw_min_std, construction_seed=5,
                            enforce_consistency=True).items():
        setattr(dev, name, value)
    return dev


# blocks of 64 columns and a rest, one and two teams to a workgroup (more than 256 blocks in all), a chunk that is not
# full, batches with almost no pulse; lr sets the longest bit line: 1, 3, 7 and 31 (the last walked pulse by pulse)
@pytest.mark.parametrize("x_size,d_size,batch,lr,sparse", [
    (5, 3, 1024, 0.0005, False), (64, 2, 1056, 0.02, False), (65, 4, 1500, 0.05, False), (129, 100, 1025, 0.004, False),
    (200, 7, 4100, 0.0005, True), (250, 5, 2048, 0.6, False), (433, 48, 2100, 0.02, False), (70, 260, 1030, 0.02, True)])
@pytest.mark.parametrize("kind", ["soft_bounds", "constant_step", "quiet", "additive", "additive_quiet"])
def test_pipelined_pulse_loop_equals_the_plain_one(x_size, d_size, batch, lr, sparse, kind):
    from aihwkit_amd.rpu_base.tiles import TileGroup
    if kind == "soft_bounds":
        dev = soft_bounds(construction_seed=5)
    elif kind == "constant_step":
        dev = constant_step(construction_seed=5)
    elif kind == "quiet":
        dev = soft_bounds(construction_seed=5, dw_min_std=0.0)
    else:
        dev = _additive(0.3 if kind == "additive" else 0.0)
    gen = torch.Generator("cuda").manual_seed(batch + x_size)
    x = torch.rand(batch, x_size, generator=gen, device="cuda") * 2 - 1
    d = torch.randn(batch, d_size, generator=gen, device="cuda") * 0.05
    if sparse:
        d[torch.rand(batch, generator=gen, device="cuda") < 0.995] = 0.0
    one, other = (_tile(x_size, d_size, dev) for _ in range(2))
    start = one.get_weights()
    for tile in (one, other):
        tile.set_learning_rate(lr)
    group = TileGroup([other])
    for _ in range(2):
        one.update(x, d, False)
        group.update([x], [d])
    assert torch.equal(one.get_weights(), other.get_weights())
    assert not torch.equal(one.get_weights(), start)
    for mine, theirs in zip(one.get_update_words(batch), other.get_update_words(batch)):
        assert torch.equal(mine, theirs)


def test_pipelined_pulse_loop_with_weights_outside_their_bounds(storage_mode):
    """A bound tensor may hold values outside the device bounds: they are cut back by the first pulse and not before."""
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x_size, d_size, batch = 130, 6, 1200
    gen = torch.Generator("cuda").manual_seed(1)
    x = torch.rand(batch, x_size, generator=gen, device="cuda") * 2 - 1
    x[:, ::5] = 0.0
    d = torch.randn(batch, d_size, generator=gen, device="cuda") * 0.05
    results = []
    for grouped in (False, True):
        tile = _tile(x_size, d_size, soft_bounds(construction_seed=5))
        if storage_mode == "xd_shared":
            w = tile._shared_weights.t()
        else:
            w = torch.empty(d_size, x_size, device="cuda")
            tile.set_shared_weights_row_major(w)
        w[:, ::3] = 2.5
        tile.set_learning_rate(0.01)
        if grouped:
            TileGroup([tile]).update([x], [d])
        else:
            tile.update(x, d, False)
        results.append(w.clone())
    assert torch.equal(results[0], results[1])
    assert bool((results[0][:, ::15] == 2.5).all())   # no x pulse: untouched
    assert float(results[0][:, 3].max()) < 2.5


@pytest.mark.parametrize("name,value", [("slope_up", float("nan")), ("dwmin_down", float("inf")), ("max_bound", float("inf"))])
def test_pipelined_pulse_loop_with_parameters_that_are_not_finite(name, value):
    """Cross-points with such a parameter, or none, follow the plain loop; the ones without a pulse stay as they are."""
    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x_size, d_size, batch = 130, 6, 1200
    host = make_meta(desired_bl=31).create_array(x_size, d_size, soft_bounds(construction_seed=5))
    hidden = host.get_hidden_parameters()
    hidden[host.get_hidden_parameter_names().index(name), :, ::3] = value
    host.set_hidden_parameters(hidden)
    start = torch.from_numpy(np.random.default_rng(3).uniform(-0.4, 0.4, (d_size, x_size)).astype(np.float32))
    host.set_weights(start)
    gen = torch.Generator("cuda").manual_seed(1)
    x = torch.rand(batch, x_size, generator=gen, device="cuda") * 2 - 1
    x[:, ::5] = 0.0
    d = torch.randn(batch, d_size, generator=gen, device="cuda") * 0.05
    one, other = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    before = one.get_weights()
    for tile in (one, other):
        tile.set_seed(17)
        tile.set_learning_rate(0.01)
    one.update(x, d, False)
    TileGroup([other]).update([x], [d])
    mine, theirs = one.get_weights().numpy(), other.get_weights().numpy()
    assert np.array_equal(mine, theirs, equal_nan=True)
    assert np.array_equal(mine[:, ::5], before.numpy()[:, ::5], equal_nan=True)
    assert not np.array_equal(mine, before.numpy(), equal_nan=True)
