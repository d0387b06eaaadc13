"""The pulse loop of tiles with several columns per lane runs on lane masks (k_update_pulsed_masks) where batch and rows are
many enough (update_mask_columns).  A group call runs the plain pulse loop on the same pulse trains and noise streams, so
both leave the same weights, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import constant_step, make_meta, soft_bounds
from test_gpu_pulse_stream import _additive, _tile

pytestmark = pytest.mark.gpu


def _device(kind):
    if kind == "soft_bounds":
        return soft_bounds(construction_seed=5)
    if kind == "constant_step":
        return constant_step(construction_seed=5)
    if kind == "quiet":
        return soft_bounds(construction_seed=5, dw_min_std=0.0)
    return _additive(0.3 if kind == "additive" else 0.0)


def _update(tile, kernel, *args):
    """An update that has to run its pulse loop on that kernel."""
    tile.set_profiling(True)
    tile.update(*args)
    assert [name for name, _ms in tile.get_profile()][-1] == kernel
    tile.set_profiling(False)


def _data(x_size, d_size, batch, sparse):
    gen = torch.Generator("cuda").manual_seed(batch + x_size)
    x = torch.rand(batch, x_size, generator=gen, device="cuda") * 2 - 1
    d = torch.randn(batch, d_size, generator=gen, device="cuda") * 0.05
    if sparse:
        d[torch.rand(batch, generator=gen, device="cuda") < sparse] = 0.0
    return x, d


# four and two columns per lane; a span of columns that is full, one more than full, mostly behind the row's end; rows that
# are dealt out by their work (1024 x 1024) and units that do not fill the last workgroup; chunks that are not full; lr sets
# the longest bit line: 1, 3, 7 and 31 (the last walked pulse by pulse); rows with hardly a pass
@pytest.mark.parametrize("x_size,d_size,batch,lr,sparse", [
    (1024, 1024, 130, 0.01, 0), (1024, 515, 300, 0.05, 0), (1025, 515, 257, 0.0005, 0), (1024, 1024, 129, 0.6, 0),
    (513, 301, 512, 0.02, 0), (257, 601, 260, 0.05, 0), (512, 513, 1000, 0.0005, 0.99), (700, 333, 450, 0.02, 0.9),
    (520, 512, 200, 0.6, 0)])
@pytest.mark.parametrize("kind", ["soft_bounds", "constant_step", "quiet", "additive", "additive_quiet"])
def test_pulse_loop_on_lane_masks_equals_the_plain_one(x_size, d_size, batch, lr, sparse, kind):
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(x_size, d_size, batch, sparse)
    one, other = (_tile(x_size, d_size, _device(kind)) for _ in range(2))
    start = one.get_weights()
    for tile in (one, other):
        tile.set_learning_rate(lr)
    group = TileGroup([other])
    for call in range(2):
        if call:  # lines along the batch
            _update(one, "update_pulsed_masks", x.t().contiguous(), d.t().contiguous(), False, True, True)
        else:
            _update(one, "update_pulsed_masks", x, d, False)
        group.update([x], [d])
    assert torch.equal(one.get_weights(), other.get_weights())
    assert not torch.equal(one.get_weights(), start)
    for mine, theirs in zip(one.get_update_words(batch), other.get_update_words(batch)):
        assert torch.equal(mine, theirs)


def test_pulse_loop_on_lane_masks_with_weights_outside_their_bounds(storage_mode):
    """They are cut back by the first pulse and not before; a negative learning rate turns the direction."""
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x_size, d_size, batch = 600, 400, 300
    x, d = _data(x_size, d_size, batch, 0)
    x[:, ::5] = 0.0
    results = []
    for grouped in (False, True):
        tile = _tile(x_size, d_size, _device("soft_bounds"))
        if storage_mode == "xd_shared":
            w = tile._shared_weights.t()
        else:
            w = torch.empty(d_size, x_size, device="cuda")
            tile.set_shared_weights_row_major(w)
        w[:, ::3] = 2.5
        tile.set_learning_rate(-0.01)
        if grouped:
            TileGroup([tile]).update([x], [d])
        else:
            _update(tile, "update_pulsed_masks", x, d, False)
        results.append(w.clone())
    assert torch.equal(results[0], results[1])
    assert bool((results[0][:, ::15] == 2.5).all())   # no x pulse: untouched
    assert float(results[0][:, 3].max()) < 2.5


def test_masks_find_their_room_after_a_larger_call_on_planes(gpu_device):
    """A row of 513 elements has masks for 1024: more words for 600 samples than bit planes for 1024 of them.  The larger call
    (of a group: bit planes) makes room for both, so that the smaller one can be captured."""
    from aihwkit_amd._cabi import lib
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(513, 301, 1024, 0)
    tile = _tile(513, 301, _device("soft_bounds"))
    tile.set_learning_rate(0.01)
    group = TileGroup([tile])
    for _ in range(2):
        group.update([x], [d])
    before = lib().rpu_device_allocation_count()
    _update(tile, "update_pulsed_masks", x[:600].contiguous(), d[:600].contiguous(), False)
    assert lib().rpu_device_allocation_count() == before


@pytest.mark.parametrize("name,value", [("slope_up", float("nan")), ("dwmin_down", float("inf")), ("max_bound", float("inf"))])
def test_pulse_loop_on_lane_masks_with_parameters_that_are_not_finite(name, value):
    """They reach the cross-points that hold them, in the plain loop's way, and no other."""
    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x_size, d_size, batch = 600, 400, 300
    host = make_meta(desired_bl=31).create_array(x_size, d_size, soft_bounds(construction_seed=5))
    hidden = host.get_hidden_parameters()
    hidden[host.get_hidden_parameter_names().index(name), :, ::3] = value
    host.set_hidden_parameters(hidden)
    host.set_weights(torch.from_numpy(np.random.default_rng(3).uniform(-0.4, 0.4, (d_size, x_size)).astype(np.float32)))
    x, d = _data(x_size, d_size, batch, 0)
    x[:, ::5] = 0.0
    one, other = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    before = one.get_weights().numpy()
    for tile in (one, other):
        tile.set_seed(17)
        tile.set_learning_rate(0.01)
    _update(one, "update_pulsed_masks", x, d, False)
    TileGroup([other]).update([x], [d])
    mine, theirs = one.get_weights().numpy(), other.get_weights().numpy()
    assert np.array_equal(mine, theirs, equal_nan=True)
    assert np.array_equal(mine[:, ::5], before[:, ::5], equal_nan=True)
    assert np.isfinite(mine[:, 1::3]).all() and not np.array_equal(mine, before, equal_nan=True)


def _long_lines_tile(x_size, d_size, kind, desired_bl=31, fixed_bl=True):
    from aihwkit_amd.rpu_base import tiles
    host = make_meta(desired_bl=desired_bl, fixed_bl=fixed_bl, update_bl_management=False).create_array(x_size, d_size, _device(kind))
    host.set_weights(torch.from_numpy(np.random.default_rng(3).uniform(-0.4, 0.4, (d_size, x_size)).astype(np.float32)))
    tile = tiles.CudaAnalogTile(host)
    tile.set_seed(17)
    return tile


# without BL management all lines are long (k_update_pulsed_words): one lane, one wave and rows and columns just beyond them, a
# block of 128 samples that is full, one short of it and one beyond it, two columns per lane in the kernel compared with, the
# shortest such line (8), lines of two words (40 pulses), samples without a pulse, a step against the gradient
@pytest.mark.parametrize("x_size,d_size,batch,desired_bl,lr,sparse", [
    (1, 1, 3, 31, 0.02, 0), (64, 16, 128, 31, 0.02, 0), (65, 17, 129, 31, 0.02, 0), (63, 15, 127, 8, 0.004, 0),
    (785, 300, 37, 31, 0.01, 0), (130, 70, 600, 31, 0.01, 0.9), (200, 33, 70, 31, 0.04, 0), (300, 500, 200, 12, -0.01, 0)])
@pytest.mark.parametrize("kind", ["soft_bounds", "constant_step", "quiet", "additive"])
def test_long_bit_lines_through_lds_equal_the_plain_loop(x_size, d_size, batch, desired_bl, lr, sparse, kind, storage_mode):
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(x_size, d_size, batch, sparse)
    two_words = lr > 31 * 0.001  # dw_min: where the bit line is not fixed
    one, other = (_long_lines_tile(x_size, d_size, kind, desired_bl, not two_words) for _ in range(2))
    start = one.get_weights()
    for tile in (one, other):
        tile.set_learning_rate(lr)
    if two_words:  # 140 rows of words: not in groups; the plain loop takes the same ones
        for _ in range(2):
            _update(one, "update_pulsed_words", x, d, False)
            assert one.get_update_words_per_sample() == 2
            x_words, d_words, _bl = one.get_update_words(batch)
            assert (x_words[1::2] & ~1).any() and (d_words[1::2] & ~1).any()
            other.set_profiling(True)
            other.update_with_words(x_words.cuda(), d_words.cuda())
            assert [name for name, _ms in other.get_profile()][-1] == "update_pulsed"
            other.set_profiling(False)
        assert torch.equal(one.get_weights(), other.get_weights())
        assert not torch.equal(one.get_weights(), start)
        return
    group = TileGroup([other])
    for _ in range(2):
        _update(one, "update_pulsed_words", x, d, False)
        group.update([x], [d])
    assert torch.equal(one.get_weights(), other.get_weights())
    assert not torch.equal(one.get_weights(), start)
    one.update(torch.zeros_like(x), d, False)  # no sample has pulses
    assert torch.equal(one.get_weights(), other.get_weights())


# k_update_lines_small at one and four lines of either operand, at its most samples, and at its most values and longest lines; the
# last of each is a call beyond
@pytest.mark.parametrize("x_size,d_size,batch,small", [
    (1, 1, 1, True), (4, 5, 2, True), (129, 10, 64, True), (129, 10, 65, False), (200, 200, 64, True), (200, 201, 64, False),
    (1100, 436, 7, True), (1100, 437, 7, False), (900, 636, 1, True), (512, 512, 16, True), (512, 513, 16, False)])
@pytest.mark.parametrize("blm", [True, False])
def test_small_updates_in_one_launch_of_pulse_trains_equal_those_of_a_group(x_size, d_size, batch, small, blm, storage_mode):
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(x_size, d_size, batch, 0)
    one, other = (_tile(x_size, d_size, _device("soft_bounds")) if blm else _long_lines_tile(x_size, d_size, "soft_bounds")
                  for _ in range(2))
    for tile in (one, other):
        tile.set_learning_rate(0.02)
    group = TileGroup([other])
    for _ in range(2):
        one.set_profiling(True)
        one.update(x, d, False)
        assert ("update_prepare" not in [name for name, _ms in one.get_profile()]) == small
        one.set_profiling(False)
        group.update([x], [d])
        for mine, theirs in zip(one.get_update_words(batch), other.get_update_words(batch)):
            assert torch.equal(mine, theirs)
        for mine, theirs in zip(one.get_update_ab(batch), other.get_update_ab(batch)):
            assert torch.equal(mine, theirs)
    assert torch.equal(one.get_weights(), other.get_weights())


# samples that share a workgroup of k_update_prepare, four or sixteen of them: one has bit lines several times longer than all others,
# the first and the last of a workgroup, and the last of one that is not full
@pytest.mark.parametrize("x_size,d_size,batch", [(70, 40, 1025), (70, 40, 2050), (60, 40, 1040), (60, 40, 1041)])
@pytest.mark.parametrize("at", [0, 3, 15, -1])
def test_the_longest_bit_line_of_many_short_samples(x_size, d_size, batch, at, storage_mode):
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(x_size, d_size, batch, 0)
    d[at] *= 6.0
    one, other = (_tile(x_size, d_size, _device("soft_bounds")) for _ in range(2))
    for tile in (one, other):
        tile.set_learning_rate(0.02)
    group = TileGroup([other])
    for _ in range(2):
        one.update(x, d, False)
        group.update([x], [d])
    for mine, theirs in zip(one.get_update_words(batch), other.get_update_words(batch)):
        assert torch.equal(mine, theirs)
    bl = one.get_update_words(batch)[2]
    assert int(bl[at]) > 2 * int(torch.cat([bl[:at], bl[at + 1:] if at >= 0 else bl[:0]]).max())
    assert torch.equal(one.get_weights(), other.get_weights())


# every kernel that makes pulse trains reads a bias column that is not stored as the row that has it: a few samples, lane masks,
# pipeline of waves, long lines, implicit pulses
@pytest.mark.parametrize("x_size,d_size,batch,pulse_type,blm", [
    (2, 3, 4, "StochasticCompressed", True), (129, 10, 64, "StochasticCompressed", True), (601, 400, 300, "StochasticCompressed", True),
    (433, 48, 1030, "StochasticCompressed", True), (65, 20, 130, "StochasticCompressed", False), (70, 33, 20, "MeanCount", True)])
@pytest.mark.parametrize("x_trans", [False, True])
def test_bias_column_that_is_not_stored(x_size, d_size, batch, pulse_type, blm, x_trans, storage_mode):
    from aihwkit_amd.rpu_base import devices as dv
    from aihwkit_amd.rpu_base import tiles
    x, d = _data(x_size - 1, d_size, batch, 0)
    x *= 0.7  # the bias is the largest line
    results = []
    for bias in (True, False):
        host = make_meta(desired_bl=31, pulse_type=getattr(dv.PulseType, pulse_type),
                         update_bl_management=blm).create_array(x_size, d_size, _device("soft_bounds"))
        host.set_weights(torch.zeros(d_size, x_size))
        tile = tiles.CudaAnalogTile(host)
        tile.set_seed(5)
        tile.set_learning_rate(0.02)
        line = x if bias else torch.cat([x, torch.ones(batch, 1, device="cuda")], 1)
        tile.update(line.t().contiguous() if x_trans else line.contiguous(), d, bias, x_trans)
        results.append(tile.get_weights())
    assert torch.equal(results[0], results[1])
    assert float(results[0][:, -1].abs().max()) > 0.0


# small calls find their maxima in the launch that makes the pulse trains (k_update_lines_small), the same tile in a group has a
# launch for them: one sample (1024 threads to it, 16 at 64), samples and lines at and next to the ends of the range (25600 values,
# lines of 1536), a last block of line elements that is not full, a gradient that is zero, values that are not finite
@pytest.mark.parametrize("x_size,d_size,batch", [(1, 1, 1), (3, 2, 64), (129, 10, 63), (130, 11, 65), (785, 256, 1), (785, 751, 2), (785, 752, 2),
                                                 (300, 100, 64), (301, 100, 64), (63, 5, 17), (1000, 17, 16)])
@pytest.mark.parametrize("um,blm,desired_bl", [(True, True, 31), (True, False, 5), (False, False, 31)])
def test_small_calls_prepare_in_the_launch_of_the_pulse_trains(x_size, d_size, batch, um, blm, desired_bl, storage_mode):
    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.rpu_base.tiles import TileGroup
    x, d = _data(x_size, d_size, batch, 0)
    d[batch // 2] = 0.0
    if batch > 2:
        x[1, 0], d[2, -1] = float("inf"), float("nan")
    pair = []
    for _ in range(2):
        host = make_meta(desired_bl=desired_bl, update_management=um, update_bl_management=blm).create_array(x_size, d_size, _device("soft_bounds"))
        host.set_weights(torch.from_numpy(np.random.default_rng(3).uniform(-0.4, 0.4, (d_size, x_size)).astype(np.float32)))
        tile = tiles.CudaAnalogTile(host)
        tile.set_seed(17)
        tile.set_learning_rate(0.004)
        pair.append(tile)
    one, other = pair
    group = TileGroup([other])
    for _ in range(2):
        one.update(x, d, False)
        group.update([x], [d])
    assert torch.equal(one.get_weights(), other.get_weights())
    for mine, theirs in zip(one.get_update_words(batch), other.get_update_words(batch)):
        assert torch.equal(mine, theirs)
    if batch > 1 and x_size > 1:  # lines that run the other way take the two launches
        before = one.get_weights()
        one.update(x.t().contiguous(), d.t().contiguous(), False, True, True)
        group.update([x], [d])
        assert torch.equal(one.get_weights(), other.get_weights()) and not torch.equal(one.get_weights(), before)
