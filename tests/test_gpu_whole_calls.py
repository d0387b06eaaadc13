"""Batches between the small ones and those of the large tiles run in one launch (k_mvm_whole) with the bits of the launches that
they take otherwise: outputs, input gradients and round counts are compared bit for bit, with noise, for weights stored either way."""
import os

import numpy as np
import pytest
import torch

from aihwkit_amd._cabi import lib
from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles
from helpers import build_pair, constant_step, io_params, make_meta

pytestmark = pytest.mark.gpu
NM, BM = dv.NoiseManagementType, dv.BoundManagementType


def host_tile(rng, x_size, d_size, out_bound, bm=BM.Iterative, nm=NM.AbsMax, **other):
    f_io = io_params(**{**dict(inp_res=1 / 126.0, out_res=1 / 510.0, out_noise=0.06, noise_management=nm, bound_management=bm,
                               out_bound=out_bound), **other})
    b_io = io_params(**{**dict(inp_res=1 / 126.0, out_res=1 / 510.0, out_noise=0.06, noise_management=nm), **other})
    dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=1)
    host, _orc, _ = build_pair(make_meta(f_io, b_io), dev, x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(rng.uniform(-0.6, 0.6, (d_size, x_size)).astype(np.float32)))
    return host


# (where every tile is bound to an [x_size, d_size] tensor anyway, no test binds one itself)
binds = pytest.mark.skipif(os.environ.get("RPU_TEST_STORAGE") == "xd_shared", reason="the tiles are bound already")


def pair_of(host, bound=False):
    """The tile on the launches that its calls take by themselves, and one that takes the others."""
    pair = []
    for small in (True, False):
        tile = tiles.CudaAnalogTile(host)
        if bound:
            tile.live = torch.empty(tile.get_x_size(), tile.get_d_size(), device="cuda")
            tile.set_shared_weights(tile.live)
        tile.set_small_calls(small)
        tile.set_seed(11)
        pair.append(tile)
    return pair


def names_of(tile, call):
    tile.set_profiling(True)
    out = call(tile)
    names = [name for name, _ms in tile.get_profile()][1:]
    tile.set_profiling(False)
    return out, names


# x_size, d_size, batch, bias: contractions on both sides of a step of 32 and of the lengths from which the padding changes (256,
# 512), the longest one and one that leaves the last waves without a step; outputs and samples around blocks of 16 and 64; both
# kinds of blocks (16 outputs, 64)
@pytest.mark.parametrize("x_size,d_size,batch,bias", [
    (65, 1000, 300, False), (100, 70, 1500, True), (129, 300, 257, True), (255, 256, 256, False), (256, 257, 303, False),
    (300, 333, 190, True), (511, 130, 255, True), (513, 128, 512, False), (785, 256, 64, True), (1025, 700, 33, False),
    (1024, 700, 500, False), (785, 256, 1100, False), (2048, 33, 160, False), (2047, 130, 60, True)])
def test_one_launch_has_the_bits_of_the_others(gpu_device, x_size, d_size, batch, bias):
    rng = np.random.default_rng(x_size + d_size)
    # of an output: of thousands, one at least is beyond two of them and none beyond six
    spread = 0.2 * np.sqrt(x_size)
    for out_bound in (0.25 * spread, 1.7 * spread, 100.0 * spread):
        pair = pair_of(host_tile(rng, x_size, d_size, out_bound))
        most, taken = 0, []
        for call in range(3):                 # rounds 0 to 2 together
            x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size - int(bias))).astype(np.float32)).cuda()
            d = torch.from_numpy(rng.normal(0, 0.05, (batch, d_size)).astype(np.float32)).cuda()
            x[batch // 2] = 0.0
            (y, names), (y_other, names_other) = (names_of(t, lambda t: t.forward(x, bias)) for t in pair)
            assert "mvm_whole" not in names_other
            taken.append(names == ["mvm_whole"])
            assert torch.equal(y, y_other), (out_bound, call)
            assert torch.equal(pair[0].get_bm_rounds(batch), pair[1].get_bm_rounds(batch))
            most = max(most, int(pair[0].get_bm_rounds(batch).max()))
            (g, names), (g_other, _) = (names_of(t, lambda t: t.backward(d, bias)) for t in pair)
            assert names != ["mvm_whole"] or torch.equal(g, g_other)
        assert (most >= 4) == (out_bound < spread) and (most > 1) == (out_bound < 50 * spread)
        # Rounds beyond the first three: once, unless the matrix is small.  The first call makes no room for results wider than the
        # quantized rows.
        once = most >= 4 and x_size * d_size > 1 << 14
        assert taken.count(True) == 1 if once else all(taken[1:]) and (taken[0] or d_size > x_size)


# weights stored [x_size, d_size]: a load runs along the outputs, of one (16 outputs to a workgroup) or four (64)
@binds
@pytest.mark.parametrize("x_size,d_size,batch,bias", [(300, 333, 190, True), (513, 130, 256, False), (785, 301, 1000, True), (65, 1000, 300, False)])
def test_weights_along_the_outputs(gpu_device, x_size, d_size, batch, bias):
    rng = np.random.default_rng(x_size)
    for out_bound in (0.05 * np.sqrt(x_size), 0.34 * np.sqrt(x_size)):
        pair = pair_of(host_tile(rng, x_size, d_size, out_bound), bound=True)
        taken = []
        for _ in range(2):
            x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size - int(bias))).astype(np.float32)).cuda()
            (y, names), (y_other, _) = (names_of(t, lambda t: t.forward(x, bias)) for t in pair)
            taken.append(names == ["mvm_whole"])
            assert torch.equal(y, y_other)
            assert torch.equal(pair[0].get_bm_rounds(batch), pair[1].get_bm_rounds(batch)) and pair[0].get_bm_rounds(batch).max() > 1
        assert any(taken)


def test_rounds_beyond_those_together_take_the_other_launches(gpu_device):
    """A call with a sample in round 3 sends those that follow to the other launches, and comes back when none has been there for 64;
    a captured one then makes no room on them."""
    rng = np.random.default_rng(3)
    x_size, d_size, batch = 300, 270, 203
    pair = pair_of(host_tile(rng, x_size, d_size, 1.0))
    calm = rng.uniform(-0.05, 0.05, (d_size, x_size)).astype(np.float32)
    x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)).cuda()

    def step():
        (y, names), (y_other, _) = (names_of(t, lambda t: t.forward(x, False)) for t in pair)
        assert torch.equal(y, y_other) and torch.equal(pair[0].get_bm_rounds(batch), pair[1].get_bm_rounds(batch))
        return names == ["mvm_whole"], int(pair[0].get_bm_rounds(batch).max())

    taken, most = step()
    assert taken and most >= 4
    for _ in range(70):                       # as long as samples go there
        taken, most = step()
        assert not taken and most >= 4
    for tile in pair:
        tile.set_weights(torch.from_numpy(calm))
    taken = [step()[0] for _ in range(70)]
    assert not any(taken[:60]) and all(taken[66:])
    # deep again, on a tile whose other launches have never fused rounds: captured
    gpu, other = pair_of(host_tile(rng, x_size, d_size, 1.0))
    for tile in (gpu, other):
        tile.forward(x, False)
    torch.cuda.synchronize()
    before = lib().rpu_device_allocation_count()
    state = gpu.dump_extra()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = gpu.forward(x, False, False, False, False, True)
    assert lib().rpu_device_allocation_count() == before
    for replay in range(3):
        graph.replay()
        torch.cuda.synchronize()
        other.load_extra(state, True)
        assert torch.equal(y, other.forward(x, False))


# backward calls of more multiply-adds than the small ones: inputs are the tile's outputs
@pytest.mark.parametrize("x_size,d_size,batch", [(300, 600, 400), (1000, 1000, 100), (257, 2048, 150), (785, 300, 420)])
def test_backward_in_one_launch(gpu_device, x_size, d_size, batch):
    rng = np.random.default_rng(x_size)
    pair = pair_of(host_tile(rng, x_size, d_size, 12.0))
    d = torch.from_numpy(rng.normal(0, 0.05, (batch, d_size)).astype(np.float32)).cuda()
    (g, names), (g_other, names_other) = (names_of(t, lambda t: t.backward(d, False)) for t in pair)
    assert names == ["mvm_whole"] and "mvm_whole" not in names_other
    assert torch.equal(g, g_other)


# settings of the converters and the order of inputs and outputs in memory
@pytest.mark.parametrize("settings", [
    dict(nm=NM.NONE), dict(nm=NM.Constant, nm_thres=0.7), dict(nm=NM.Max), dict(inp_asymmetry=0.3, out_asymmetry=0.2),
    dict(inp_res=-1.0), dict(out_res=-1.0, out_noise=0.0), dict(bm_test_negative_bound=False)])
@pytest.mark.parametrize("trans", [False, True])
def test_settings_and_orders(gpu_device, settings, trans):
    rng = np.random.default_rng(5)
    x_size, d_size, batch = 300, 270, 203
    pair = pair_of(host_tile(rng, x_size, d_size, 4.0, **settings))
    most = 0
    for call in range(2):
        x = torch.from_numpy(rng.uniform(-1, 1, (x_size, batch) if trans else (batch, x_size)).astype(np.float32)).cuda()
        (y, names), (y_other, _) = (names_of(t, lambda t: t.forward(x, False, trans, trans)) for t in pair)
        assert names == ["mvm_whole"] or most >= 4   # (rounds beyond the first three: the next call takes the others)
        assert torch.equal(y, y_other)
        assert torch.equal(pair[0].get_bm_rounds(batch), pair[1].get_bm_rounds(batch))
        most = int(pair[0].get_bm_rounds(batch).max())


@binds
def test_rows_that_are_not_finite_stay_to_themselves(gpu_device):
    """A weight that is not finite reaches the outputs of its own row and no others (rows of 300 end within a step)."""
    rng = np.random.default_rng(2)
    pair = pair_of(host_tile(rng, 300, 270, 1e6))
    x = torch.from_numpy(rng.uniform(-1, 1, (203, 300)).astype(np.float32)).cuda()
    for tile in pair:
        tile.live = torch.empty(270, 300, device="cuda")
        tile.set_shared_weights_row_major(tile.live)
        torch.cuda.synchronize()
        tile.live[100, 0:40] = float("nan")
    y, y_other = (t.forward(x, False) for t in pair)
    keep = torch.arange(270) != 100
    assert bool(torch.isfinite(y[:, keep]).all()) and torch.equal(y[:, keep], y_other[:, keep])


@pytest.mark.parametrize("warm", [False, True])
def test_captured_after_a_larger_call(gpu_device, warm):
    """The captured call makes no room, whether or not a call before it has (round by round, or three together); replays, with eager
    calls between them, find counters and marks as they have to be."""
    rng = np.random.default_rng(8)
    host = host_tile(rng, 300, 512, 4.0)
    gpu, other = pair_of(host)
    for tile in (gpu, other):
        tile.forward(torch.zeros(4096, 300, device="cuda"), False)
    x_dev = torch.zeros(140, 300, device="cuda")
    if warm:
        gpu.forward(x_dev, False)
    torch.cuda.synchronize()
    before = lib().rpu_device_allocation_count()
    state = gpu.dump_extra()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_dev = gpu.forward(x_dev, False, False, False, False, True)
    for replay in range(4):
        x = torch.from_numpy(rng.uniform(-1, 1, (140, 300)).astype(np.float32)).cuda()
        if replay % 2 and warm:
            gpu.forward(x[:100], False)
        x_dev.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert lib().rpu_device_allocation_count() == before
        other.load_extra(state, True)         # a replay draws what the captured call drew
        assert torch.equal(y_dev, other.forward(x, False))
        before = lib().rpu_device_allocation_count()

