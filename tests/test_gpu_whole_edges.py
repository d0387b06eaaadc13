"""Edges of the one launch of medium batches (k_mvm_whole): few samples, strides that coincide, converters of more steps than its
division is exact for, inputs at the ends of their range, rounds that it leaves to one workgroup.  Compared bit for bit with the
launches that such calls take otherwise."""
import numpy as np
import pytest
import torch

from aihwkit_amd.rpu_base import tiles
from test_gpu_whole_calls import NM, binds, host_tile, names_of, pair_of

pytestmark = pytest.mark.gpu


def without_small_calls(tile, rng):
    """Puts the tile into a group with one whose rows are too long for the launch of small batches: its own calls of few samples
    then take the launch of medium ones."""
    return tiles.TileGroup([tile, tiles.CudaAnalogTile(host_tile(rng, 2100, 16, 12.0))])


# one sample with transposed output has strides of one element both ways; 13.3 million weights are too many
# for the launch of small batches
@pytest.mark.parametrize("x_size,d_size,batch,grouped", [
    (300, 270, 1, True), (300, 270, 5, True), (300, 270, 15, True), (512, 512, 16, True), (100, 70, 17, True), (300, 20, 1, True),
    (300, 17, 1, True), (96, 30000, 1, True), (512, 26000, 1, False)])
@pytest.mark.parametrize("trans", [False, True])
def test_few_samples(gpu_device, x_size, d_size, batch, grouped, trans):
    rng = np.random.default_rng(x_size + d_size + batch)
    spread = 0.2 * np.sqrt(x_size)
    stood = set()
    for out_bound in (0.45 * spread, 0.9 * spread, 1.5 * spread, 2.4 * spread, 100.0 * spread):
        pair = pair_of(host_tile(rng, x_size, d_size, out_bound))
        group = without_small_calls(pair[0], rng) if grouped else None
        for call in range(3):
            x = torch.from_numpy(rng.uniform(-1, 1, (x_size, batch) if trans else (batch, x_size)).astype(np.float32)).cuda()
            (y, names), (y_other, names_other) = (names_of(t, lambda t: t.forward(x, False, trans, trans)) for t in pair)
            rounds = pair[0].get_bm_rounds(batch)
            if names == ["mvm_whole"]:
                stood.update(rounds.tolist())
            assert "mvm_whole" not in names_other
            assert torch.equal(y, y_other), (out_bound, call)
            assert torch.equal(rounds, pair[1].get_bm_rounds(batch))
        del group
    assert {1, 2, 3} <= stood


# steps of a converter: more than 2^60, and as many as its rule still lets through
@pytest.mark.parametrize("settings", [dict(inp_res=3e-19), dict(out_res=3e-19, out_noise=0.0), dict(inp_res=1 / 1.1e18),
                                      dict(out_res=1 / 1.1e18, out_noise=0.0)])
def test_converters_of_many_steps(gpu_device, settings):
    rng = np.random.default_rng(7)
    x_size, d_size, batch = 300, 600, 203
    pair = pair_of(host_tile(rng, x_size, d_size, 30.0, **settings))
    for call in range(2):
        x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)).cuda()
        d = torch.from_numpy(rng.normal(0, 0.05, (400, d_size)).astype(np.float32)).cuda()
        y, y_other = (t.forward(x, False) for t in pair)
        assert torch.equal(y, y_other)
        g, g_other = (t.backward(d, False) for t in pair)
        assert torch.equal(g, g_other)


# gradients so small that the factor of their noise management is infinite, on rows that end within a step of the contraction and on
# whole ones; and values that are not numbers: the rest of the batch is as ever, and so are the rows themselves
@pytest.mark.parametrize("x_size,d_size,batch", [(300, 270, 800), (300, 300, 700), (200, 512, 600)])
@pytest.mark.parametrize("value", [1e-40, 1e-38, 3e38, float("inf"), float("nan")])
def test_inputs_at_the_ends_of_their_range(gpu_device, x_size, d_size, batch, value):
    rng = np.random.default_rng(d_size)
    pair = pair_of(host_tile(rng, x_size, d_size, 12.0))
    d = rng.normal(0, 0.05, (batch, d_size)).astype(np.float32)
    d[17] = value
    d[18] = value * np.sign(d[18])
    d[19, 5] = value
    x = rng.normal(0, 0.05, (203, x_size)).astype(np.float32)
    x[17] = value
    x[18] = value * np.sign(x[18])
    x[19, 5] = value
    d, x = torch.from_numpy(d).cuda(), torch.from_numpy(x).cuda()
    (g, names), (g_other, _) = (names_of(t, lambda t: t.backward(d, False)) for t in pair)
    assert names == ["mvm_whole"]
    assert torch.equal(torch.nan_to_num(g, 1e30), torch.nan_to_num(g_other, 1e30))
    (y, names), (y_other, _) = (names_of(t, lambda t: t.forward(x, False)) for t in pair)
    assert names == ["mvm_whole"] or d_size > x_size
    assert torch.equal(torch.nan_to_num(y, 1e30), torch.nan_to_num(y_other, 1e30))


def microseconds(call, calls=40):
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    call()
    torch.cuda.synchronize()
    start.record()
    for _ in range(calls):
        call()
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) * 1000 / calls


# 1500 x 1500, 10 samples: a round that one workgroup runs alone takes 400 us, the launches of the others 25 to 45.  two: there are no more
# than two rounds; captured: without saturation, replayed with it; alternating: calls without saturation, now and then one with it
@binds
@pytest.mark.parametrize("program", ["two", "captured", "alternating"])
def test_no_rounds_are_left_alone_time_and_again(gpu_device, program):
    rng = np.random.default_rng(1)
    x_size, d_size, batch = 1500, 1500, 10
    pair = pair_of(host_tile(rng, x_size, d_size, 4.0, **(dict(max_bm_factor=1) if program == "two" else {})))
    x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size)).astype(np.float32)).cuda()
    weights = torch.from_numpy(rng.uniform(-1, 1, (d_size, x_size)).astype(np.float32)).cuda()
    weights /= float((x / x.abs().amax(dim=1, keepdim=True) @ weights.t()).abs().amax())   # largest output of a sample: up to 1
    calm, saturating = weights, weights * (6.0 if program != "alternating" else 12.0)       # beyond 4, beyond 8
    took, results, graphs = [], [], []
    for tile in pair:
        tile.live = torch.empty(d_size, x_size, device="cuda")
        tile.set_shared_weights_row_major(tile.live)
        tile.live.copy_(calm)
        torch.cuda.synchronize()

        def forward():
            return tile.forward(x, False, False, False, False, True)

        if program == "two":
            tile.live.copy_(saturating)
            call = forward
        elif program == "captured":
            for _ in range(12):
                forward()
            torch.cuda.synchronize()
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1]):
                y = forward()
            tile.live.copy_(saturating)
            graph = graphs[-1]

            def call():
                graph.replay()
                return y
        else:
            def call():
                tile.live.copy_(saturating)
                y = forward()
                tile.live.copy_(calm)
                for _ in range(10):
                    forward()
                return y
        torch.cuda.synchronize()
        took.append(min(microseconds(call) for _ in range(3)))
        results.append(call().clone())
        if program != "alternating":
            assert int(tile.get_bm_rounds(batch).max()) == 2
    assert torch.equal(*results)
    assert took[0] < 1.5 * took[1], took


def test_padded_rows(gpu_device):
    """Rows of inputs and outputs that are slices of wider ones: a group whose tiles run one by one (running averages) takes the launch
    for the others, and what lies between the rows stays as it was."""
    rng = np.random.default_rng(12)
    x_size, d_size, batch = 300, 270, 203
    host = host_tile(rng, x_size, d_size, 1.7 * 0.2 * np.sqrt(x_size))
    x = torch.from_numpy(rng.uniform(-1, 1, (batch, x_size + 7)).astype(np.float32)).cuda()
    results = []
    for tile in pair_of(host):
        average = tiles.CudaAnalogTile(host_tile(rng, 64, 32, 12.0, nm=NM.AverageAbsMax))
        group = tiles.TileGroup([tile, average])
        wide = torch.full((batch, d_size + 13), 5.0, device="cuda")
        other = torch.empty(batch, 32, device="cuda")
        took = []
        for _ in range(2):
            _, names = names_of(tile, lambda t: group.forward([x[:, 3:3 + x_size], x[:, :64]], outs=[wide[:, :d_size], other]))
            took.append(names == ["mvm_whole"])
        assert bool((wide[:, d_size:] == 5.0).all())
        results.append((wide, tile.get_bm_rounds(batch), took))
    assert any(results[0][2]) and not any(results[1][2])
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert int(results[0][1].max()) > 1
