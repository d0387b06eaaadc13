"""Small batches run noise management, conversion, contraction and all bound-management rounds in one launch (k_mvm_few).
Exact-arithmetic setting: outputs and round counts equal the oracle's bit for bit, whatever the blocks of the launch."""
import ctypes as C

import numpy as np
import pytest
import torch

from aihwkit_amd._cabi import lib
from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles
from helpers import build_pair, constant_step, io_params, make_meta, noise_free_io

pytestmark = pytest.mark.gpu
F = np.float32
NM, BM = dv.NoiseManagementType, dv.BoundManagementType


def grid(rng, top, shape, unit):
    return (rng.integers(-top, top + 1, shape) / unit).astype(F)


def exact_pair(rng, x_size, d_size, out_bound, w_top, seed=1):
    f_io = noise_free_io(inp_res=1 / 64.0, out_res=1 / 512.0, noise_management=NM.AbsMax, bound_management=BM.Iterative,
                         out_bound=out_bound)
    b_io = noise_free_io(inp_res=1 / 64.0, out_res=1 / 512.0, noise_management=NM.Max)
    dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=seed)
    host, orc, _ = build_pair(make_meta(f_io, b_io), dev, x_size, d_size, gpu=False)
    w = grid(rng, w_top, (d_size, x_size), 64.0)
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    return host, orc


# x_size, d_size, batch, bias: lengths on both sides of a load (64 inputs), of a block (16, 32, 64 outputs; 1, 2, 4 samples),
# of eight blocks of outputs, one workgroup for a sample, the longest rows; the last ones take the larger blocks
@pytest.mark.parametrize("x_size,d_size,batch,bias", [
    (1, 1, 1, False), (2, 3, 2, True), (63, 15, 3, False), (64, 16, 1, False), (65, 17, 5, True), (130, 128, 1, False),
    (257, 129, 2, False), (2048, 33, 3, False), (2048, 257, 16, False), (300, 512, 7, True), (200, 65, 101, False),
    (96, 257, 130, False), (129, 10, 1027, False)])
def test_small_calls_equal_the_oracle(gpu_device, x_size, d_size, batch, bias):
    rng = np.random.default_rng(x_size * 1000 + d_size)
    host, orc = exact_pair(rng, x_size, d_size, 1.0, 16)
    x = grid(rng, 64, (batch, x_size - int(bias)), 64.0)
    x *= rng.choice([0.0, 1 / 64.0, 1.0, 1.0], (batch, 1)).astype(F) if batch > 2 else F(1.0)
    x[:, : x.shape[1] // 2] *= rng.choice([0.0, 1.0], (batch, 1)).astype(F)
    d = grid(rng, 64, (batch, d_size), 64.0)
    y_o, g_o = orc.forward(x, bias), orc.backward(d, bias)
    rounds = orc.bm_rounds(batch)
    for mode in (0, 1, -1):                          # rounds one by one, rounds 0 to 2 together, by the calls before
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_fused_rounds(mode)
        for _ in range(2):                           # the second call finds the counters and marks of the first
            gpu.set_profiling(True)
            y = gpu.forward(torch.from_numpy(x).cuda(), bias).cpu().numpy()
            assert [name for name, _ms in gpu.get_profile()][1:] == ["mvm_few"]
            gpu.set_profiling(False)
            assert np.array_equal(y, y_o)
            assert np.array_equal(gpu.get_bm_rounds(batch).numpy(), rounds)
            assert np.array_equal(gpu.backward(torch.from_numpy(d).cuda(), bias).cpu().numpy(), g_o)


# batch, shapes: small calls next to others that share their input's quantized rows; next to tiles of the large-tile kernel;
# the largest blocks with the longest rows, which take the most LDS
@pytest.mark.parametrize("batch,shapes,others", [
    (128, [(257, 16), (257, 512), (257, 33), (257, 600), (64, 16)], ()),
    (60, [(257, 16), (257, 512), (257, 33), (257, 600), (64, 16)], (1, 3)),
    (1024, [(40, 130)] * 8 + [(64, 256)] * 2 + [(64, 40), (64, 30), (33, 20)], ()),
    (5, [(130, 16), (130, 200), (2048, 40), (1, 1)], ()), (16, [(2048, 300)] * 13, ())])
def test_groups_with_small_calls_equal_the_oracle(gpu_device, batch, shapes, others):
    rng = np.random.default_rng(batch)
    pairs = [exact_pair(rng, x, d, 2.0, 32, seed=k + 1) for k, (x, d) in enumerate(shapes)]
    grouped = [tiles.CudaAnalogTile(host) for host, _ in pairs]
    for k in others:
        grouped[k].set_small_calls(False)
    group = tiles.TileGroup(grouped)
    by_size = {x: grid(rng, 64, (batch, x), 64.0) for x, _ in shapes}
    ds = [grid(rng, 64, (batch, d), 64.0) for _, d in shapes]
    x_dev = {n: torch.from_numpy(x).cuda() for n, x in by_size.items()}
    for _ in range(2):
        got = group.forward([x_dev[x] for x, _ in shapes])
        rounds = [t.get_bm_rounds(batch).numpy().copy() for t in grouped]
        back = group.backward([torch.from_numpy(d).cuda() for d in ds])
        for (x, _), (_, orc), r, y, d, g in zip(shapes, pairs, rounds, got, ds, back):
            assert np.array_equal(y.cpu().numpy(), orc.forward(by_size[x]))
            assert np.array_equal(r, orc.bm_rounds(batch))
            assert np.array_equal(g.cpu().numpy(), orc.backward(d))


# 40 tiles with one block of outputs each, of four samples: twelve of those to a tile fill the GPU (two to a CU).  With noise,
# so that a sum in another order would show in the bits of some output; a shared input, so that the other launches show too
@pytest.mark.parametrize("mixed", [False, True])
def test_groups_take_one_launch_up_to_what_the_gpu_holds(gpu_device, mixed):
    rng = np.random.default_rng(9)
    io = dict(inp_res=1 / 127.0, out_res=-1.0, out_noise=0.1, noise_management=NM.AbsMax)
    meta = make_meta(io_params(bound_management=BM.Iterative, out_bound=4.0, **io), io_params(**io))
    sizes = [(96, 64)] * 39 + [(96, 1800 if mixed else 64)]     # alone, the large one takes other launches from 70 samples on
    grouped = []
    for k, (x_size, d_size) in enumerate(sizes):
        host, _orc, _ = build_pair(meta, constant_step(construction_seed=k + 1), x_size, d_size, gpu=False)
        host.set_weights(torch.from_numpy(rng.uniform(-0.5, 0.5, (d_size, x_size)).astype(F)))
        grouped.append(tiles.CudaAnalogTile(host))
    cus = torch.cuda.get_device_properties(0).multi_processor_count

    def one_launch(tile, x):
        tile.set_profiling(True)
        y = tile.forward(x, False)
        names = [name for name, _ms in tile.get_profile()][1:]
        tile.set_profiling(False)
        return y, names == ["mvm_few"]

    blocks = 39 + (32 if mixed else 1)                           # 1800 outputs: 29 blocks, an eighth of them to each XCD
    largest = 4 * (2 * cus // blocks)
    before = torch.from_numpy(rng.uniform(-1, 1, (largest + 1, 96)).astype(F)).cuda()
    assert one_launch(grouped[0], before)[1]                     # a tile of no group: up to its own limit
    group = tiles.TileGroup(grouped)
    for batch in (largest, largest + 1):
        x = torch.from_numpy(rng.uniform(-1, 1, (batch, 96)).astype(F)).cuda()
        for k, t in enumerate(grouped):
            t.set_seed(100 + k)
        got = group.forward([x] * len(grouped))
        assert group.get_shared_input_sets() == ((0, 0) if batch == largest else (1, 40))
        for k, (t, y) in enumerate(zip(grouped, got)):
            t.set_seed(100 + k)
            alone, small = one_launch(t, x)
            assert small == (batch == largest)
            assert torch.equal(alone, y)                         # the same sums as in the call of the group
        d = [torch.from_numpy(rng.uniform(-1, 1, (batch, n)).astype(F)).cuda() for _, n in sizes]
        for k, t in enumerate(grouped):
            t.set_seed(200 + k)
        back = group.backward(d)
        for k, (t, g, v) in enumerate(zip(grouped, d, back)):
            t.set_seed(200 + k)
            assert torch.equal(t.backward(g, False), v)


def test_small_calls_share_no_quantized_rows(gpu_device):
    """Tiles with the same input: a call in one launch writes no rows that they could share, the other launches do."""
    rng = np.random.default_rng(4)
    grouped = [tiles.CudaAnalogTile(exact_pair(rng, 96, 40, 2.0, 32)[0]) for _ in range(3)]
    group = tiles.TileGroup(grouped)
    x = torch.from_numpy(grid(rng, 64, (5, 96), 64.0)).cuda()
    small = group.forward([x] * 3)
    assert group.get_shared_input_sets() == (0, 0)
    for t in grouped:
        t.set_small_calls(False)
    other = group.forward([x] * 3)
    assert group.get_shared_input_sets() == (1, 3)
    for y, z in zip(small, other):
        assert torch.equal(y, z)


# a program that has warmed up on its largest batch captures smaller ones: they find their scratch there
@pytest.mark.parametrize("grouped", [False, True])
def test_small_calls_after_larger_ones_allocate_nothing(gpu_device, grouped):
    rng = np.random.default_rng(0)
    host, orc = exact_pair(rng, 300, 512, 1.0, 16)
    gpu = tiles.CudaAnalogTile(host)
    group = tiles.TileGroup([gpu])

    def forward(x):
        return group.forward([x])[0] if grouped else gpu.forward(x, False)

    for batch in (1024, 1024, 1024):
        forward(torch.from_numpy(grid(rng, 64, (batch, 300), 64.0)).cuda())
    torch.cuda.synchronize()
    before = lib().rpu_device_allocation_count()
    for batch in (7, 32, 1):
        x = grid(rng, 64, (batch, 300), 64.0)
        assert np.array_equal(forward(torch.from_numpy(x).cuda()).cpu().numpy(), orc.forward(x))
    assert lib().rpu_device_allocation_count() == before


def test_small_calls_captured_after_a_larger_one(gpu_device):
    """The tile's first small call is captured, after a larger call only; replays on new inputs, with eager small calls and
    synchronizations between them, find counters and marks as they have to be."""
    rng = np.random.default_rng(8)
    host, orc = exact_pair(rng, 300, 512, 0.5, 16)
    gpu = tiles.CudaAnalogTile(host)
    gpu.forward(torch.from_numpy(grid(rng, 64, (1024, 300), 64.0)).cuda(), False)
    x_dev = torch.zeros(7, 300, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_dev = gpu.forward(x_dev, False, False, False, False, True)
    most = 0
    for replay in range(5):
        x = grid(rng, 64, (7, 300), 64.0)
        if replay % 2:                                           # before and after replays: a call that is not captured
            assert np.array_equal(gpu.forward(torch.from_numpy(x).cuda(), False).cpu().numpy(), orc.forward(x))
        x_dev.copy_(torch.from_numpy(x))
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y_dev.cpu().numpy(), orc.forward(x))
        assert np.array_equal(gpu.get_bm_rounds(7).numpy(), orc.bm_rounds(7))
        most = max(most, int(orc.bm_rounds(7).max()))
    assert most >= 3


def test_larger_calls_make_no_room_for_small_ones(gpu_device):
    """The first call of a tile allocates the same number of buffers whether or not it could have small calls after it, and
    more outputs than inputs (the results of rounds 1 and 2 are rows of outputs) still find their room."""
    rng = np.random.default_rng(3)
    allocations = []
    for small in (True, False):
        host, orc = exact_pair(rng, 40, 500, 0.5, 16)             # rounds 1 and 2 have samples
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_small_calls(small)
        x = grid(rng, 64, (700, 40), 64.0)
        before = lib().rpu_device_allocation_count()
        assert np.array_equal(gpu.forward(torch.from_numpy(x).cuda(), False).cpu().numpy(), orc.forward(x))
        allocations.append(lib().rpu_device_allocation_count() - before)
        before = lib().rpu_device_allocation_count()
        for batch in (200, 3):
            y = gpu.forward(torch.from_numpy(x[:batch]).cuda(), False).cpu().numpy()
            assert np.array_equal(y, orc.forward(x[:batch])) and orc.bm_rounds(batch).max() >= 3
        assert lib().rpu_device_allocation_count() == before or not small
    assert allocations[0] == allocations[1]


# outputs that lie over the inputs of the call (of another tile of the group): the inputs are read before anything is stored
@pytest.mark.parametrize("size,batch", [(200, 7), (64, 3)])
def test_small_calls_onto_their_own_input_equal_the_oracle(gpu_device, size, batch):
    rng = np.random.default_rng(size)
    host, orc = exact_pair(rng, size, size, 8.0, 16)
    gpu, other = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    x = grid(rng, 64, (batch, size), 64.0)
    want = orc.forward(x)
    assert np.any(want) and orc.bm_rounds(batch).max() == 1   # a second round reads the inputs again
    buf = torch.from_numpy(x).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    assert lib().rpu_tile_forward(gpu._h, buf.data_ptr(), buf.data_ptr(), batch, 0, 0, 0, 0, stream) == 0
    assert np.array_equal(buf.cpu().numpy(), want)
    first, second = torch.from_numpy(x).cuda(), torch.from_numpy(x).cuda()
    group = tiles.TileGroup([gpu, other])
    ins = (C.c_void_p * 2)(first.data_ptr(), second.data_ptr())
    outs = (C.c_void_p * 2)(second.data_ptr(), first.data_ptr())
    assert lib().rpu_group_forward(group._g, ins, outs, batch, 0, stream) == 0
    assert np.array_equal(first.cpu().numpy(), want) and np.array_equal(second.cpu().numpy(), want)


# input and outputs as column slices of one matrix: their rows interleave, but no element is both; then outputs that begin on
# the last column of the input, which every tile has to read before any stores.  (The tiles that take the one launch quantize
# their rows for themselves, the others share them.)
@pytest.mark.parametrize("over,sets", [(0, (0, 0)), (1, (1, 2))])
def test_small_calls_on_interleaved_columns(gpu_device, over, sets):
    rng = np.random.default_rng(12)
    batch, x_size, outs = 7, 96, (64, 33)
    pairs = [exact_pair(rng, x_size, d, 8.0 if over else 2.0, 16, seed=k + 1) for k, d in enumerate(outs)]
    group = tiles.TileGroup([tiles.CudaAnalogTile(host) for host, _ in pairs])
    buf = torch.from_numpy(grid(rng, 64, (batch, 4 + x_size + sum(outs) + 5), 64.0)).cuda()
    x = buf[:, 4:4 + x_size]
    want = [orc.forward(x.cpu().numpy().copy()) for _, orc in pairs]
    assert not over or max(orc.bm_rounds(batch).max() for _, orc in pairs) == 1   # a second round reads the inputs again
    at = 4 + x_size - over
    ys = [buf[:, at:at + outs[0]], buf[:, at + outs[0]:at + sum(outs)]]
    group.forward([x, x], outs=ys)
    assert group.get_shared_input_sets() == sets
    for y, w in zip(ys, want):
        assert np.array_equal(y.cpu().numpy(), w)


# What is random in the converters, drawn for element, sample and round: a tile of the same seed in the launches of larger
# batches draws the same.  Weights and inputs on a grid, so that sums in any order are the same bits; only noise on the inputs
# takes them off it: sums of at most 300 terms below 1, each partial sum off by half an ulp of at most 2^-15 (300 < 2^9)
@pytest.mark.parametrize("settings,off", [
    (dict(out_noise=0.06), 0.0), (dict(inp_sto_round=True), 0.0), (dict(out_sto_round=True), 0.0),
    (dict(out_noise=0.2, out_asymmetry=0.1, inp_asymmetry=0.5, out_res=-1.0), 0.0),
    (dict(inp_noise=0.02, out_res=-1.0), 300 * 2.0 ** -16)])
@pytest.mark.parametrize("x_size,d_size,batch,bias", [(130, 128, 1, False), (300, 512, 7, True), (64, 700, 3, False), (200, 65, 101, False)])
def test_small_calls_draw_what_larger_ones_draw(gpu_device, settings, off, x_size, d_size, batch, bias):
    rng = np.random.default_rng(x_size)
    f_io = noise_free_io(**{**dict(inp_res=1 / 64.0, out_res=1 / 512.0, noise_management=NM.AbsMax,
                                   bound_management=BM.Iterative, out_bound=1.0), **settings})
    b_io = noise_free_io(**{**dict(inp_res=1 / 64.0, out_res=1 / 512.0, noise_management=NM.Max), **settings})
    dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=1)
    host, _orc, _ = build_pair(make_meta(f_io, b_io), dev, x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(grid(rng, 16, (d_size, x_size), 64.0)))
    x = torch.from_numpy(grid(rng, 64, (batch, x_size - int(bias)), 64.0)).cuda()
    d = torch.from_numpy(grid(rng, 64, (batch, d_size), 64.0)).cuda()
    for mode in (0, 1):                              # round by round, rounds 0 to 2 together
        tile = tiles.CudaAnalogTile(host)
        tile.set_fused_rounds(mode)
        got = []
        for small in (False, True):
            tile.set_small_calls(small)
            tile.set_seed(11)
            tile.set_profiling(True)
            y = tile.forward(x, bias)
            assert ([name for name, _ms in tile.get_profile()][1:] == ["mvm_few"]) == small
            tile.set_profiling(False)
            got.append((y, tile.get_bm_rounds(batch), tile.backward(d, bias)))
        (y0, r0, g0), (y1, r1, g1) = got
        assert torch.equal(r0, r1) and r0.max() >= 3
        # (the output of a sample is scaled back by what its rounds scaled the input down)
        scale = float(y0.abs().max()) if off else 1.0
        assert float((y0 - y1).abs().max()) <= off * scale and float((g0 - g1).abs().max()) <= off
        assert not off or float((y0 - y1).abs().max()) > 0.0      # noise did take them off the grid
