"""Contraction of the large-tile kernel on the bf16 matrix pipe (operands split into bf16 parts without loss) against
64-bit sums: inputs on the DAC grid (one part), any other inputs (three parts), and values that only the fp32 pipe takes."""
import numpy as np
import pytest
import torch

from helpers import make_meta, noise_free_io
from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles

pytestmark = pytest.mark.gpu

# workgroup tiles of 64 x 128, 64 x 64, 128 x 64 and 128 x 128 outputs x samples, contraction stages of 32, each with a
# remainder; at least one 64 x 64 tile per CU, or the 32 x 32 kernel runs the call
SHAPES = [(33, 64, 16384), (65, 65, 16400), (433, 48, 16500), (31, 129, 5505), (160, 1003, 1601), (513, 257, 3401),
          (1024, 128, 8193), (1001, 1000, 4100), (96, 1000, 8192)]


def _tile(x_size, d_size, io, w):
    meta = make_meta(io, io, pulse_type=dv.PulseType.NONE)
    host = meta.create_array(x_size, d_size, dv.IdealResistiveDeviceParameter())
    host.set_weights(torch.from_numpy(w))
    return tiles.CudaAnalogTile(host)


def _close(got, want, terms, lengths, n=None):
    """A sum of n products in fp32 is off by at most (n + 2) half units of the sum of the absolute products; random signs
    leave far less than a quarter of that bound.  Over all sums: n / 2 roundings of sums no larger than the last one, each
    off by 2^-24 / sqrt(3) of it (root mean square), and two more of the operand and of the result.  A lost low part would
    show: 2^-18 of every product."""
    error = np.abs(got.double().cpu().numpy() - want)
    bound = 0.25 * (lengths + 2) * 2.0 ** -24 * terms + 1e-37
    assert np.all(error <= bound)
    roundings = (lengths if n is None else n) / 2 + 2
    assert np.sqrt(np.mean(error ** 2)) <= 2.0 ** -24 * np.sqrt(roundings / 3 * np.mean(want ** 2))


@pytest.mark.parametrize("scale", [0.3, 1e-12, 1e10])
@pytest.mark.parametrize("x_size,d_size,batch", SHAPES)
def test_unquantized_products_against_64_bit_sums(gpu_device, x_size, d_size, batch, scale):
    rng = np.random.default_rng(x_size)
    io = noise_free_io()
    io.is_perfect = True
    w = (scale * rng.standard_normal((d_size, x_size))).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    x = rng.standard_normal((batch, x_size)).astype(np.float32)
    d = rng.standard_normal((batch, d_size)).astype(np.float32)
    w64 = w.astype(np.float64)
    _close(tile.forward(torch.from_numpy(x).cuda()), x @ w64.T, np.abs(x) @ np.abs(w64).T, x_size)
    _close(tile.backward(torch.from_numpy(d).cuda()), d @ w64, np.abs(d) @ np.abs(w64), d_size)


@pytest.mark.parametrize("x_size,d_size,batch", SHAPES)
@pytest.mark.parametrize("steps", [63, 256, 300])  # of the DAC on either side of zero: the last is not held by one bf16
def test_quantized_products_against_64_bit_sums(gpu_device, x_size, d_size, batch, steps):
    rng = np.random.default_rng(d_size)
    io = noise_free_io(inp_res=1.0 / (2 * steps))
    io.out_res, io.out_bound = -1.0, float("inf")
    w = rng.uniform(-0.6, 0.6, (d_size, x_size)).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    w64 = w.astype(np.float64)
    step = np.float32(2.0 * np.float32(1.0 / (2 * steps)))  # the range is [-1, 1]
    for call, width, axis in ((tile.forward, x_size, w64.T), (tile.backward, d_size, w64)):
        v = rng.uniform(-1.0, 1.0, (batch, width)).astype(np.float32)
        # away from the middle between two steps, where the fp32 quotient may round to either; the range itself is met
        k = np.rint(v / step)
        v = ((k + np.clip(v / step - k, -0.4, 0.4)) * step).astype(np.float32)
        v[:, 0] = 1.0
        q = np.clip(np.rint(v / step), -steps, steps).astype(np.float64) * float(step)
        got = call(torch.from_numpy(v).cuda())
        # the reference's own rounding of k * step and of the clipped range: one half unit per product
        _close(got, q @ axis, np.abs(q) @ np.abs(axis), 4 * width + 16, width)


@pytest.mark.parametrize("x_size,d_size,batch", [(100, 50, 16500), (256, 256, 4100), (300, 300, 12000)])
def test_values_out_of_the_range_of_the_parts(gpu_device, x_size, d_size, batch):
    """Infinities, NaN and values near the end of the fp32 range give what fp32 products give."""
    rng = np.random.default_rng(1)
    io = noise_free_io()
    io.is_perfect = True
    w = rng.uniform(-0.5, 0.5, (d_size, x_size)).astype(np.float32)
    w[3, 7], w[40, 9], w[5, 5], w[6, 6], w[7, -1] = np.inf, -np.inf, 3.4e38, np.nan, 2e38
    tile = _tile(x_size, d_size, io, w)
    x = (rng.random((batch, x_size)) + 0.5).astype(np.float32)
    x[10, 3], x[11, 3], x[12, 1], x[13, 0] = np.inf, 3e38, np.nan, -np.inf
    with np.errstate(all="ignore"):
        want = (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)
    got = tile.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    # the bound of _close: where products of 1e38 cancel, the error is relative to them and not to what is left
    with np.errstate(all="ignore"):
        bound = (x_size + 2) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T)
        assert np.all((np.abs(got.astype(np.float64) - want) <= bound + 1e-37)[fine])


def _chain(x, w):
    """x w^T as multiply-adds of two terms at a time in fp32, as the fp32 matrix pipe makes it."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    if x.shape[1] % 2:
        x, w = np.pad(x, ((0, 0), (0, 1))), np.pad(w, ((0, 0), (0, 1)))
    acc = np.zeros((x.shape[0], w.shape[0]), np.float32)
    for k in range(0, x.shape[1], 2):
        acc = (acc + (np.outer(x[:, k], w[:, k]) + np.outer(x[:, k + 1], w[:, k + 1]))).astype(np.float32)
    return acc


@pytest.mark.parametrize("stepped", [False, True])
@pytest.mark.parametrize("terms", [1, 2, 3, 5, 8, 15, 16, 17, 27, 32, 33, 64, 433, 1024])
def test_no_further_from_64_bit_sums_than_a_chain_in_fp32(gpu_device, terms, stepped):
    """Root mean square error over 256 x 64 outputs; the two that are compared are each known to 1 / sqrt(2 * 16384)."""
    rng = np.random.default_rng(terms)
    out_size, batch, steps = 64, 16384, 63
    io = noise_free_io(inp_res=1.0 / (2 * steps) if stepped else -1.0)
    io.out_res, io.out_bound, io.is_perfect = -1.0, float("inf"), not stepped
    w = rng.uniform(-0.6, 0.6, (out_size, terms)).astype(np.float32)
    x = rng.uniform(-1.0, 1.0, (batch, terms)).astype(np.float32)
    want_x = x.astype(np.float64)
    if stepped:
        x[:, 0] = 1.0  # meets the range
        step = np.float32(2.0 * np.float32(1.0 / (2 * steps)))
        want_x = np.rint(x / step).astype(np.float64) * float(step)
        x = want_x.astype(np.float32)
    some = slice(0, batch, batch // 256)
    want = want_x[some] @ w.T.astype(np.float64)
    chain = np.sqrt(np.mean((_chain(x[some], w) - want) ** 2))
    forward = _tile(terms, out_size, io, w).forward(torch.from_numpy(x).cuda())
    backward = _tile(out_size, terms, io, np.ascontiguousarray(w.T)).backward(torch.from_numpy(x).cuda())
    for got in (forward, backward):
        error = np.sqrt(np.mean((got[some].double().cpu().numpy() - want) ** 2))
        assert error <= 1.04 * chain


@pytest.mark.parametrize("small", ["weights", "inputs", "weights of quantized inputs"])
@pytest.mark.parametrize("x_size,d_size,batch", [(40, 64, 16500), (433, 48, 16500), (513, 257, 3401)])
def test_values_near_the_lower_end_of_the_range(gpu_device, x_size, d_size, batch, small):
    """An operand times 2^-120 gives 2^-120 times the result: the operands keep all their bits (multiples of 2^-144).
    Where the result and its scaling are below the range of normal floats, each is rounded to a multiple of 2^-149."""
    rng = np.random.default_rng(x_size)
    quantized = small == "weights of quantized inputs"
    io = noise_free_io(inp_res=1.0 / 126 if quantized else -1.0)
    io.out_res, io.out_bound, io.is_perfect = -1.0, float("inf"), not quantized
    w = (rng.integers(-2 ** 23, 2 ** 23, (d_size, x_size)) * 2.0 ** -24).astype(np.float32)
    tiny = np.float32(2.0 ** -120)
    normal, low = _tile(x_size, d_size, io, w), _tile(x_size, d_size, io, w if small == "inputs" else w * tiny)
    for call, width in (("forward", x_size), ("backward", d_size)):
        v = torch.from_numpy((rng.integers(-2 ** 23, 2 ** 23, (batch, width)) * 2.0 ** -24).astype(np.float32)).cuda()
        want = getattr(normal, call)(v).double()
        got = getattr(low, call)(v * float(tiny) if small == "inputs" else v).double() * 2.0 ** 120
        assert float((got - want).abs().max()) <= 4 * 2.0 ** -30


@pytest.mark.parametrize("terms", [16, 64])
def test_a_range_that_is_nearly_a_multiple_of_the_step(gpu_device, terms):
    """63 steps reach 5e-7 beyond the range: the inputs that meet it are the range, not 63 steps."""
    rng = np.random.default_rng(terms)
    io = noise_free_io(inp_res=float(np.float32((1.0 + 5e-7) / 126)))
    io.out_res, io.out_bound = -1.0, float("inf")
    step = 2.0 * float(np.float32(io.inp_res))
    assert 3e-7 < 63 * step - 1.0 < 1e-6
    w = rng.uniform(-0.6, 0.6, (64, terms)).astype(np.float32)
    x = np.where(rng.random((16384, terms)) < 0.5, -1.0, 1.0).astype(np.float32)
    got = _tile(terms, 64, io, w).forward(torch.from_numpy(x).cuda())[::64].double().cpu().numpy()
    want, chain = x[::64] @ w.T.astype(np.float64), _chain(x[::64], w)
    assert np.sqrt(np.mean((got - want) ** 2)) <= 1.04 * np.sqrt(np.mean((chain - want) ** 2))


@pytest.mark.parametrize("shapes,batch,perfect", [([(12, 160), (300, 256)], 4096, False),    # a tile of few terms among others
                                                  ([(200, 512)] * 4, 4100, True),             # two rounds of square tiles' work
                                                  ([(15, 128), (16, 131), (64, 300)], 8200, False)])
def test_grouped_products_in_three_parts_against_64_bit_sums(gpu_device, shapes, batch, perfect):
    rng = np.random.default_rng(len(shapes))
    steps = 63
    io = noise_free_io(inp_res=-1.0 if perfect else 1.0 / (2 * steps))
    io.out_res, io.out_bound, io.is_perfect = -1.0, float("inf"), perfect
    step = 2.0 * float(np.float32(1.0 / (2 * steps)))
    weights = [rng.uniform(-0.6, 0.6, (d, x)).astype(np.float32) for x, d in shapes]
    group = tiles.TileGroup([_tile(x, d, io, w) for (x, d), w in zip(shapes, weights)])
    inputs = []
    for x, _ in shapes:
        v = (rng.integers(-steps, steps + 1, (batch, x)) * step).astype(np.float32)
        v[:, 0] = 1.0  # meets the range
        inputs.append(v)
    for got, v, w in zip(group.forward([torch.from_numpy(v).cuda() for v in inputs]), inputs, weights):
        q = v.astype(np.float64) if perfect else np.rint(v / step) * step
        w64 = w.astype(np.float64)
        _close(got, q @ w64.T, np.abs(q) @ np.abs(w64).T, 4 * w.shape[1] + 16, w.shape[1])


def _profiled(tile, parts, call, *args):
    """The result of an exact call that has to run on the operands split into parts (k_product), or not to."""
    tile.set_profiling(True)
    out = call(*args)
    assert ("product" in [name for name, _ms in tile.get_profile()]) == parts
    tile.set_profiling(False)
    return out


# exact calls that fill the GPU (k_product): a term, an output and a sample more than a tile holds, one less than that, the terms
# in one and in several shares, a share of one stage, the fewest terms, just above the least work, few samples of large matrices (the
# split of the weights would be most of the call); which of forward, backward and update are such calls
@pytest.mark.parametrize("x_size,d_size,batch,parts", [
    (1025, 900, 1000, "fbu"), (2049, 129, 3300, "fbu"), (127, 2500, 2600, "bu"), (128, 2500, 2600, "fbu"), (129, 2100, 4097, "fbu"),
    (511, 1200, 1400, "fbu"), (512, 1217, 1400, "fbu"), (100, 101, 16384, "u"), (1024, 1024, 769, "fbu"), (640, 257, 5000, "fbu"),
    (2048, 2048, 300, "fbu"), (4096, 4096, 64, ""), (1024, 16384, 128, "bu")])
@pytest.mark.parametrize("trans", [False, True])
def test_exact_products_of_calls_that_fill_the_gpu(gpu_device, x_size, d_size, batch, parts, trans):
    rng = np.random.default_rng(x_size)
    io = noise_free_io()
    io.is_perfect = True
    w = (0.3 * rng.standard_normal((d_size, x_size))).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    lay = (lambda v: torch.from_numpy(np.ascontiguousarray(v.T if trans else v)).cuda())
    back = (lambda v: v.t() if trans else v)
    x, d = rng.standard_normal((batch, x_size)).astype(np.float32), rng.standard_normal((batch, d_size)).astype(np.float32)
    x[:, -1] = 1.0  # the bias column, which is not stored
    x64, d64, w64 = x.astype(np.float64), d.astype(np.float64), w.astype(np.float64)
    y = _profiled(tile, "f" in parts, tile.forward, lay(x[:, :-1]), True, trans, trans)
    _close(back(y), x64 @ w64.T, np.abs(x64) @ np.abs(w64).T, x_size)
    dx = _profiled(tile, "b" in parts, tile.backward, lay(d), True, trans, trans)
    _close(back(dx), (d64 @ w64)[:, :-1], (np.abs(d64) @ np.abs(w64))[:, :-1], d_size)
    lr = 0.125
    tile.set_learning_rate(lr)
    _profiled(tile, "u" in parts, tile.update, lay(x[:, :-1]), lay(d), True, trans, trans)
    want, terms = d64.T @ x64, np.abs(d64).T @ np.abs(x64)
    _close(tile.get_weights(), w64 - lr * want, np.abs(w64) + lr * terms, batch)
    delta = torch.full((x_size, d_size), 7.0, device="cuda")  # overwritten, whatever it holds
    tile.set_delta_weights(delta)
    before = tile.get_weights()
    _profiled(tile, "u" in parts, tile.update, lay(x[:, :-1]), lay(d), True, trans, trans)
    assert torch.equal(tile.get_weights(), before)
    _close(delta.t(), want, terms, batch)


# on either side of the line between the launches on parts and the 32 x 32 kernel, which takes longer for one of the storages
@pytest.mark.parametrize("x_size,d_size,batch", [(1025, 900, 900), (2048, 2048, 130), (2048, 2048, 256), (1024, 4096, 192), (4096, 1024, 224),
                                                 (3072, 3072, 96), (3072, 3072, 256), (4096, 4096, 192), (1024, 16384, 128)])
def test_exact_calls_have_the_same_bits_on_either_storage(gpu_device, x_size, d_size, batch):
    gen = torch.Generator("cuda").manual_seed(1)
    io = noise_free_io()
    io.is_perfect = True
    w = np.random.default_rng(1).standard_normal((d_size, x_size)).astype(np.float32)
    one, other = _tile(x_size, d_size, io, w), _tile(x_size, d_size, io, w)
    if not tiles.CudaAnalogTile.bind_shared_weights:
        bound = torch.empty(x_size, d_size, device="cuda")
        other.set_shared_weights(bound)
    x, d = torch.randn(batch, x_size, generator=gen, device="cuda"), torch.randn(batch, d_size, generator=gen, device="cuda")
    assert torch.equal(one.forward(x), other.forward(x))
    assert torch.equal(one.backward(d), other.backward(d))


def test_exact_products_of_rows_that_are_slices_of_longer_ones(gpu_device):
    """A group that holds a tile on running-average noise management runs its tiles one by one, on the slices that it is given:
    unaligned ones here."""
    rng = np.random.default_rng(7)
    x_size, d_size, batch = 1025, 900, 901
    io = noise_free_io()
    io.is_perfect = True
    average = noise_free_io(noise_management=dv.NoiseManagementType.AverageAbsMax)
    w = rng.standard_normal((d_size, x_size)).astype(np.float32)
    tile, other = _tile(x_size, d_size, io, w), _tile(20, 30, average, w[:30, :20])
    group = tiles.TileGroup([tile, other])
    for own, grouped, width, outputs, small in ((tile.forward, group.forward, x_size, d_size, 20), (tile.backward, group.backward, d_size, x_size, 30)):
        v = torch.randn(batch, width + 6, device="cuda")[:, 3:3 + width]
        out = torch.full((batch, outputs + 10), 7.0, device="cuda")
        rows = [out[:, 5:5 + outputs], torch.empty(batch, 50 - small, device="cuda")]
        _profiled(tile, True, lambda: grouped([v, torch.randn(batch, small, device="cuda")], outs=rows))
        assert torch.equal(rows[0], own(v.contiguous()))
        assert bool((out[:, :5] == 7.0).all()) and bool((out[:, 5 + outputs:] == 7.0).all())


@pytest.mark.parametrize("x_size,d_size,batch", [(1025, 900, 900), (300, 300, 12001)])
def test_exact_products_with_values_out_of_the_range_of_the_parts(gpu_device, x_size, d_size, batch):
    """In the last share of the terms, at the last rows, and none but there: the other tiles are as they are without them."""
    rng = np.random.default_rng(2)
    io = noise_free_io()
    io.is_perfect = True
    w = rng.uniform(-0.5, 0.5, (d_size, x_size)).astype(np.float32)
    x = (rng.random((batch, x_size)) + 0.5).astype(np.float32)
    plain = _tile(x_size, d_size, io, w).forward(torch.from_numpy(x).cuda()).cpu().numpy()
    w[-1, -1], x[-1, -2], x[-2, -1], x[-3, 5] = np.inf, 3e38, np.nan, 1e30
    got = _tile(x_size, d_size, io, w).forward(torch.from_numpy(x).cuda()).cpu().numpy()
    with np.errstate(all="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
        want32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    assert np.array_equal(got[np.isinf(want32)], want32[np.isinf(want32)])
    fine = np.isfinite(want32)
    with np.errstate(all="ignore"):
        bound = (x_size + 2) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T)
        assert np.all((np.abs(got.astype(np.float64) - want) <= bound + 1e-37)[fine])
    assert np.array_equal(got[:-128 - batch % 128, :-128 - d_size % 128], plain[:-128 - batch % 128, :-128 - d_size % 128])


@pytest.mark.parametrize("x_size,d_size,batch", [(1024, 1100, 1024), (700, 3000, 1300), (2049, 2048, 600)])
def test_one_term_that_is_not_zero(gpu_device, x_size, d_size, batch):
    """One product, rounded once: half a unit in its last place.  The seven small products of its parts, together at most 2^-7
    of it, round as often on the way to their sum: 7 * 2^-31 of the product, up to 2^24 units.  Two products left out, of a
    low with a middle part, would be up to half a unit more."""
    rng = np.random.default_rng(x_size)
    io = noise_free_io()
    io.is_perfect = True
    w = rng.standard_normal((d_size, x_size)).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    w64 = w.astype(np.float64)

    def close(got, want):
        unit = np.spacing(np.abs(want).astype(np.float32)).astype(np.float64)
        assert np.max(np.abs(got.cpu().numpy().astype(np.float64) - want) / unit) <= 0.5 + 7.0 * 2.0 ** -7

    def one_a_row(rows, width):
        v = np.zeros((rows, width), np.float32)
        v[np.arange(rows), rng.integers(0, width, rows)] = rng.standard_normal(rows)
        return v

    x, d = one_a_row(batch, x_size), one_a_row(batch, d_size)
    close(tile.forward(torch.from_numpy(x).cuda()), x @ w64.T)
    close(tile.backward(torch.from_numpy(d).cuda()), d @ w64)
    x = np.ascontiguousarray(one_a_row(x_size, batch).T)  # every weight meets one sample
    d = rng.standard_normal((batch, d_size)).astype(np.float32)
    tile.set_weights(torch.zeros(d_size, x_size))
    tile.set_learning_rate(0.5)
    tile.update(torch.from_numpy(x).cuda(), torch.from_numpy(d).cuda(), False)
    close(tile.get_weights(), -0.5 * (d.T.astype(np.float64) @ x))


# 2^86 a product: the parts of one are finite with 2^16 in either operand, the sum of 512 of them is not
@pytest.mark.parametrize("x_size,d_size,batch", [(16384, 100, 100), (4097, 256, 256), (1024, 1024, 1024), (1024, 512, 16384)])
def test_exact_products_of_large_values_have_the_sums_of_fp32(gpu_device, x_size, d_size, batch):
    """No sum is near the end of the range of fp32; each has the error of one in fp32, half a unit a term."""
    io = noise_free_io()
    io.is_perfect = True
    below = (95 - int(np.ceil(np.log2(x_size)))) // 2 - 1  # the largest values that are multiplied in parts
    for e, few in ((43, False), (43, True), (below, False), (below, True)):
        v = np.full((batch, x_size), 1.9 * 2.0 ** e, np.float32)
        w = np.full((d_size, x_size), 1.9 * 2.0 ** e, np.float32)
        if few:  # in the last of the tiles alone, of one sign
            v[:-1], w[:-1] = 1.0, -0.5
        got = _tile(x_size, d_size, io, w).forward(torch.from_numpy(v).cuda()).cpu().numpy().astype(np.float64)
        want = np.outer(v[:, 0].astype(np.float64), w[:, 0].astype(np.float64)) * x_size
        assert np.all(np.abs(got - want) <= (x_size + 2) * 2.0 ** -24 * np.abs(want))


def test_large_tiles_of_large_values_have_the_sums_of_fp32(gpu_device):
    """As above, in the kernel that splits what it stages (exact calls of a group)."""
    x_size, d_size, batch = 512, 512, 8192
    io = noise_free_io()
    io.is_perfect = True
    for e in (43, 42):
        w = np.full((d_size, x_size), 1.9 * 2.0 ** e, np.float32)
        group = tiles.TileGroup([_tile(x_size, d_size, io, w) for _ in range(2)])
        v = torch.full((batch, x_size), float(np.float32(1.9 * 2.0 ** e)), device="cuda")
        want = float(w[0, 0]) ** 2 * x_size
        for got in group.forward([v, v]):
            assert float((got.double() - want).abs().max()) <= (x_size + 2) * 2.0 ** -24 * want


# fewer samples can take other launches (rows padded further, parts), and more shares of the terms
@pytest.mark.parametrize("x_size,d_size,batch", [(768, 2304, 4096), (1024, 1024, 4096), (1000, 1500, 1203), (300, 300, 4096), (2048, 64, 16400)])
def test_exact_calls_make_room_for_those_of_fewer_samples(gpu_device, x_size, d_size, batch):
    """The first step makes room for every smaller one, so that those can be captured after it."""
    from aihwkit_amd._cabi import lib
    rng = np.random.default_rng(x_size)
    io = noise_free_io()
    io.is_perfect = True
    w = rng.standard_normal((d_size, x_size)).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    tile.set_learning_rate(2.0 ** -10)
    x, d = torch.randn(batch, x_size, device="cuda"), torch.randn(batch, d_size, device="cuda")

    def step(n):
        tile.update(x[:n], d[:n], False)
        return tile.forward(x[:n]), tile.backward(d[:n])

    step(batch)
    before = lib().rpu_device_allocation_count()
    for n in range(batch - 31, 0, -(batch // 64 + 1)):
        y, dx = step(n)
        assert lib().rpu_device_allocation_count() == before, n
    w64 = tile.get_weights().double()  # in the room of larger calls
    for got, v, m in ((y, x[:n], w64.t()), (dx, d[:n], w64)):
        want, terms = (v.double().cpu() @ m).numpy(), (v.double().cpu().abs() @ m.abs()).numpy()
        _close(got, want, terms, m.shape[0])


def test_exact_calls_without_memory_for_their_parts(gpu_device):
    """The GPU refuses the scratch: the calls take the launches that need less, and find theirs from then on."""
    from aihwkit_amd._cabi import lib
    x_size, d_size, batch = 768, 1100, 1030
    rng = np.random.default_rng(5)
    io = noise_free_io()
    io.is_perfect = True
    w = (0.3 * rng.standard_normal((d_size, x_size))).astype(np.float32)
    tile = _tile(x_size, d_size, io, w)
    tile.set_exact_scratch_test_hook(1 << 50)  # more than any GPU has
    lr = 0.125
    tile.set_learning_rate(lr)
    x, d = rng.standard_normal((batch, x_size)).astype(np.float32), rng.standard_normal((batch, d_size)).astype(np.float32)
    x64, d64, w64 = x.astype(np.float64), d.astype(np.float64), w.astype(np.float64)
    xg, dg = torch.from_numpy(x).cuda(), torch.from_numpy(d).cuda()
    before = None
    for _ in range(2):
        tile.set_weights(torch.from_numpy(w))
        _close(tile.forward(xg), x64 @ w64.T, np.abs(x64) @ np.abs(w64).T, x_size)
        _close(tile.backward(dg), d64 @ w64, np.abs(d64) @ np.abs(w64), d_size)
        tile.update(xg, dg, False)
        _close(tile.get_weights(), w64 - lr * (d64.T @ x64), np.abs(w64) + lr * (np.abs(d64).T @ np.abs(x64)), batch)
        assert before is None or lib().rpu_device_allocation_count() == before
        before = lib().rpu_device_allocation_count()
