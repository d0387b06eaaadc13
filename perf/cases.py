"""Work that programs on this library spend their time in, as cases that can be timed and compared.

A case is a dict of plain values; ``kind`` says which program it is, the rest are its sizes and options.  Every pass
is one step of that program through the public classes of ``aihwkit_amd`` with its operands resident in HBM, and
returns what the step produces (outputs, input gradients, and the weights it leaves behind).

kinds
  ``infer``     forward of one inference tile, the plain (blocking) call: what a single layer costs when asked alone
  ``train``     training step of one analog layer: noisy forward, noisy backward, pulsed update
  ``hwa``       hardware-aware training step of a layer: weight modifier, noisy forward, exact backward and update
  ``layers``    forward of linear layers split into tiles of at most 512 x 512 (PCM tiles after a day of drift)
  ``transfer``  two mini-batches of an MLP of Tiki-Taka transfer tiles, one column transferred on the way
  ``lenet``     forward of a LeNet5-shaped stack of PCM tiles (two convolutions, two linear layers)
  ``conv``      training step of one convolution layer through the indexed interface

Random draws are keyed by the tile's seed and a call counter, so a state made from the same seed repeats its results.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from aihwkit_amd.benchmark_configs import config2, config3, config5_io, conv_index_matrix, io_params, make_meta
from aihwkit_amd.benchmark_configs import constant_step, soft_bounds
from aihwkit_amd.inference import InferenceTile
from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles

DAY = 86400.0
GPT2_SMALL = "768x2304,768x768,768x3072,3072x768"   # the linear layers of one block, in x out


def listed():
    return [
        # one vector through one mapped tile (512 is the reference's default tile limit): latency of a single call
        dict(name="infer_one", kind="infer", x=512, d=512, batch=1),
        # last layer of a 784-256-128-10 MLP with its bias column: a training step that is launches and host path only
        dict(name="train_small", kind="train", x=129, d=10, batch=64, device="soft_bounds", storage="xd",
             bl_management=True, bias=True),
        # benchmark configuration 1
        dict(name="train_512", kind="train", x=512, d=512, batch=100, device="constant_step", storage="row_major",
             bl_management=True, bias=False),
        # benchmark configuration 2 on a tile bound to its [x, d] tensor, as the reference's Python holds CUDA tiles
        dict(name="train_1024", kind="train", x=1024, d=1024, batch=256, device="soft_bounds", storage="xd",
             bl_management=True, bias=False),
        # ragged sizes, bias column, and bit lines of the full 31 pulses (update BL management switched off)
        dict(name="train_ragged", kind="train", x=785, d=300, batch=37, device="soft_bounds", storage="row_major",
             bl_management=False, bias=True),
        # a token-scale batch on the tile of configuration 2
        dict(name="train_tokens", kind="train", x=1024, d=1024, batch=16384, device="soft_bounds", storage="row_major",
             bl_management=True, bias=False),
        # benchmark configuration 5: all linear layers of a transformer block, a prompt of 1024 tokens ...
        dict(name="layers_prefill", kind="layers", shapes=GPT2_SMALL, tokens=1024),
        # ... and the same layers while a few sequences generate token by token
        dict(name="layers_decode", kind="layers", shapes=GPT2_SMALL, tokens=8),
        # benchmark configuration 3
        dict(name="transfer_mlp", kind="transfer", sizes="784,256,128,10", batch=64),
        # benchmark configuration 4
        dict(name="lenet", kind="lenet", batch=512),
        # a wide 3 x 3 convolution, 131072 patches (bench.py's configuration 6)
        dict(name="conv_train", kind="conv", c_in=48, c_out=48, side=34, kernel=3, images=128),
        # hardware-aware training of a transformer projection as one tile
        dict(name="hwa_train", kind="hwa", x=768, d=2304, batch=1024),
    ]


def _log_int(rng, low, high):
    """An integer of [low, high], uniform in its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choices(("train", "hwa", "infer", "layers", "transfer", "lenet", "conv"), (6, 2, 2, 2, 1, 1, 2))[0]
    if kind == "train":
        x, d = _log_int(rng, 16, 1024), _log_int(rng, 10, 1024)
        # at most a fifth of the largest listed step: bit lines of 31 pulses cost more per sample than short ones
        batch = _log_int(rng, 1, max(1, min(4096, (1 << 32) // (x * d))))
        return dict(kind=kind, x=x, d=d, batch=batch, device=rng.choice(("soft_bounds", "constant_step", "linear_step")),
                    storage=rng.choice(("xd", "row_major")), bl_management=rng.random() < 0.75, bias=rng.random() < 0.5)
    if kind == "hwa":
        return dict(kind=kind, x=_log_int(rng, 64, 3072), d=_log_int(rng, 64, 3072), batch=_log_int(rng, 8, 2048))
    if kind == "infer":
        return dict(kind=kind, x=_log_int(rng, 16, 1024), d=_log_int(rng, 10, 1024), batch=_log_int(rng, 1, 4096))
    if kind == "layers":
        shapes = ",".join("%dx%d" % (_log_int(rng, 256, 3072), _log_int(rng, 256, 3072)) for _ in range(rng.randint(1, 3)))
        return dict(kind=kind, shapes=shapes, tokens=_log_int(rng, 1, 2048))
    if kind == "transfer":
        hidden = [_log_int(rng, 32, 512) for _ in range(rng.randint(1, 2))]
        return dict(kind=kind, sizes=",".join(str(s) for s in [784] + hidden + [10]), batch=_log_int(rng, 4, 256))
    if kind == "lenet":
        return dict(kind=kind, batch=_log_int(rng, 1, 1024))
    return dict(kind=kind, c_in=_log_int(rng, 3, 64), c_out=_log_int(rng, 8, 64), side=rng.randint(10, 36), kernel=3,
                images=_log_int(rng, 1, 128))


# -- preparation -------------------------------------------------------------------------------------------------------

class _Rand:
    """Seeded draws on the GPU (inputs) and on the host (weights)."""

    def __init__(self, seed):
        self.gpu = torch.Generator("cuda").manual_seed(seed)
        self.host = np.random.default_rng(seed)

    def uniform(self, shape, low, high):
        return torch.rand(shape, generator=self.gpu, device="cuda") * (high - low) + low

    def normal(self, shape, std):
        return torch.randn(shape, generator=self.gpu, device="cuda") * std

    def weights(self, d, x, w_max):
        return torch.from_numpy(self.host.uniform(-w_max, w_max, (d, x)).astype(np.float32))


def _training_io(bound_management):
    kw = dict(out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax)
    if bound_management:
        kw["bound_management"] = dv.BoundManagementType.Iterative
    return io_params(**kw)


def _training_tile(case, rand, seed):
    """Analog layer with the IO of configurations 1 and 2 (7-bit DAC, 9-bit ADC, output noise, abs-max noise management,
    iterative bound management in the forward pass), its weight tensor and a copy of the weights it starts from."""
    meta = make_meta(_training_io(True), _training_io(False), desired_bl=31, update_management=True,
                     update_bl_management=case["bl_management"])
    if case["device"] == "constant_step":
        dev = constant_step(dw_min_dtod=0.0, dw_min_std=0.0, up_down_dtod=0.0, w_max_dtod=0.0, w_min_dtod=0.0)
    elif case["device"] == "soft_bounds":
        dev = soft_bounds()
    else:
        dev = dv.LinearStepResistiveDeviceParameter()
        dev.gamma_up = dev.gamma_down = 0.1
    dev.construction_seed = 123
    dev.enforce_consistency = True
    host = meta.create_array(case["x"], case["d"], dev)
    host.set_weights(rand.weights(case["d"], case["x"], 0.6))
    return _bound(tiles.CudaAnalogTile(host), case["storage"], seed)


def _bound(tile, storage, seed):
    tile.set_learning_rate(0.01)
    tile.set_seed(seed + 1)
    x_size, d_size = tile.get_x_size(), tile.get_d_size()
    if storage == "xd":
        live = torch.empty(x_size, d_size, device="cuda")
        tile.set_shared_weights(live)
    else:
        live = torch.empty(d_size, x_size, device="cuda")
        tile.set_shared_weights_row_major(live)
    torch.cuda.synchronize()
    return tile, live, live.clone()


def _pcm_tile(d, x, io, weights, seed):
    tile = InferenceTile(d, x, forward_io=io)
    tile.set_weights(weights)
    tile.cuda()
    tile.tile.set_seed(seed)
    tile.drift_weights(DAY)
    return tile


def _split(size, limit=512):
    """Sizes of the tiles that a dimension is split into (the reference's tile array: near-equal parts)."""
    n = -(-size // limit)
    return [size // n + (1 if k < size % n else 0) for k in range(n)]


def _shapes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]


def prepare(case, seed):
    rand = _Rand(seed)
    return dict(case=case, **globals()["_prepare_" + case["kind"]](case, rand, seed))


def _prepare_infer(case, rand, seed):
    tile = _pcm_tile(case["d"], case["x"], config5_io(), rand.weights(case["d"], case["x"], 0.3), seed + 1)
    return dict(tile=tile, x=rand.normal((case["batch"], case["x"]), 1.0))


def _prepare_train(case, rand, seed):
    tile, live, start = _training_tile(case, rand, seed)
    return dict(tile=tile, live=live, start=start,
                x=rand.uniform((case["batch"], case["x"] - int(case["bias"])), -1.0, 1.0),
                g=rand.normal((case["batch"], case["d"]), 0.05))


def _prepare_hwa(case, rand, seed):
    meta = make_meta(_training_io(True), io_params(is_perfect=True), pulse_type=dv.PulseType.NONE)
    host = meta.create_array(case["x"], case["d"], dv.IdealResistiveDeviceParameter())
    host.set_weights(rand.weights(case["d"], case["x"], 0.1))
    tile, live, start = _bound(tiles.CudaAnalogTile(host), "xd", seed)
    modifier = tiles.WeightModifierParameter()
    modifier.type = tiles.WeightModifierType.AddNormal
    modifier.std_dev = 0.1
    return dict(tile=tile, live=live, start=start, modifier=modifier, x=rand.normal((case["batch"], case["x"]), 1.0),
                g=rand.normal((case["batch"], case["d"]), 0.01))


def _prepare_layers(case, rand, seed):
    layers, count = [], 0
    for in_size, out_size in _shapes(case):
        x = rand.normal((case["tokens"], in_size), 1.0)
        in_parts, out_parts = _split(in_size), _split(out_size)
        partial = torch.empty(len(in_parts), case["tokens"], out_size, device="cuda")
        members, inputs, outputs, i0 = [], [], [], 0
        for i, n_in in enumerate(in_parts):
            o0 = 0
            for n_out in out_parts:
                weights = torch.from_numpy((0.02 * rand.host.standard_normal((n_out, n_in))).astype(np.float32))
                tile = _pcm_tile(n_out, n_in, config5_io(), weights, seed + 1 + count)
                tile.compensate_in_tile(True)
                members.append(tile)
                inputs.append(x[:, i0:i0 + n_in])
                outputs.append(partial[i][:, o0:o0 + n_out])
                o0, count = o0 + n_out, count + 1
            i0 += n_in
        layers.append((tiles.TileGroup([t.tile for t in members]), members, inputs, outputs, partial))
    return dict(layers=layers)


def _prepare_transfer(case, rand, seed):
    sizes = [int(s) for s in case["sizes"].split(",")]
    layers = []
    for k, (n_in, n_out) in enumerate(zip(sizes[:-1], sizes[1:])):
        meta, device = config3()
        host = meta.create_array(n_in + 1, n_out, device)
        host.set_weights(rand.weights(n_out, n_in + 1, 0.3))
        tile = tiles.CudaAnalogTile(host)
        tile.set_learning_rate(0.1)
        tile.set_seed(seed + 1 + k)
        layers.append((tile, [(rand.uniform((case["batch"], n_in), 0.0, 1.0), rand.normal((case["batch"], n_out), 0.1))
                              for _ in range(2)]))
    return dict(layers=layers)


def _prepare_lenet(case, rand, seed):
    io = io_params(inp_res=1 / 254.0, out_res=1 / 254.0, out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax,
                   bound_management=dv.BoundManagementType.Iterative)
    stack = []
    for k, (in_shape, out_size) in enumerate((((1, 28, 28), 16), ((16, 12, 12), 32), (512, 128), (128, 10))):
        conv = isinstance(in_shape, tuple)
        in_size = (in_shape[0] * 25 if conv else in_shape) + 1
        weights = rand.weights(out_size, in_size, 1.0 / math.sqrt(in_size))
        tile = _pcm_tile(out_size, in_size, io, weights, seed + 1 + k)
        tile.compensate_in_tile(True)
        if conv:
            tile.set_matrix_indices(conv_index_matrix(in_shape, (5, 5))[0])
        stack.append((conv, tile, out_size))
    return dict(stack=stack, x=rand.uniform((case["batch"], 1, 28, 28), 0.0, 1.0))


def _prepare_conv(case, rand, seed):
    c_in, c_out, side, k, n = (case[name] for name in ("c_in", "c_out", "side", "kernel", "images"))
    meta, dev = config2()
    x_size, out_side = c_in * k * k + 1, side - k + 1
    host = meta.create_array(x_size, c_out, dev)
    host.set_weights(rand.weights(c_out, x_size, 0.1))
    tile, live, start = _bound(tiles.CudaAnalogTile(host), "xd", seed)
    tile.set_matrix_indices(conv_index_matrix((c_in, side, side), (k, k))[0])
    return dict(tile=tile, live=live, start=start, x=rand.uniform((n, c_in, side, side), 0.0, 1.0),
                g=rand.normal((n, c_out, out_side, out_side), 0.01))


# -- one pass ----------------------------------------------------------------------------------------------------------
# The steps that update a tile begin by putting its first weights back (a device copy, as bench.py's step does):
# repeated updates on one batch would otherwise carry the weights away from the distribution stated here, and with them
# the number of bound-management rounds that the forward pass needs.

def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_infer(state):
    return state["tile"].forward(state["x"], is_test=True)


def _run_train(state):
    tile, bias = state["tile"], state["case"]["bias"]
    state["live"].copy_(state["start"], non_blocking=True)
    y = tile.forward(state["x"], bias, False, False, False, True)
    dx = tile.backward(state["g"], bias, False, False, True)
    tile.update(state["x"], state["g"], bias, False, False, True)
    return y, dx, state["live"]


def _run_hwa(state):
    tile = state["tile"]
    state["live"].copy_(state["start"], non_blocking=True)
    tile.modify_weights(state["modifier"])
    y = tile.forward(state["x"], False, False, False, False, True)
    dx = tile.backward(state["g"], False, False, False, True)
    tile.update(state["x"], state["g"], False, False, False, True)
    return y, dx, state["live"]


def _run_layers(state):
    outs = []
    for group, _, inputs, outputs, partial in state["layers"]:
        group.forward(inputs, is_test=True, non_blocking=True, outs=outputs)
        outs.append(partial.sum(dim=0) if partial.shape[0] > 1 else partial[0])
    return outs


def _run_transfer(state):
    # the loop update -> forward -> backward, so that the outputs show the weights that the updates left
    outs = []
    for k in range(2):
        for tile, batches in state["layers"]:
            tile.update(batches[k][0], batches[k][1], True, False, False, True)
        for tile, batches in state["layers"]:
            outs.append(tile.forward(batches[1 - k][0], True, False, False, False, True))
        for tile, batches in reversed(state["layers"]):
            outs.append(tile.backward(batches[1 - k][1], True, False, False, True))
    return outs


def _run_lenet(state):
    h = state["x"]
    for conv, tile, out_size in state["stack"]:
        if conv:
            side = h.size(3) - 4
            y = tile.forward_indexed(h, torch.empty(h.size(0), out_size, side, side, device="cuda"), is_test=True)
            h = F.max_pool2d(torch.tanh(y), 2)
        else:
            h = tile.forward(h.reshape(h.size(0), -1), is_test=True, bias=True)
            if out_size != 10:
                h = torch.tanh(h)
    return h


def _run_conv(state):
    tile, x, g = state["tile"], state["x"], state["g"]
    state["live"].copy_(state["start"], non_blocking=True)
    y = tile.forward_indexed(x, torch.empty_like(g), False, True)
    dx = tile.backward_indexed(g, torch.empty_like(x), True)
    tile.update_indexed(x, g, True)
    return y, dx, state["live"]


# -- what a pass cannot do without -------------------------------------------------------------------------------------
# One contraction round per pass (re-runs by bound management are not counted).  A pulsed update counts as the rank-B
# product that it stands for; its device steps (one per coinciding pulse) come on top.

def _device_bytes(device):
    """Bytes of a cross-point in an update: weight read and written, parameter arrays read."""
    return 8 + 4 * (4 if device == "constant_step" else 6)


def work(case):
    kind = case["kind"]
    if kind == "infer":
        x, d, b = case["x"], case["d"], case["batch"]
        return dict(bytes=4 * (x * d + b * (x + d)), flops=2 * x * d * b)
    if kind in ("train", "hwa"):
        x, d, b = case["x"], case["d"], case["batch"]
        per_device = _device_bytes(case["device"]) if kind == "train" else 8
        return dict(bytes=per_device * x * d + 4 * b * 2 * (x + d), flops=6 * x * d * b)
    if kind == "layers":
        b = case["tokens"]
        return dict(bytes=sum(4 * (x * d + b * (x + d)) for x, d in _shapes(case)),
                    flops=sum(2 * x * d * b for x, d in _shapes(case)))
    if kind == "transfer":
        sizes, b = [int(s) for s in case["sizes"].split(",")], case["batch"]
        pairs = [(x + 1, d) for x, d in zip(sizes[:-1], sizes[1:])]
        # two mini-batches: the fast device is updated twice, the slow one is read twice
        return dict(bytes=sum(2 * ((_device_bytes("soft_bounds") + 4) * x * d + 4 * b * 2 * (x + d)) for x, d in pairs),
                    flops=sum(12 * x * d * b for x, d in pairs))
    if kind == "lenet":
        b = case["batch"]
        macs = 576 * 26 * 16 + 64 * 401 * 32 + 513 * 128 + 129 * 10
        return dict(bytes=4 * (b * (784 + 10) + 26 * 16 + 401 * 32 + 513 * 128 + 129 * 10), flops=2 * b * macs)
    x, d, n = case["c_in"] * case["kernel"] ** 2 + 1, case["c_out"], case["images"]
    patches = n * (case["side"] - case["kernel"] + 1) ** 2
    return dict(bytes=_device_bytes("soft_bounds") * x * d + 4 * 2 * (n * case["c_in"] * case["side"] ** 2 + patches * d),
                flops=6 * x * d * patches)


def tolerance(case):
    """Weights and exact passes agree to the rounding of 32-bit sums.  Outputs of a noisy pass are multiples of an ADC
    step: another order of summation moves a few in 10^5 of them over a rounding edge, by one whole step.  A step is a
    hundredth of a wide tile's output (root mean square) and up to most of it behind few lines or small weights."""
    if case["kind"] == "lenet":     # a moved step of a convolution output reaches the image's logits through two layers
        return {"rel": 1e-2, "max": 0.9}
    return {"rel": 3e-3 if case["kind"] in ("layers", "infer") else 2e-3, "max": 0.9}
