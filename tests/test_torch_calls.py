"""The native calls on torch tensors (csrc/torch_calls.cpp) leave tensors without a storage of their own -- inside a
function transform or a tracer -- to the general path, which raises; they used to end the process.  Each case runs in a
process of its own, all calls on tensors that claim to be on a GPU."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import struct, sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from aihwkit_amd._cabi import torch_calls
from helpers import constant_step, make_meta

transform = sys.argv[1]
m, sizes = torch_calls(), struct.pack("=ii", 8, 4)
tile = make_meta().create_array(8, 4, constant_step())
tile.set_learning_rate(0.01)
h = tile._h.value

CALLS = {
    "forward": lambda x, d: m.forward(h, x, 8, 4, False, False, False, False, True),
    "backward": lambda x, d: m.backward(h, d, 4, 8, False, False, False, False, True),
    "update": lambda x, d: m.update(h, x, d, 8, 4, False, False, False, False, True),
    "group_forward": lambda x, d: m.group_forward(0, sizes, [x], None, False, True),
    "group_backward": lambda x, d: m.group_backward(0, sizes, [d], None, False, True),
    "group_update": lambda x, d: m.group_update(0, sizes, [x], [d], True),
}

def f(x, d):
    for name, call in CALLS.items():
        print(name, flush=True)
        assert call(x, d) is None
    return x + 1

with FakeTensorMode():
    x, d = (torch.empty(3, 2, n, device="cuda") for n in (8, 4))
    assert x.is_cuda
    if transform == "vmap":
        torch.vmap(f)(x, d)
    elif transform == "vjp":
        torch.func.vjp(f, x[0], d[0])
    elif transform == "jvp":
        torch.func.jvp(f, (x[0], d[0]), (x[1], d[1]))
    else:
        f(x[0], d[0])
print("done")
"""


@pytest.mark.parametrize("transform", ["vmap", "vjp", "jvp", "none"])
def test_tensors_without_storage_are_left_to_the_general_path(transform):
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    run = subprocess.run([sys.executable, "-c", SCRIPT, transform], env=env, capture_output=True, text=True, timeout=240)
    assert run.returncode == 0 and run.stdout.strip().endswith("done"), run.stdout + run.stderr[-1500:]


def _tile(x_size, d_size):
    import torch

    from aihwkit_amd.rpu_base import tiles
    from helpers import constant_step, make_meta, noise_free_io
    host = make_meta(noise_free_io(), noise_free_io()).create_array(x_size, d_size, constant_step(construction_seed=1))
    host.set_weights(torch.full((d_size, x_size), 0.25))
    tile = tiles.CudaAnalogTile(host)
    tile.set_learning_rate(0.01)
    return tile


@pytest.mark.gpu
def test_calls_inside_a_function_transform_raise():
    import torch

    from aihwkit_amd.rpu_base.tiles import TileGroup
    tile = _tile(8, 4)
    group = TileGroup([tile])
    x, d = torch.ones(3, 2, 8, device="cuda"), torch.ones(3, 2, 4, device="cuda")
    for call in (lambda x, d: tile.forward(x), lambda x, d: tile.backward(d), lambda x, d: tile.update(x, d, False),
                 lambda x, d: group.forward([x])[0], lambda x, d: group.backward([d])[0], lambda x, d: group.update([x], [d])):
        with pytest.raises(RuntimeError):
            torch.vmap(call)(x, d)
    assert tile.forward(x[0]).shape == (2, 4)


@pytest.mark.gpu
def test_outputs_that_share_their_memory_until_written():
    """A lazily cloned output tensor gets its copy before a group writes to it: the tensor it was cloned from stays."""
    import torch

    from aihwkit_amd.rpu_base.tiles import TileGroup
    group = TileGroup([_tile(8, 4)])
    x, d = torch.ones(2, 8, device="cuda"), torch.ones(2, 4, device="cuda")
    for call, inputs, size in ((group.forward, [x], 4), (group.backward, [d], 8)):
        first = torch.full((2, size), 7.0, device="cuda")
        out = torch._lazy_clone(first)
        call(inputs, outs=[out])
        assert bool((first == 7.0).all()) and bool((out != 7.0).all())


@pytest.fixture
def without_native_calls(monkeypatch, tmp_path):
    """No module at the place where it is looked for."""
    from aihwkit_amd import _cabi
    _cabi.lib()
    monkeypatch.setattr(_cabi, "_torch_calls", None)
    monkeypatch.setattr(_cabi, "_HERE", str(tmp_path))
    with pytest.warns(RuntimeWarning, match="make -C"):
        _cabi.torch_calls()


def test_tiles_take_the_general_path_without_the_native_calls(without_native_calls):
    import torch

    from helpers import constant_step, make_meta
    from aihwkit_amd.rpu_base.tiles import CudaAnalogTile
    tile = make_meta().create_array(8, 4, constant_step())  # on the host: the GPU tile's methods get as far as the tensors
    tile._update_without_allocation = False
    x, d = torch.ones(3, 8), torch.ones(3, 4)
    for call in (lambda: CudaAnalogTile.forward(tile, x), lambda: CudaAnalogTile.backward(tile, d),
                 lambda: CudaAnalogTile.update(tile, x, d, False)):
        with pytest.raises(RuntimeError, match="x_input|d_input"):  # the words of that path for tensors on the CPU
            call()


@pytest.mark.gpu
def test_results_without_the_native_calls(without_native_calls, monkeypatch):
    import torch

    from aihwkit_amd import _cabi
    from aihwkit_amd.rpu_base.tiles import TileGroup

    def results():
        tile, other = _tile(40, 24), _tile(40, 24)
        group = TileGroup([other])
        g = torch.Generator("cuda").manual_seed(3)
        x, d = (torch.rand(7, n, generator=g, device="cuda") - 0.5 for n in (40, 24))
        tile.update(x, d, False)
        group.update([x], [d])
        return [tile.forward(x), tile.backward(d), tile.get_weights()] + group.forward([x]) + group.backward([d])

    general = results()
    monkeypatch.undo()
    assert not isinstance(_cabi.torch_calls(), _cabi._GeneralPath)
    for a, b in zip(general, results()):
        assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))
