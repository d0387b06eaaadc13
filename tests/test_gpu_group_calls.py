"""Groups whose calls take the one launch of small batches upload their argument blocks only when these have changed: whatever
changes between calls, every tile gets what its own call gives, bit for bit."""
import copy
import time

import numpy as np
import pytest
import torch

from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles
from helpers import build_pair, constant_step, io_params, make_meta

pytestmark = pytest.mark.gpu


def twins(rng, shapes):
    io = dict(inp_res=1 / 126.0, out_res=1 / 510.0, out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax)
    meta = make_meta(io_params(bound_management=dv.BoundManagementType.Iterative, out_bound=3.0, **io), io_params(**io))
    grouped, alone = [], []
    for k, (x_size, d_size) in enumerate(shapes):
        host, _orc, _ = build_pair(meta, constant_step(construction_seed=k + 1), x_size, d_size, gpu=False)
        host.set_weights(torch.from_numpy(rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(np.float32)))
        grouped.append(tiles.CudaAnalogTile(host))
        alone.append(copy.deepcopy(grouped[-1]))
        for t in (grouped[-1], alone[-1]):
            t.set_seed(50 + k)
    return tiles.TileGroup(grouped), grouped, alone


# more tiles than the launch's own arguments hold; and few
@pytest.mark.parametrize("shapes", [[(130, 70), (300, 40), (64, 200)], [(40, 16)] * 64, [(40, 16)] * 65])
def test_calls_of_a_group_follow_what_changes(gpu_device, shapes):
    rng = np.random.default_rng(len(shapes))
    group, grouped, alone = twins(rng, shapes)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    for step, batch in enumerate((3, 3, 3, 5, 3, 3, 3, 3)):
        if step == 4:                                        # other weights
            for t, u in zip(grouped, alone):
                w = torch.from_numpy(rng.uniform(-0.3, 0.3, (t.get_d_size(), t.get_x_size())).astype(np.float32))
                t.set_weights(w)
                u.set_weights(w)
        if step == 5:                                        # other draws
            for k, (t, u) in enumerate(zip(grouped, alone)):
                t.set_seed(900 + k)
                u.set_seed(900 + k)
        xs = [torch.from_numpy(rng.uniform(-1, 1, (batch, x)).astype(np.float32)).cuda() for x, _ in shapes]
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[step == 6]):          # another stream
            got = group.forward(xs)
        torch.cuda.synchronize()
        for t, u, x, y in zip(grouped, alone, xs, got):
            assert torch.equal(y, u.forward(x, False)), step
            assert torch.equal(t.get_bm_rounds(batch), u.get_bm_rounds(batch))
        if step % 3 == 2:                                    # the other direction has blocks of its own
            ds = [torch.from_numpy(rng.normal(0, 1, (batch, d)).astype(np.float32)).cuda() for _, d in shapes]
            for u, d, g in zip(alone, ds, group.backward(ds)):
                assert torch.equal(g, u.backward(d, False))


def test_directions_in_turn_upload_nothing(gpu_device):
    """Forward and backward calls in turn, as a training step makes them, take what each takes when it is repeated: neither displaces the
    argument blocks of the other (one set of blocks for both: 46 us against 33)."""
    rng = np.random.default_rng(4)
    group, _grouped, _alone = twins(rng, [(128, 128)] * 38)
    xs = [torch.from_numpy(rng.uniform(-1, 1, (4, 128)).astype(np.float32)).cuda() for _ in range(38)]
    ys = [torch.empty(4, 128, device="cuda") for _ in range(38)]
    gs = [torch.empty(4, 128, device="cuda") for _ in range(38)]

    def forward():
        group.forward(xs, non_blocking=True, outs=ys)

    def backward():
        group.backward(xs, non_blocking=True, outs=gs)

    def microseconds(*calls):
        best = float("inf")
        for _ in range(5):
            torch.cuda.synchronize()
            start = time.perf_counter()
            for _ in range(100):
                for call in calls:
                    call()
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - start) * 1e4)
        return best

    apart = microseconds(forward) + microseconds(backward)
    in_turn = microseconds(forward, backward)
    assert in_turn < 1.25 * apart, (in_turn, apart)
