"""Fewer launches for the bound-management rounds of the forward pass (rpu_tile_set_fused_rounds): rounds 0 and 1 in one
launch (mode 1), the rounds after round 0 in one launch (mode 2), both (mode 3), rounds 0 to 2 in one launch (modes 5
and 7).  Outputs and round counts must be bit
for bit those of the separate launches (mode 0), which the other GPU tests hold against the oracle."""
import numpy as np
import pytest
import torch

from aihwkit_amd.rpu_base import devices as dv
from aihwkit_amd.rpu_base import tiles
from helpers import build_pair, config2, config2_data, io_params, make_meta, noise_free_io, soft_bounds

pytestmark = pytest.mark.gpu
F = np.float32
NM, BM = dv.NoiseManagementType, dv.BoundManagementType


def both_ways(meta, dev, x_size, d_size, w, x, seed=5, bias=False, x_trans=False, d_trans=False, calls=3):
    host, _orc, _ = build_pair(meta, dev, x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(w))
    results = []
    xin = torch.from_numpy(np.ascontiguousarray(x.T if x_trans else x)).cuda()
    for mode in (0, 1, 2, 3, 5, 7, -1):              # -1: the tile's own choice, which changes from call to call
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_small_calls(False)                   # those have no launches to share
        gpu.set_fused_rounds(mode)
        gpu.set_seed(seed)
        outs = []
        for _ in range(calls):                       # the second call reuses every buffer of the first
            y = gpu.forward(xin, bias, x_trans, d_trans).cpu().numpy()
            outs.append((y, gpu.get_bm_rounds(x.shape[0]).numpy().copy()))
        results.append(outs)
    for other in results[1:]:
        for (y0, r0), (y1, r1) in zip(results[0], other):
            assert np.array_equal(r0, r1)
            assert np.array_equal(y0, y1)
    return results[0][0]


def test_benchmark_configuration_with_noise_is_bit_equal(gpu_device):
    meta, dev = config2()
    w, x, _d = config2_data(1024, 1024, 256)
    y, rounds = both_ways(meta, dev, 1024, 1024, w, x)
    assert rounds.mean() > 1.9 and np.abs(y).max() > 1.0


@pytest.mark.parametrize("bound_management", [BM.Iterative, BM.IterativeWorstCase])
@pytest.mark.parametrize("shape,bias,trans", [((512, 300, 100), False, False), ((257, 96, 33), True, False),
                                              ((1024, 256, 64), False, True), ((768, 1000, 256), False, False),
                                              ((256, 1024, 1100), False, False)])     # 1120 workgroups: the later rounds walk
def test_shapes_layouts_and_many_rounds(gpu_device, shape, bias, trans, bound_management):
    """Samples that stop after round 0, after round 1 and later (a small out_bound sends many to rounds 2 .. 4), a zero
    sample, a bias column (rows that are not 16-byte aligned), transposed layouts, the worst-case switch of the scale."""
    x_size, d_size, batch = shape
    rng = np.random.default_rng(x_size)
    io = io_params(out_noise=0.1, out_bound=3.0, noise_management=NM.AbsMax, bound_management=bound_management)
    meta = make_meta(io, noise_free_io())
    dev = soft_bounds(construction_seed=3)
    w = rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(F)
    x = rng.uniform(-1, 1, (batch, x_size - (1 if bias else 0))).astype(F)
    x *= rng.choice([0.02, 0.2, 1.0], (batch, 1)).astype(F)       # with abs-max scaling the rounds follow the weights ...
    x[:, : x.shape[1] // 2] *= rng.choice([0.05, 1.0], (batch, 1)).astype(F)   # ... and how the input mass is spread
    x[3] = 0.0
    y, rounds = both_ways(meta, dev, x_size, d_size, w, x, bias=bias, x_trans=trans, d_trans=trans)
    if not bias:                                                  # (the bias column keeps a zero sample alive)
        assert rounds[3] == 0 and not (y.T if trans else y)[3].any()
    if bound_management == BM.Iterative:
        assert len(set(rounds.tolist())) >= 2 and (x_size < 512 or rounds.max() >= 3)
    else:                                                         # the worst-case scale of round 1 always fits
        assert set(rounds.tolist()) <= {0, 1, 2} and (rounds == 2).any()


def test_the_tile_chooses_by_its_last_call(gpu_device):
    """Default mode: the first call runs the separate launches, later ones the fused launch when most samples needed a
    second round, or round 0 and one launch for the rest when none did -- seen here only through equal results and
    through the number of round launches in the profile of a call."""
    meta, dev = config2()
    w, x, _d = config2_data(1024, 1024, 256)
    host, _orc, _ = build_pair(meta, dev, 1024, 1024, gpu=False)
    host.set_weights(torch.from_numpy(w))
    ref = tiles.CudaAnalogTile(host)
    ref.set_fused_rounds(0)
    auto = tiles.CudaAnalogTile(host)
    xin = torch.from_numpy(x).cuda()
    launches = []
    for call in range(4):
        for t in (ref, auto):
            t.set_seed(100 + call)
        auto.set_profiling(True)
        y = auto.forward(xin).cpu().numpy()
        launches.append(sum(1 for name, _ms in auto.get_profile() if name == "mvm_round"))
        auto.set_profiling(False)
        assert np.array_equal(y, ref.forward(xin).cpu().numpy())
    assert launches[0] == 5 and launches[-1] == 2            # rounds 0 to 2 (round 2 listed samples), and one launch for rounds 3 and 4
    quiet = x * np.float32(0.01) + 0                          # nothing saturates ...
    w_small = (w * 0.05).astype(F)
    auto.set_weights(torch.from_numpy(w_small))
    ref.set_weights(torch.from_numpy(w_small))
    quiet_launches = []
    for call in range(11):
        for t in (ref, auto):
            t.set_seed(200 + call)
        auto.set_profiling(True)
        y = auto.forward(torch.from_numpy(quiet).cuda()).cpu().numpy()
        quiet_launches.append(sum(1 for name, _ms in auto.get_profile() if name == "mvm_round"))
        auto.set_profiling(False)
        assert np.array_equal(y, ref.forward(torch.from_numpy(quiet).cuda()).cpu().numpy())
    # ... the estimate of the last busy round falls after eight calls below it: rounds 0, 1, 2 and one launch from round 3 on
    # until then, round 0 and one launch for whatever is left after
    assert quiet_launches[2] == 4 and quiet_launches[-1] == 2
    auto.set_weights(torch.from_numpy(w))                     # saturation again: that launch runs the rounds it finds
    ref.set_weights(torch.from_numpy(w))
    for t in (ref, auto):
        t.set_seed(77)
    y = auto.forward(xin).cpu().numpy()
    assert np.array_equal(y, ref.forward(xin).cpu().numpy())
    assert np.array_equal(auto.get_bm_rounds(256).numpy(), ref.get_bm_rounds(256).numpy())


def test_groups_share_one_launch_for_the_later_rounds_and_recover(gpu_device):
    """A tile group whose last call listed no sample for round 1 runs all later rounds as one launch; when its inputs
    then do saturate, that launch runs the rounds itself (waiting between them).  Exact-arithmetic setting: every call
    must equal the oracle bit for bit, through quiet -> saturating -> quiet sequences, for groups on either side of the
    size at which the later rounds take the walking kernel."""
    from helpers import constant_step
    rng = np.random.default_rng(21)
    for n_tiles, batch, d_size in ((3, 96, 64), (9, 1100, 300)):
        grouped, oracles = [], []
        for k in range(n_tiles):
            x_size = int(rng.choice([64, 96, 130]))
            f_io = noise_free_io(inp_res=1 / 128.0, out_res=1 / 512.0, noise_management=NM.AbsMax,
                                 bound_management=BM.Iterative, out_bound=2.0)
            dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=k + 1)
            host, orc, _ = build_pair(make_meta(f_io, noise_free_io()), dev, x_size, d_size, gpu=False)
            w = (rng.integers(-60, 61, (d_size, x_size)) / 64.0).astype(F)
            host.set_weights(torch.from_numpy(w))
            orc.set_weights(w)
            grouped.append(tiles.CudaAnalogTile(host))
            grouped[-1].set_small_calls(False)
            oracles.append(orc)
        group = tiles.TileGroup(grouped)
        sizes = [t.get_x_size() for t in grouped]
        loud = [(rng.integers(-64, 65, (batch, n)) / 64.0).astype(F) for n in sizes]     # several rounds per sample
        quiet = []
        for n in sizes:                                                                # one input line: nothing saturates
            x = np.zeros((batch, n), F)
            x[np.arange(batch), rng.integers(0, n, batch)] = 0.5
            quiet.append(x)
        seen_rounds = []
        for xs in (quiet, quiet, loud, loud, quiet, quiet, loud):
            got = group.forward([torch.from_numpy(x).cuda() for x in xs])
            for y, orc, x, t in zip(got, oracles, xs, grouped):
                assert np.array_equal(y.cpu().numpy(), orc.forward(x))
                assert np.array_equal(t.get_bm_rounds(batch).numpy(), orc.bm_rounds(batch))
            seen_rounds.append(max(int(t.get_bm_rounds(batch).max()) for t in grouped))
        assert seen_rounds[0] == 1 and seen_rounds[2] >= 3


@pytest.mark.parametrize("batch,out_blocks", [(96, (64, 130, 40)), (1100, (300,) * 6)])
def test_tiles_of_a_split_layer_share_their_quantized_input(gpu_device, batch, out_blocks):
    """A layer split into column and row blocks: the tiles of one input block are handed the same column slice of the
    layer input, and the group quantizes it once for all of them (rounds 0 and 1; the rows of later rounds are each
    tile's own, since the tiles saturate on different samples).  Exact-arithmetic setting against the oracle, through
    quiet and saturating calls; one tile of each input block has a DAC of its own and must not take part."""
    from helpers import constant_step
    rng = np.random.default_rng(batch)
    in_blocks = (96, 104)
    grouped, oracles, where = [], [], []
    i0 = 0
    for bi, n_in in enumerate(in_blocks):
        o0 = 0
        for bo, n_out in enumerate(out_blocks):
            own_dac = bo == len(out_blocks) - 1
            f_io = noise_free_io(inp_res=1 / 64.0 if own_dac else 1 / 128.0, out_res=1 / 512.0, noise_management=NM.AbsMax,
                                 bound_management=BM.Iterative, out_bound=1.0 + bo)
            dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=7 * bi + bo + 1)
            host, orc, _ = build_pair(make_meta(f_io, noise_free_io()), dev, n_in, n_out, gpu=False)
            w = (rng.integers(-60, 61, (n_out, n_in)) / 64.0).astype(F) * F(0.25 if bo % 2 else 1.0)
            host.set_weights(torch.from_numpy(w))
            orc.set_weights(w)
            grouped.append(tiles.CudaAnalogTile(host))
            grouped[-1].set_small_calls(False)       # those quantize the rows for themselves
            oracles.append(orc)
            where.append((bi, i0, n_in, o0, n_out))
            o0 += n_out
        i0 += n_in
    group = tiles.TileGroup(grouped)
    loud = (rng.integers(-64, 65, (batch, sum(in_blocks))) / 64.0).astype(F)
    loud *= rng.choice([1 / 64.0, 0.25, 1.0], (batch, 1)).astype(F)
    loud[5] = 0.0
    quiet = np.zeros_like(loud)
    quiet[np.arange(batch), rng.integers(0, 96, batch)] = 0.5
    quiet[np.arange(batch), 96 + rng.integers(0, 104, batch)] = -0.25
    most = 0
    for x in (loud, quiet, quiet, loud, loud):
        x_layer = torch.from_numpy(x).cuda()
        partial = torch.full((len(in_blocks), batch, sum(out_blocks)), float("nan"), device="cuda")
        xs = [x_layer[:, i:i + n] for _bi, i, n, _o, _m in where]
        ys = [partial[bi][:, o:o + m] for bi, _i, _n, o, m in where]
        group.forward(xs, outs=ys)
        assert group.get_shared_input_sets() == (len(in_blocks), len(in_blocks) * (len(out_blocks) - 1))
        got = partial.cpu().numpy()
        for (bi, i, n, o, m), orc, t in zip(where, oracles, grouped):
            assert np.array_equal(got[bi][:, o:o + m], orc.forward(np.ascontiguousarray(x[:, i:i + n])))
            rounds = t.get_bm_rounds(batch).numpy()
            assert np.array_equal(rounds, orc.bm_rounds(batch))
            most = max(most, int(rounds.max()))
    assert most >= 3                                   # rows of rounds after round 1 were needed, and differ by tile


def test_shared_input_rows_leave_noisy_results_unchanged(gpu_device):
    """The same with the benchmark's analog noise on the outputs: a group call on column slices of one input equals the
    tiles called one by one with the same seeds, bit for bit; tiles whose DAC draws random numbers (input noise,
    stochastic rounding) keep rows of their own."""
    rng = np.random.default_rng(3)
    batch, n_in = 200, 160
    ios = [io_params(out_noise=0.06, out_bound=4.0, noise_management=NM.AbsMax, bound_management=BM.Iterative),
           io_params(out_noise=0.06, out_bound=4.0, noise_management=NM.AbsMax, bound_management=BM.Iterative),
           io_params(out_noise=0.06, out_bound=4.0, inp_noise=0.01, noise_management=NM.AbsMax, bound_management=BM.Iterative),
           io_params(out_noise=0.06, out_bound=4.0, inp_sto_round=True, noise_management=NM.AbsMax,
                     bound_management=BM.Iterative),
           io_params(out_noise=0.06, out_bound=12.0, noise_management=NM.AbsMaxNPSum, bound_management=BM.IterativeWorstCase),
           io_params(out_noise=0.06, out_bound=12.0, noise_management=NM.AbsMaxNPSum, bound_management=BM.IterativeWorstCase)]
    alone, grouped = [], []
    for k, io in enumerate(ios):
        host, _orc, _ = build_pair(make_meta(io, noise_free_io()), soft_bounds(construction_seed=k + 1), n_in, 70 + 10 * k,
                                   gpu=False)
        host.set_weights(torch.from_numpy(rng.uniform(-0.4, 0.4, (70 + 10 * k, n_in)).astype(F)))
        alone.append(tiles.CudaAnalogTile(host))
        grouped.append(tiles.CudaAnalogTile(host))
        for t in (alone[-1], grouped[-1]):
            t.set_small_calls(False)                 # those quantize the rows for themselves
    group = tiles.TileGroup(grouped)
    for call in range(3):
        x = torch.from_numpy((rng.uniform(-1, 1, (batch, n_in)) * rng.choice([0.05, 1.0], (batch, 1))).astype(F)).cuda()
        for k, (a, g) in enumerate(zip(alone, grouped)):
            a.set_seed(50 * call + k)
            g.set_seed(50 * call + k)
        got = group.forward([x] * len(grouped))
        assert group.get_shared_input_sets() == (2, 4)
        for a, g, y in zip(alone, grouped, got):
            assert np.array_equal(y.cpu().numpy(), a.forward(x).cpu().numpy())
            assert np.array_equal(g.get_bm_rounds(batch).numpy(), a.get_bm_rounds(batch).numpy())


def test_more_than_sixteen_rounds_in_one_launch(gpu_device):
    """No input quantization and a large max_bm_factor: samples whose outputs exceed a tiny out_bound by five orders of
    magnitude halve their input seventeen to twenty times.  The single launch for the later rounds walks all of them
    (its arrival words are per round) and must agree with the separate launches."""
    rng = np.random.default_rng(17)
    x_size, d_size, batch = 96, 64, 40
    io = io_params(inp_res=-1.0, out_res=-1.0, out_noise=0.0, out_bound=2e-5, max_bm_factor=1 << 22,
                   noise_management=NM.AbsMax, bound_management=BM.Iterative)
    meta = make_meta(io, noise_free_io())
    dev = soft_bounds(construction_seed=9)
    w = rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(F)
    x = rng.uniform(-1, 1, (batch, x_size)).astype(F)
    x[::3] *= F(1 / 64.0)                                        # abs-max scaling: the spread of a row decides, ...
    x[::3, 0] = 1.0                                              # ... so these rows are one large and many small inputs
    y, rounds = both_ways(meta, dev, x_size, d_size, w, x)
    assert rounds.max() >= 18 and len(set(rounds.tolist())) >= 3
    assert np.abs(y).max() > 0.0


def test_a_wait_that_runs_out_is_reported_and_the_tile_recovers(gpu_device):
    """The launch that runs several rounds makes its workgroups wait for each other.  The test hook shortens that wait and
    makes it expect one arrival too many, so that it runs out while every workgroup still leaves its kernel: the next
    call on the tile must fail with the time-out message, and the calls after it (one launch per round again) must give
    the results of the separate launches."""
    meta, dev = config2()
    for io in (meta.forward_io, meta.backward_io):
        io.out_noise = 0.0
    w, x, _d = config2_data(1024, 1024, 256)
    host, _orc, _ = build_pair(meta, dev, 1024, 1024, gpu=False)
    host.set_weights(torch.from_numpy(w))
    ref, tile = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    ref.set_fused_rounds(0)
    xin = torch.from_numpy(x).cuda()
    want = ref.forward(xin).cpu().numpy()
    assert ref.get_bm_rounds(256).max() >= 3                     # rounds beyond the first merged one have work
    tile.set_fused_rounds(2)
    assert np.array_equal(tile.forward(xin).cpu().numpy(), want)  # the merged launch, waits intact
    tile.set_round_wait_test_hook(2000, 1)
    tile.forward(xin)                                             # stops after its first round
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="forward round barrier timed out in round 1; results of call"):
        tile.forward(xin)
    tile.set_round_wait_test_hook(0, 0)
    tile.set_profiling(True)
    assert np.array_equal(tile.forward(xin).cpu().numpy(), want)  # recovered: separate launches although mode 2 stands
    assert sum(1 for name, _ms in tile.get_profile() if name == "mvm_round") == 5
    tile.set_profiling(False)
    assert np.array_equal(tile.get_bm_rounds(256).numpy(), ref.get_bm_rounds(256).numpy())
    tile.set_fused_rounds(2)                                      # an explicit choice arms the merged launch again
    tile.set_profiling(True)
    assert np.array_equal(tile.forward(xin).cpu().numpy(), want)
    assert sum(1 for name, _ms in tile.get_profile() if name == "mvm_round") == 2
    tile.set_profiling(False)


def test_a_group_reports_a_wait_that_runs_out(gpu_device):
    """The same for the launch that runs the later rounds of a whole group."""
    from helpers import constant_step
    rng = np.random.default_rng(5)
    batch, d_size = 96, 64
    grouped, oracles = [], []
    for k in range(3):
        x_size = (64, 96, 130)[k]
        f_io = noise_free_io(inp_res=1 / 128.0, out_res=1 / 512.0, noise_management=NM.AbsMax,
                             bound_management=BM.Iterative, out_bound=2.0)
        dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=k + 1)
        host, orc, _ = build_pair(make_meta(f_io, noise_free_io()), dev, x_size, d_size, gpu=False)
        w = (rng.integers(-60, 61, (d_size, x_size)) / 64.0).astype(F)
        host.set_weights(torch.from_numpy(w))
        orc.set_weights(w)
        grouped.append(tiles.CudaAnalogTile(host))
        grouped[-1].set_small_calls(False)                        # these run no rounds in launches of their own
        oracles.append(orc)
    group = tiles.TileGroup(grouped)
    sizes = [t.get_x_size() for t in grouped]
    loud = [(rng.integers(-64, 65, (batch, n)) / 64.0).astype(F) for n in sizes]
    quiet = []
    for n in sizes:
        x = np.zeros((batch, n), F)
        x[np.arange(batch), rng.integers(0, n, batch)] = 0.5
        quiet.append(x)

    def run(xs):
        return [y.cpu().numpy() for y in group.forward([torch.from_numpy(x).cuda() for x in xs])]

    run(quiet)                                                    # nothing listed: the next call merges its later rounds
    group.set_round_wait_test_hook(2000, 1)
    run(loud)                                                     # the merged launch runs round 1 and gives up after it
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="forward round barrier timed out"):
        run(loud)
    group.set_round_wait_test_hook(0, 0)
    for xs in (loud, quiet, quiet, loud):                         # one launch per round from now on: exact again
        for y, orc, x in zip(run(xs), oracles, xs):
            assert np.array_equal(y, orc.forward(x))


def test_calls_in_one_launch_leave_what_the_others_know(gpu_device):
    """Forward calls of a group that list samples for round 1, with backward calls between them that run as one launch
    (k_mvm_few) and list nothing: the next forward call must still expect work in round 1 and not choose the launch for
    rounds that are expected empty.  That launch would run into the shortened wait, and the call after it fail."""
    from helpers import constant_step
    rng = np.random.default_rng(6)
    batch, sizes = 120, ((64, 64), (130, 96))
    grouped, oracles = [], []
    for k, (x_size, d_size) in enumerate(sizes):
        f_io = noise_free_io(inp_res=1 / 128.0, out_res=1 / 512.0, noise_management=NM.AbsMax,
                             bound_management=BM.Iterative, out_bound=2.0)
        dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=k + 1)
        host, orc, _ = build_pair(make_meta(f_io, noise_free_io()), dev, x_size, d_size, gpu=False)
        w = (rng.integers(-60, 61, (d_size, x_size)) / 64.0).astype(F)
        host.set_weights(torch.from_numpy(w))
        orc.set_weights(w)
        grouped.append(tiles.CudaAnalogTile(host))
        oracles.append(orc)
    group = tiles.TileGroup(grouped)
    xs = [(rng.integers(-64, 65, (batch, n)) / 64.0).astype(F) for n, _ in sizes]
    ds = [torch.from_numpy((rng.integers(-64, 65, (batch, n)) / 64.0).astype(F)).cuda() for _, n in sizes]
    for _ in range(2):
        for t in grouped:
            t.set_small_calls(False)
        group.set_round_wait_test_hook(2000, 1)
        got = group.forward([torch.from_numpy(x).cuda() for x in xs])
        for y, orc, x in zip(got, oracles, xs):
            assert np.array_equal(y.cpu().numpy(), orc.forward(x)) and orc.bm_rounds(batch).max() >= 2
        for t in grouped:
            t.set_small_calls(True)
        group.set_round_wait_test_hook(0, 0)                      # (the hook keeps to the launches that wait)
        group.backward(ds)


def test_worst_case_second_round_on_a_fresh_tile_matches_the_oracle(gpu_device):
    """IterativeWorstCase: round 1 runs at the AbsMaxNPSum scale.  The init kernel quantizes the rows of that round ahead
    and must use the scale its threads have just computed, not one read back from the per-sample state that the group's
    first thread is still storing (on a fresh tile that state holds anything).  Exact-arithmetic setting, first call of
    fresh tiles in every launch mode against the oracle, at a batch that takes the walking kernel for the later rounds."""
    from helpers import constant_step
    rng = np.random.default_rng(31)
    x_size, d_size, batch = 512, 256, 1100
    f_io = noise_free_io(inp_res=1 / 128.0, out_res=1 / 512.0, out_bound=2.0, noise_management=NM.AbsMax,
                         bound_management=BM.IterativeWorstCase)
    dev = constant_step(w_max_dtod=0.0, w_min_dtod=0.0, w_max=1.0, w_min=-1.0, construction_seed=2)
    host, orc, _ = build_pair(make_meta(f_io, noise_free_io()), dev, x_size, d_size, gpu=False)
    w = (rng.integers(-60, 61, (d_size, x_size)) / 64.0).astype(F)
    host.set_weights(torch.from_numpy(w))
    orc.set_weights(w)
    x = rng.uniform(-1, 1, (batch, x_size)).astype(F)
    x *= rng.choice([0.02, 0.2, 1.0], (batch, 1)).astype(F)
    want, rounds = orc.forward(x), orc.bm_rounds(batch)
    assert (rounds >= 2).mean() > 0.3
    xin = torch.from_numpy(x).cuda()
    for mode in (0, 1, 3, 5, 7, -1):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_fused_rounds(mode)
        y = gpu.forward(xin).cpu().numpy()
        assert np.array_equal(gpu.get_bm_rounds(batch).numpy(), rounds), mode
        assert np.array_equal(y, want), mode


@pytest.mark.parametrize("shape", [(160, 1100, 1030), (64, 80, 9000), (100, 700, 500)])
def test_large_calls_share_one_launch_for_the_later_rounds(gpu_device, shape):
    """Calls whose rounds run on the large tiles (rows quantized ahead, and written by the last workgroup of a sample tile),
    or have more workgroups than the GPU holds: quiet inputs, then saturating ones that the one launch does not expect,
    then quiet ones again.  All sums are exact, so every kernel gives the same bits."""
    x_size, d_size, batch = shape
    rng = np.random.default_rng(d_size)
    io = noise_free_io(inp_res=1 / 64.0, out_res=1 / 256.0, out_bound=2.0, noise_management=NM.NONE, bound_management=BM.Iterative)
    w = (rng.integers(-32, 33, (d_size, x_size)) / 64.0).astype(F)
    host, _orc, _ = build_pair(make_meta(io, noise_free_io()), soft_bounds(construction_seed=3, w_max_dtod=0.0, w_min_dtod=0.0),
                               x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(w))
    loud = (rng.integers(-64, 65, (batch, x_size)) / 64.0).astype(F)
    quiet = (rng.integers(-1, 2, (batch, x_size)) / 64.0).astype(F)
    results = []
    for mode in (0, 2, -1):
        gpu = tiles.CudaAnalogTile(host)
        gpu.set_fused_rounds(mode)
        outs = []
        for x in [quiet] * 3 + [loud] * 2 + [quiet] * 2:
            gpu.set_profiling(True)
            y = gpu.forward(torch.from_numpy(x).cuda()).cpu().numpy()
            launches = sum(1 for name, _ms in gpu.get_profile() if name == "mvm_round")
            assert mode < 0 or (launches == 2) == (mode == 2)     # round 0, and all the others
            gpu.set_profiling(False)
            outs.append((y, gpu.get_bm_rounds(batch).numpy().copy()))
        results.append(outs)
    assert results[0][0][1].max() == 1 and results[0][3][1].max() >= 3
    for other in results[1:]:
        for (y0, r0), (y1, r1) in zip(results[0], other):
            assert np.array_equal(r0, r1)
            assert np.array_equal(y0, y1)


def _quiet_and_loud(rng, x_size, d_size, batch):
    io = noise_free_io(inp_res=1 / 64.0, out_res=1 / 256.0, out_bound=2.0, noise_management=NM.NONE, bound_management=BM.Iterative)
    w = (rng.integers(-32, 33, (d_size, x_size)) / 64.0).astype(F)
    host, _orc, _ = build_pair(make_meta(io, noise_free_io()), soft_bounds(construction_seed=3, w_max_dtod=0.0, w_min_dtod=0.0),
                               x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(w))
    loud = torch.from_numpy((rng.integers(-64, 65, (batch, x_size)) / 64.0).astype(F)).cuda()
    quiet = torch.from_numpy((rng.integers(-1, 2, (batch, x_size)) / 64.0).astype(F)).cuda()
    return host, quiet, loud


@pytest.mark.parametrize("shape", [(160, 1100, 1030), (64, 80, 9000), (100, 700, 500)])
def test_large_calls_go_on_without_the_workgroups_that_stop_waiting(gpu_device, shape):
    """The launch that walks the rounds of a large call loses every workgroup that has waited for its limit, here one poll:
    those that are left, at the end the one that finished a round, run the rounds to the same bits, and no call fails."""
    host, quiet, loud = _quiet_and_loud(np.random.default_rng(shape[1]), *shape)
    ref, tile = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    ref.set_fused_rounds(0)
    tile.set_fused_rounds(2)
    tile.set_round_wait_test_hook(1, 0)
    for x in (quiet, loud, loud, quiet, loud):
        tile.set_profiling(True)
        y = tile.forward(x)
        assert sum(1 for name, _ms in tile.get_profile() if name == "mvm_round") == 2    # round 0, and all the others
        tile.set_profiling(False)
        assert torch.equal(y, ref.forward(x))
        assert torch.equal(tile.get_bm_rounds(shape[2]), ref.get_bm_rounds(shape[2]))
    assert ref.get_bm_rounds(shape[2]).max() >= 3


@pytest.mark.parametrize("spins", [0, 1])
def test_more_than_sixteen_rounds_walked_by_one_launch(gpu_device, spins):
    """As test_more_than_sixteen_rounds_in_one_launch, with more 32 x 32 tiles than the GPU has CUs."""
    rng = np.random.default_rng(17)
    x_size, d_size, batch = 96, 64, 4200
    io = io_params(inp_res=-1.0, out_res=-1.0, out_noise=0.0, out_bound=2e-5, max_bm_factor=1 << 22,
                   noise_management=NM.AbsMax, bound_management=BM.Iterative)
    host, _orc, _ = build_pair(make_meta(io, noise_free_io()), soft_bounds(construction_seed=9), x_size, d_size, gpu=False)
    host.set_weights(torch.from_numpy(rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(F)))
    x = rng.uniform(-1, 1, (batch, x_size)).astype(F)
    x[::3] *= F(1 / 64.0)
    x[::3, 0] = 1.0
    xin = torch.from_numpy(x).cuda()
    ref, tile = tiles.CudaAnalogTile(host), tiles.CudaAnalogTile(host)
    ref.set_fused_rounds(0)
    tile.set_fused_rounds(2)
    tile.set_round_wait_test_hook(spins, 0)
    for _ in range(2):
        assert torch.equal(tile.forward(xin), ref.forward(xin))
        rounds = tile.get_bm_rounds(batch)
        assert torch.equal(rounds, ref.get_bm_rounds(batch)) and rounds.max() >= 18
