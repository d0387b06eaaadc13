#!/usr/bin/env python3
"""Benchmark of the analog-tile hot path on one MI355X.

A step is one forward + one backward + one pulsed update of a single analog tile over one batch of
synthetic inputs that are resident in HBM (benchmark configuration 2: 1024 x 1024 SoftBounds tile with
device-to-device and cycle-to-cycle variation, batch 256, BL 31, update management and update-BL
management on, 7-bit DAC / 9-bit ADC, out_noise 0.06, abs-max noise management, iterative bound
management in the forward pass).

Prints ONE JSON line: `value` is the pulsed-update rate in Gdevice-updates/s (x_size * d_size * batch
per update call / time of the update call); the noisy forward / backward rates (GFLOP/s counted as
2 * x * d * batch per call, bound-management re-runs not counted) are in `forward` / `backward`.
`roofline` covers the dominant kernel of the step (the per-cross-point update kernel) against HBM
bandwidth, `roofline_forward` the MFMA contraction kernel against the fp32 matrix peak, `cpu_baseline`
the CPU oracle timed on this host.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, "oracle")):  # oracle/: only the cpu_baseline legs import from it
    if _p not in sys.path:
        sys.path.insert(0, _p)

HBM_PEAK_GBS = 8000.0      # MI355X HBM3E
FP32_MFMA_PEAK_TFLOPS = 157.3  # MI355X dense fp32 matrix
SPLIT_MFMA_PEAK_TFLOPS = 2500.0 / 3  # dense bf16 matrix, three products per element (large-tile contraction)

# Counter values at configuration 2 from rocprofv3 runs of `bench.py --pmc` (one run per counter group; the summaries,
# with the commands, are under profiles/).  They are constants of this file, not measured in a benchmark run, and
# the JSON line says so ("traffic_source").
# FETCH_SIZE / WRITE_SIZE are KiB per dispatch; a device copy of 64 MiB in the same runs reads FETCH_SIZE = 32782 and
# WRITE_SIZE = 65536, so FETCH_SIZE is scaled by 2.0 and WRITE_SIZE by 1.0.
PMC_TRAFFIC_BYTES = {
    "k_update_pulsed_masks": (16615 * 2.0 + 4096 * 1.0) * 1024,
    "k_mvm_round": (6851 * 2.0 + 2115 * 1.0) * 1024,  # a round over all 256 samples
    # the launches of a forward call whose rounds 0 to 2 share one launch: k_mvm_dual<0, 3>, then k_mvm_rounds_rest
    "forward_fused_3": ((14557 + 586) * 2.0 + (3157 + 1024) * 1.0) * 1024,
}
PMC_SOURCE = {"k_update_pulsed_masks": "profiles/k_update_pulsed_masks_config2.txt", "k_mvm_round": "profiles/k_mvm_round_config2.txt",
              "forward_fused_3": "profiles/k_mvm_dual_config2.txt"}


def batch_sweep() -> int:
    """Call time against the batch on the configuration-2 tile: shows where a second workgroup per CU starts to cost
    its full time."""
    import numpy as np
    import torch

    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.benchmark_configs import config2

    meta, dev = config2()
    host = meta.create_array(1024, 1024, dev)
    host.set_weights(torch.from_numpy(np.random.default_rng(0).uniform(-0.6, 0.6, (1024, 1024)).astype(np.float32)))
    tile = tiles.CudaAnalogTile(host)
    out = {"workload": "config2 tile, forward / backward call time against the batch", "unit": "us", "calls": 200,
           "batches": {}}
    for batch in (32, 64, 128, 256, 512, 1024, 2000):
        x = torch.rand(batch, 1024, device="cuda") * 2 - 1
        d = torch.randn(batch, 1024, device="cuda") * 0.1
        entry = {}
        for name, fn, arg in (("forward", tile.forward, x), ("backward", tile.backward, d)):
            for _ in range(10):
                fn(arg, non_blocking=True)
            torch.cuda.synchronize()
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(200):
                fn(arg, non_blocking=True)
            stop.record()
            torch.cuda.synchronize()
            entry[name] = round(start.elapsed_time(stop) / 200 * 1000, 1)
        out["batches"][str(batch)] = entry
    print(json.dumps(out))
    return 0


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--no-cpu-baseline", action="store_true", help="skip the CPU oracle timing")
    ap.add_argument("--no-other-batches", action="store_true",
                    help="skip the supplementary runs of the same tile at batch 16384 (contraction) and 8 (update)")
    ap.add_argument("--pmc", action="store_true",
                    help="counter-collection mode for rocprofv3 --pmc: one 64 MiB calibration copy, then 3 update, "
                         "3 forward, 3 backward calls and 3 update calls of the aggregated variant; no timing, "
                         "no JSON line")
    ap.add_argument("--batch-sweep", action="store_true",
                    help="instead of the benchmark line: forward and backward call times of the configuration-2 tile "
                         "at batches 32 .. 2000 (HIP events over 200 calls each), one JSON line")
    ap.add_argument("--storage", default="row_major", choices=("row_major", "xd_shared"),
                    help="xd_shared: every GPU tile is bound to an [x_size, d_size] shared weight tensor, as the reference's "
                         "Python binds its CUDA tiles (the library then works on that layout in place); configuration 2 "
                         "reports that mode as a second block in any case")
    ap.add_argument("--config", type=int, default=2, choices=(1, 2, 3, 4, 5, 6),
                    help="benchmark configuration: 2 is the graded one; 3 is the Tiki-Taka MLP of transfer tiles; "
                         "5 is the forward pass of the GPT-2-small linear layers as PCM inference tiles; 6 "
                         "(supplementary) is one wide convolution layer through the indexed interface")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs on one GPU; an analog tile is an independent unit and the path "
              "uses no collective, so --gpus must be 1.", file=sys.stderr)
        return 2

    import numpy as np
    import torch

    from aihwkit_amd._cabi import lib
    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.benchmark_configs import config1, config1_data, config2, config2_data

    lib()  # fails loudly if the HIP library is not built
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        return 1
    torch.cuda.set_device(0)

    if args.storage == "xd_shared":
        tiles.CudaAnalogTile.bind_shared_weights = True
    if args.batch_sweep:
        return batch_sweep()
    if args.config == 3:
        return bench_config3(args)
    if args.config == 4:
        return bench_config4(args)
    if args.config == 5:
        return bench_config5(args)
    if args.config == 6:
        return bench_config6(args)

    if args.config == 2:
        x_size, d_size, batch = 1024, 1024, 256
        meta, dev = config2()
        w, x, d = config2_data(x_size, d_size, batch)
        workload = "config2: 1024x1024 SoftBounds (dtod + ctoc), batch 256, BL 31, UM+UBLM, 7/9-bit IO, iterative BM"
        bytes_per_device = 32.0  # w read + w write + 6 parameter arrays
    else:
        x_size, d_size, batch = 512, 512, 100
        meta, dev = config1()
        w, x, d = config1_data(x_size, d_size, batch)
        workload = "config1: 512x512 ConstantStep (no variation), batch 100, BL 31, UM+UBLM"
        bytes_per_device = 24.0
    lr = 0.01
    host = meta.create_array(x_size, d_size, dev)
    host.set_weights(torch.from_numpy(w))
    tile = tiles.CudaAnalogTile(host)
    tile.set_learning_rate(lr)
    tile.set_seed(1234)
    xg = torch.from_numpy(x).cuda()
    dg = torch.from_numpy(d).cuda()

    if args.pmc:
        src = torch.ones(16 * 1024 * 1024, dtype=torch.float32, device="cuda")  # 64 MiB read + 64 MiB written
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        torch.cuda.synchronize()
        # forward first, on the stated weights (updates change them, and with them the rounds a forward call needs)
        for _ in range(3):
            tile.forward(xg, False, False, False, False, False)
        for _ in range(3):
            tile.backward(dg, False, False, False, False)
        for _ in range(3):
            tile.update(xg, dg, False, False, False, False)
        if args.config == 2:
            tile_v = tiles.CudaAnalogTile(host)
            tile_v.set_learning_rate(lr)
            tile_v.set_seed(1234)
            tile_v.set_update_variant("aggregated", 32)
            for _ in range(3):
                tile_v.update(xg, dg, False, False, False, False)
            del tile_v
        if args.config == 2 and not args.no_other_batches:
            rng = np.random.default_rng(3)
            xb = torch.from_numpy(rng.uniform(-1, 1, (16384, x_size)).astype(np.float32)).cuda()
            db = torch.from_numpy(rng.normal(0, 0.05, (16384, d_size)).astype(np.float32)).cuda()
            for _ in range(2):
                tile.forward(xb, False, False, False, False, False)
            for _ in range(2):
                tile.backward(db, False, False, False, False)
        print("pmc run done: 1 copy of 64 MiB, 3 forward, 3 backward, 3 update calls, 3 update calls of the aggregated "
              "variant, then (unless --no-other-batches) 2 forward and 2 backward calls at batch 16384", file=sys.stderr)
        return 0

    # The contract loop works on the configuration as stated: repeated updates with the same inputs let the weights of
    # a SoftBounds tile shrink until no sample saturates the ADC any more (1.0 bound-management rounds instead of the
    # stated 2.1), so every step starts from the initial weights (a 4 MB device copy into the tile's weight matrix, on
    # the same stream and inside the timed region) and takes the next of POOL pre-uploaded (x, d) batches.
    POOL = 8
    rng_pool = np.random.default_rng(77)
    x_pool = [xg] + [torch.from_numpy(rng_pool.uniform(-1, 1, x.shape).astype(np.float32)).cuda() for _ in range(POOL - 1)]
    d_pool = [dg] + [torch.from_numpy((d.std() * rng_pool.standard_normal(d.shape)).astype(np.float32)).cuda()
                     for _ in range(POOL - 1)]
    if args.storage == "xd_shared":
        w_live = tile._shared_weights           # the [x_size, d_size] tensor the tile was bound to when it was made
    else:
        w_live = torch.empty(d_size, x_size, dtype=torch.float32, device="cuda")
        tile.set_shared_weights_row_major(w_live)   # the tile's weight matrix is this tensor from now on (zero copy)
    torch.cuda.synchronize()
    w_init = w_live.clone()                     # the initial weights as the tile holds them (clipped to the device bounds)
    step_no = [0]

    def step():
        k = step_no[0] % POOL
        step_no[0] += 1
        w_live.copy_(w_init, non_blocking=True)
        tile.forward(x_pool[k], False, False, False, False, True)
        tile.backward(d_pool[k], False, False, False, True)
        tile.update(x_pool[k], d_pool[k], False, False, False, True)

    def time_calls(fn, n):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        for _ in range(max(3, n)):   # as many untimed calls as timed ones: the clocks of an idle GPU take a while to rise
            fn()
        torch.cuda.synchronize()
        start.record()
        for _ in range(n):
            fn()
        end.record()
        torch.cuda.synchronize()
        return start.elapsed_time(end) / n

    def kernel_ms(fn, n_calls, of=None):
        # Per-kernel durations from HIP events that the library records on the launch stream around each
        # kernel.  The first bracket of a call is empty ("_bracket"): the time between two consecutive event
        # records with nothing in between, taken out of every kernel's bracket.
        acc = {}
        for _ in range(n_calls):
            fn()
            for name, ms in (of or tile).get_profile():
                acc.setdefault(name, []).append(ms)
        bracket = float(np.mean(acc.pop("_bracket")))
        out = {k: (float(np.sum(v)) / n_calls - bracket * (len(v) // n_calls), len(v) // n_calls) for k, v in acc.items()}
        out["_bracket"] = (bracket, 1)
        return out

    def contraction(prof):
        # (ms, launches) of a call's contraction: its round launches, or the one launch that runs a small or medium batch
        return prof[next(k for k in ("mvm_few", "mvm_whole", "mvm_round") if k in prof)]

    def one_launch(prof):
        return next(("k_%s (whole call)" % k for k in ("mvm_few", "mvm_whole") if k in prof), None)

    def pulse_loop(prof):
        # (kernel, ms) of the pulse loop of an update call: its plain form, the one on lane masks, the pipelined one
        name = next(k for k in prof if k.startswith("update_pulsed"))
        return "k_" + name, prof[name][0]

    def backward_kernel(prof):
        return one_launch(prof) or "k_mvm_round"

    n = max(args.steps, 10)
    # forward / backward alone, on the initial weights (they do not change the tile)
    ms_forward = time_calls(lambda: tile.forward(xg, False, False, False, False, True), n)
    ms_backward = time_calls(lambda: tile.backward(dg, False, False, False, True), n)
    tile.set_profiling(True)
    prof_forward = kernel_ms(lambda: tile.forward(xg, False, False, False, False, True), n)
    rounds = tile.get_bm_rounds(batch).numpy()  # of the last forward call, before backward reuses the state
    prof_backward = kernel_ms(lambda: tile.backward(dg, False, False, False, True), n)
    tile.set_profiling(False)

    # the contract loop: W warm-up steps, then exactly K timed steps
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    # bound-management rounds the forward calls of that loop ran: the next step's forward call, read back
    w_live.copy_(w_init)
    tile.forward(x_pool[step_no[0] % POOL], False, False, False, False, True)
    loop_rounds = float(tile.get_bm_rounds(batch).numpy().mean())
    w_live.copy_(w_init)

    # update alone
    ms_update = time_calls(lambda: tile.update(xg, dg, False, False, False, True), n)
    tile.set_profiling(True)
    prof_update = kernel_ms(lambda: tile.update(xg, dg, False, False, False, True), n)
    tile.set_profiling(False)

    # The same tile bound to an [x_size, d_size] shared weight tensor, which is how the reference's Python holds every
    # CUDA tile: the library works on that layout in place (forward addresses the weights as backward does on the
    # row-major tile and the other way round, the update walks the cross-points with x and d exchanged).
    xd_block = None
    if args.storage != "xd_shared":
        w_xd = torch.empty(x_size, d_size, dtype=torch.float32, device="cuda")
        tile_x = tiles.CudaAnalogTile(host)
        tile_x.set_learning_rate(lr)
        tile_x.set_seed(1234)
        tile_x.set_shared_weights(w_xd)
        torch.cuda.synchronize()
        w_xd_init = w_xd.clone()
        msx_f = time_calls(lambda: tile_x.forward(xg, False, False, False, False, True), n)
        msx_b = time_calls(lambda: tile_x.backward(dg, False, False, False, True), n)
        tile_x.set_profiling(True)
        px_f = kernel_ms(lambda: tile_x.forward(xg, False, False, False, False, True), n, tile_x)
        rounds_x = float(tile_x.get_bm_rounds(batch).numpy().mean())
        px_b = kernel_ms(lambda: tile_x.backward(dg, False, False, False, True), n, tile_x)
        tile_x.set_profiling(False)
        sx = [0]

        def step_x():
            k = sx[0] % POOL
            sx[0] += 1
            w_xd.copy_(w_xd_init, non_blocking=True)
            tile_x.forward(x_pool[k], False, False, False, False, True)
            tile_x.backward(d_pool[k], False, False, False, True)
            tile_x.update(x_pool[k], d_pool[k], False, False, False, True)

        for _ in range(args.warmup):
            step_x()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            step_x()
        torch.cuda.synchronize()
        msx_step = (time.perf_counter() - t0) * 1e3 / args.steps
        w_xd.copy_(w_xd_init)
        msx_u = time_calls(lambda: tile_x.update(xg, dg, False, False, False, True), n)
        tile_x.set_profiling(True)
        px_u = kernel_ms(lambda: tile_x.update(xg, dg, False, False, False, True), n, tile_x)
        tile_x.set_profiling(False)
        ubytes = bytes_per_device * x_size * d_size + 4.0 * (x_size + d_size) * batch
        fl = 2.0 * x_size * d_size * batch
        xd_block = {
            "storage": "xd_shared",
            "what": "the same workload on a tile bound to an [x_size, d_size] shared weight tensor (zero copy)",
            "value": float(x_size) * d_size * batch / (msx_u * 1e-3) / 1e9, "unit": "Gdevice-updates/s",
            "ms_per_step": msx_step,
            "update": {"ms_per_call": msx_u, "kernels_ms": {k: v[0] for k, v in px_u.items()}},
            "forward": {"ms_per_call": msx_f, "gflops": fl / (msx_f * 1e-3) / 1e9, "mean_bm_rounds": rounds_x,
                        "kernels_ms": {k: v[0] for k, v in px_f.items()}, "round_launches": contraction(px_f)[1]},
            "backward": {"ms_per_call": msx_b, "gflops": fl / (msx_b * 1e-3) / 1e9,
                         "kernels_ms": {k: v[0] for k, v in px_b.items()}},
            "roofline": {"kernel": pulse_loop(px_u)[0], "bound": "hbm", "achieved": ubytes / (pulse_loop(px_u)[1] * 1e-3) / 1e9,
                         "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": ubytes / (pulse_loop(px_u)[1] * 1e-3) / 1e9 / HBM_PEAK_GBS,
                         "traffic": None, "algorithmic_bytes": ubytes, "kernel_ms": pulse_loop(px_u)[1]},
            "roofline_forward": {"kernel": "all round launches of a call", "bound": "mfma",
                                 "achieved": fl / (contraction(px_f)[0] * 1e-3) / 1e12, "peak": FP32_MFMA_PEAK_TFLOPS,
                                 "unit": "TFLOP/s", "frac": fl / (contraction(px_f)[0] * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                                 "kernel_ms": contraction(px_f)[0]},
            "roofline_backward": {"kernel": backward_kernel(px_b), "bound": "mfma",
                                  "achieved": fl / (contraction(px_b)[0] * 1e-3) / 1e12, "peak": FP32_MFMA_PEAK_TFLOPS,
                                  "unit": "TFLOP/s", "frac": fl / (contraction(px_b)[0] * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                                  "kernel_ms": contraction(px_b)[0]},
        }
        del tile_x

    # coincidences (device pulses) of one update call, from the packed words of the last call: the pulses of sample b
    # in slot k are (x lines that fired) x (d lines that fired)
    xw, dw, _ = tile.get_update_words(batch)
    xb_, db_ = xw.numpy().view(np.uint32) >> 1, dw.numpy().view(np.uint32) >> 1
    pulses = float(sum((((xb_ >> k) & 1).sum(1, dtype=np.float64) * ((db_ >> k) & 1).sum(1, dtype=np.float64)).sum() for k in range(31)))

    # opt-in variant of the update, by name (never the headline value): groups of 32 or 64 samples in closed form
    variants = None
    if args.config == 2:
        variants = {}
        ub = bytes_per_device * x_size * d_size + 4.0 * (x_size + d_size) * batch
        for group in (32, 64):
            tile_v = tiles.CudaAnalogTile(host)
            tile_v.set_learning_rate(lr)
            tile_v.set_seed(1234)
            tile_v.set_update_variant("aggregated", group)
            ms_v = time_calls(lambda: tile_v.update(xg, dg, False, False, False, True), n)
            tile_v.set_profiling(True)
            prof_v = kernel_ms(lambda: tile_v.update(xg, dg, False, False, False, True), n, tile_v)
            tile_v.set_profiling(False)
            kv = prof_v["update_aggregated"][0]
            variants["aggregated_%d" % group] = {
                "what": "NOT the reference's per-pulse arithmetic: coincidences counted per %d samples and applied in "
                        "closed form with one moment-matched noise draw (rpu_tile_set_update_variant); passes the "
                        "unchanged 64-seed test of the weight change at this configuration" % group,
                "ms_per_call": ms_v, "gdevice_updates_per_s": float(x_size) * d_size * batch / (ms_v * 1e-3) / 1e9,
                "kernel": "k_update_aggregated", "kernel_ms": kv, "hbm_gbs": ub / (kv * 1e-3) / 1e9,
                "frac_of_hbm_peak": ub / (kv * 1e-3) / 1e9 / HBM_PEAK_GBS}
            del tile_v

    # The same tile at other batch sizes (supplementary; the main figures are at the configuration's batch): the
    # contraction at a token-scale batch, where the matrix pipe and not launch latency sets the time, on a second
    # tile with the initial weights like the forward / backward figures above, and the update at a batch of 8, where
    # few pulses per cross-point leave it to the memory system.  They come after the graded measurements: in the
    # first GPU process of a freshly started machine the update call measured 8 % slower (0.099 against 0.090 ms)
    # whenever this part had run before it (cause unknown; later processes on the same machine were not affected).
    other = None
    if args.config == 2 and not args.no_other_batches:
        tile_b = tiles.CudaAnalogTile(host)
        tile_b.set_seed(1234)
        rng = np.random.default_rng(3)
        big = 16384
        xb = torch.from_numpy(rng.uniform(-1, 1, (big, x_size)).astype(np.float32)).cuda()
        db = torch.from_numpy(rng.normal(0, 0.05, (big, d_size)).astype(np.float32)).cuda()
        tile_b.set_profiling(True)
        prof_fb = kernel_ms(lambda: tile_b.forward(xb, False, False, False, False, True), 5, tile_b)
        rounds_b = float(tile_b.get_bm_rounds(big).numpy().mean())
        prof_bb = kernel_ms(lambda: tile_b.backward(db, False, False, False, True), 5, tile_b)
        tile_b.set_profiling(False)
        fl = 2.0 * x_size * d_size * big
        other = {
            "forward_batch_16384": {"kernel": "k_mvm_big<0, 128, 4, 1, false> (all rounds of a call)", "kernel_ms": prof_fb["mvm_round"][0],
                                    "mean_bm_rounds": rounds_b,
                                    "useful_tflops": fl / (prof_fb["mvm_round"][0] * 1e-3) / 1e12,
                                    "frac_of_mfma_peak_useful": fl / (prof_fb["mvm_round"][0] * 1e-3) / 1e12 / SPLIT_MFMA_PEAK_TFLOPS,
                                    "frac_of_mfma_peak_executed": rounds_b * fl / (prof_fb["mvm_round"][0] * 1e-3) / 1e12
                                    / SPLIT_MFMA_PEAK_TFLOPS},
            "backward_batch_16384": {"kernel": "k_mvm_big<1, 128, 4, 1, false>", "kernel_ms": prof_bb["mvm_round"][0],
                                     "tflops": fl / (prof_bb["mvm_round"][0] * 1e-3) / 1e12,
                                     "frac_of_mfma_peak": fl / (prof_bb["mvm_round"][0] * 1e-3) / 1e12 / SPLIT_MFMA_PEAK_TFLOPS},
        }
        del xb, db, tile_b

    if other is not None:
        tile.set_profiling(True)
        prof_u8 = kernel_ms(lambda: tile.update(xg[:8].contiguous(), dg[:8].contiguous(), False, False, False, True), 10)
        tile.set_profiling(False)
        bytes8 = bytes_per_device * x_size * d_size + 4.0 * (x_size + d_size) * 8
        other["update_batch_8"] = {"kernel": pulse_loop(prof_u8)[0], "kernel_ms": pulse_loop(prof_u8)[1],
                                   "gbs": bytes8 / (pulse_loop(prof_u8)[1] * 1e-3) / 1e9,
                                   "frac_of_hbm_peak": bytes8 / (pulse_loop(prof_u8)[1] * 1e-3) / 1e9 / HBM_PEAK_GBS,
                                   "note": "algorithmic bytes over kernel time; the calls repeat on the same 32 MB of "
                                           "arrays, part of which the memory-side cache still holds from the call "
                                           "before, so this can exceed what HBM alone delivers"}

    devices_per_call = float(x_size) * d_size * batch
    flops_per_call = 2.0 * x_size * d_size * batch
    update_bytes = bytes_per_device * x_size * d_size + 4.0 * (x_size + d_size) * batch
    k_update, k_update_ms = pulse_loop(prof_update)
    k_fwd_ms = contraction(prof_forward)[0]   # all round launches of one forward call
    fused_forward = contraction(prof_forward)[1] < 5 and args.config == 2  # rounds 0 and 1 ran as one launch
    fused_3 = fused_forward and contraction(prof_forward)[1] == 2           # rounds 0 to 2, then one launch for the rest
    fwd_traffic = "forward_fused_3" if fused_3 else ("k_mvm_round" if args.config == 2 and not fused_forward else None)
    k_bwd_ms = contraction(prof_backward)[0]

    out = {
        "metric": "pulsed-update Gdevice-updates/s + noisy fwd GFLOP/s, 1024^2 tile, 1 MI355X",
        "value": devices_per_call / (ms_update * 1e-3) / 1e9,
        "unit": "Gdevice-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": workload, "x_size": x_size, "d_size": d_size, "batch": batch, "lr": lr,
                   "step": "initial weights restored (4 MB device copy, timed) + forward + backward + update on the next "
                           "of %d pre-uploaded input batches" % POOL,
                   "mean_bm_rounds_in_step_loop": loop_rounds},
        "update": {"ms_per_call": ms_update, "kernels_ms": {k: v[0] for k, v in prof_update.items()},
                   "pulses_per_call": pulses, "pulses_per_cross_point": pulses / (x_size * d_size)},
        "forward": {"ms_per_call": ms_forward, "gflops": flops_per_call / (ms_forward * 1e-3) / 1e9,
                    "mean_bm_rounds": float(rounds.mean()), "kernels_ms": {k: v[0] for k, v in prof_forward.items()},
                    "round_launches": contraction(prof_forward)[1],
                    "note": "with most samples in a second round the tile runs rounds 0 and 1 as one launch (round 2 as well "
                            "when its recent calls listed samples for it), with none the rounds after round 0 as one "
                            "launch (rpu_tile_set_fused_rounds, default: by what its last calls needed); same outputs"},
        "backward": {"ms_per_call": ms_backward, "gflops": flops_per_call / (ms_backward * 1e-3) / 1e9,
                     "kernels_ms": {k: v[0] for k, v in prof_backward.items()}},
        "roofline": {"kernel": k_update, "bound": "hbm", "achieved": update_bytes / (k_update_ms * 1e-3) / 1e9,
                     "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": update_bytes / (k_update_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                     "traffic": PMC_TRAFFIC_BYTES["k_update_pulsed_masks"] if args.config == 2 else None,
                     "traffic_source": ("constant from " + PMC_SOURCE["k_update_pulsed_masks"] + " (rocprofv3 --pmc FETCH_SIZE / "
                                        "WRITE_SIZE), not measured in this run") if args.config == 2 else None,
                     "algorithmic_bytes": update_bytes, "kernel_ms": k_update_ms},
        "roofline_forward": {"kernel": "k_mvm_dual + k_mvm_rounds_rest (all rounds of a call)" if fused_forward
                             else one_launch(prof_forward) or "k_mvm_round (all rounds of a call)", "bound": "mfma",
                             "achieved": flops_per_call / (k_fwd_ms * 1e-3) / 1e12, "peak": FP32_MFMA_PEAK_TFLOPS,
                             "unit": "TFLOP/s", "frac": flops_per_call / (k_fwd_ms * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                             "traffic": PMC_TRAFFIC_BYTES[fwd_traffic] if fwd_traffic else None,
                             "traffic_source": ("constant from " + PMC_SOURCE[fwd_traffic] + ", not measured in this run")
                             if fwd_traffic else None,
                             "algorithmic_flops": flops_per_call, "kernel_ms": k_fwd_ms},
        "roofline_backward": {"kernel": backward_kernel(prof_backward), "bound": "mfma",
                              "achieved": flops_per_call / (k_bwd_ms * 1e-3) / 1e12, "peak": FP32_MFMA_PEAK_TFLOPS,
                              "unit": "TFLOP/s", "frac": flops_per_call / (k_bwd_ms * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                              "kernel_ms": k_bwd_ms},
    }
    out["config"]["storage"] = args.storage
    if xd_block is not None:
        out["storage_xd_shared"] = xd_block
    if variants is not None:
        out["update_variants"] = variants
    if other is not None:
        out["same_tile_other_batches"] = other

    if not args.no_cpu_baseline:
        from oracle_lib import OracleTile

        orc = OracleTile(x_size, d_size, meta._config(dev))
        orc.set_weights(w)
        orc.set_learning_rate(lr)
        orc.set_seed(7)
        orc.forward(x[:8])
        t0 = time.perf_counter()
        orc.forward(x)
        cpu_fwd = time.perf_counter() - t0
        t0 = time.perf_counter()
        orc.backward(d)
        cpu_bwd = time.perf_counter() - t0
        n_upd = 3
        t0 = time.perf_counter()
        for _ in range(n_upd):
            orc.update(x, d)
        cpu_upd = (time.perf_counter() - t0) / n_upd
        # all host cores: the update of one tile is a sequence per cross-point and the oracle (like the reference's CPU
        # path) runs it on one thread, so the cores are used the way a model uses them: one independent tile per core
        import threading

        cores = int(os.environ.get("OMP_NUM_THREADS", "0")) or os.cpu_count() or 1
        cores = max(1, min(cores, os.cpu_count() or 1))
        many = []
        for k in range(cores):
            o = OracleTile(x_size, d_size, meta._config(dev))
            o.set_weights(w)
            o.set_learning_rate(lr)
            o.set_seed(100 + k)
            many.append(o)
        threads = [threading.Thread(target=lambda o=o: o.update(x, d)) for o in many]   # ctypes releases the GIL
        t0 = time.perf_counter()
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        cpu_all = time.perf_counter() - t0
        out["cpu_baseline"] = {
            "value": devices_per_call / cpu_upd / 1e9, "unit": "Gdevice-updates/s", "cores": 1, "kind": "port",
            "sample": f"{n_upd} full update calls, 1 forward and 1 backward call of the same workload on the CPU oracle "
                      "(1 thread).  The oracle draws its random numbers faster than the reference's CPU path: it takes about "
                      "0.23 s per update call where the compiled reference took 1.2 s when it was measured on another machine, "
                      "so this baseline is about five times faster than the reference itself would be",
            "update_ms": cpu_upd * 1e3, "forward_ms": cpu_fwd * 1e3, "forward_gflops": flops_per_call / cpu_fwd / 1e9,
            "backward_ms": cpu_bwd * 1e3, "backward_gflops": flops_per_call / cpu_bwd / 1e9,
            "host_cpus": os.cpu_count(),
            "all_cores": {"value": cores * devices_per_call / cpu_all / 1e9, "unit": "Gdevice-updates/s", "cores": cores,
                          "sample": f"one full update call on each of {cores} independent tiles at once, one thread per tile "
                                    "(a tile's update does not split over threads)", "wall_ms": cpu_all * 1e3},
        }
    print(json.dumps(out))
    return 0


def bench_config3(args) -> int:
    """Configuration 3: MLP 784-256-128-10 as three Tiki-Taka transfer tiles (SoftBounds A / C pairs, one column
    transferred every two mini-batches), batch 64.  A step = forward, backward and update of every tile on
    synthetic inputs and errors of the tile's shapes."""
    import numpy as np
    import torch

    from aihwkit_amd.rpu_base import tiles
    from aihwkit_amd.benchmark_configs import CONFIG3_SHAPES, config3

    torch.cuda.set_device(0)
    batch, lr = 64, 0.1
    rng = np.random.default_rng(0)
    layer = []
    for x_size, d_size in CONFIG3_SHAPES:
        meta, tr = config3()
        host = meta.create_array(x_size, d_size, tr)
        host.set_weights(torch.from_numpy(rng.uniform(-0.3, 0.3, (d_size, x_size)).astype(np.float32)))
        tile = tiles.CudaAnalogTile(host)
        tile.set_learning_rate(lr)
        tile.set_seed(99 + x_size)
        x = torch.from_numpy(rng.uniform(0, 1, (batch, x_size)).astype(np.float32)).cuda()
        d = torch.from_numpy((0.1 * rng.standard_normal((batch, d_size))).astype(np.float32)).cuda()
        layer.append((tile, x, d))

    def step():
        for tile, x, _ in layer:
            tile.forward(x, False, False, False, False, True)
        for tile, _, d in reversed(layer):
            tile.backward(d, False, False, False, True)
        for tile, x, d in layer:
            tile.update(x, d, False, False, False, True)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    devices = float(sum(x * d for x, d in CONFIG3_SHAPES)) * batch
    out = {
        "metric": "Tiki-Taka MLP 784-256-128-10 (three transfer tiles), training steps/s at batch 64, 1 MI355X",
        "value": 1e3 / ms_per_step, "unit": "steps/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": ms_per_step, "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic",
        "config": {"storage": args.storage, "workload": "config3: transfer compound of two SoftBounds devices per tile, tiles 785x256, 257x128, "
                               "129x10, batch 64, one column transferred every 2 mini-batches, stochastic pulses, 7/9-bit IO",
                   "batch": batch, "lr": lr, "step": "forward + backward + update of the three tiles"},
        "gdevice_updates_per_s": devices / (ms_per_step * 1e-3) / 1e9,
    }
    if not args.no_cpu_baseline:
        from transfer_oracle import TransferOracle

        cpu_ms = 0.0
        for (x_size, d_size), (_, x, d) in zip(CONFIG3_SHAPES, layer):
            meta, tr = config3()
            # the oracle samples nothing itself: it takes the device arrays of a host tile of the library
            host = meta.create_array(x_size, d_size, tr)
            orc = TransferOracle(x_size, d_size, meta._config(tr._vec_par[0]), tr._to_transfer_c())
            names, hidden, start = host.get_hidden_parameter_names(), host.get_hidden_parameters().numpy(), 0
            for k in range(len(tr._vec_par)):
                stop = names.index(f"hidden_weights_{k}")
                orc.set_device_hidden(k, hidden[start:stop].copy())
                start = stop + 1
            orc.set_learning_rate(lr)
            xh, dh = x.cpu().numpy(), d.cpu().numpy()
            t0 = time.perf_counter()
            for _ in range(2):  # two mini-batches: one transfer
                orc.forward(xh)
                orc.backward(dh)
                orc.update(xh, dh)
            cpu_ms += (time.perf_counter() - t0) * 1e3 / 2
        out["cpu_baseline"] = {"value": 1e3 / cpu_ms, "unit": "steps/s", "cores": 1, "kind": "port",
                               "sample": "2 steps of the same three tiles on the CPU transfer oracle (1 thread)",
                               "ms_per_step": cpu_ms, "host_cpus": os.cpu_count()}
    print(json.dumps(out))
    return 0


def bench_config5(args) -> int:
    """Configuration 5: forward pass of the four GPT-2-small linear shapes for 1024 tokens through PCM inference
    tiles (weights N(0, 0.02) programmed with PCM noise and drifted to one day, global drift compensation, 8-bit
    DAC / ADC, out_noise 0.04, abs-max noise management); the partial outputs of the input splits are summed
    digitally.  A step = the forward pass of all 38 tiles."""
    import torch

    from aihwkit_amd.benchmark_configs import CONFIG5_LAYERS, config5_groups, config5_layers, config5_step

    torch.cuda.set_device(0)
    tokens = 1024
    layers = config5_layers(tokens)
    n_tiles = sum(len(row) for grid in layers for _, row in grid)
    flops = sum(2.0 * tokens * in_size * out_size for in_size, out_size, _, _ in CONFIG5_LAYERS)

    def step_per_tile():
        outs = []
        for grid in layers:
            total = None
            for x_part, row in grid:
                y = torch.cat([tile.forward(x_part, is_test=True) for tile in row], dim=1)
                total = y if total is None else total + y
            outs.append(total)
        return outs

    for _ in range(3):
        step_per_tile()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(max(args.steps // 4, 3)):
        step_per_tile()
    torch.cuda.synchronize()
    ms_per_tile_loop = (time.perf_counter() - t0) * 1e3 / max(args.steps // 4, 3)

    groups = config5_groups(layers, tokens)

    def step():
        return config5_step(groups)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    out = {
        "metric": "noisy inference forward of the GPT-2-small linear shapes as 38 PCM tiles, tokens/s, 1 MI355X",
        "value": tokens / (ms_per_step * 1e-3), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms_per_step, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"storage": args.storage, "workload": "config5: 768->2304, 768->768, 768->3072, 3072->768 split into 38 tiles of at most 512 x 512, "
                               "1024 tokens, PCM programming noise + drift to 1 day + global drift compensation, 8-bit IO, "
                               "out_noise 0.04, abs-max noise management", "tokens": tokens, "tiles": n_tiles},
        "useful_tflops": flops / (ms_per_step * 1e-3) / 1e12,
        "ms_per_step_one_call_per_tile": ms_per_tile_loop,
    }
    print(json.dumps(out))
    return 0


def bench_config4(args) -> int:
    """Configuration 4: forward pass of a LeNet5-shaped stack for 512 images of 28 x 28: two 5 x 5 convolutions
    (1 -> 16, 16 -> 32) as indexed analog tiles, tanh and 2 x 2 max pooling in torch between them, then 512 -> 128 -> 10
    fully connected tiles.  Weights are programmed with PCM noise and drifted to one day with global drift
    compensation; 8-bit DAC / ADC.  A step = the forward pass of the 512 images."""
    import numpy as np
    import torch
    import torch.nn.functional as F

    from aihwkit_amd.inference import InferenceTile
    from aihwkit_amd.benchmark_configs import conv_index_matrix, io_params
    from aihwkit_amd.rpu_base import devices as dv

    torch.cuda.set_device(0)
    batch = 512
    rng = np.random.default_rng(0)
    io = io_params(inp_res=1 / 254.0, out_res=1 / 254.0, out_noise=0.06, noise_management=dv.NoiseManagementType.AbsMax,
                   bound_management=dv.BoundManagementType.Iterative)
    shapes = (("conv", (1, 28, 28), 16), ("conv", (16, 12, 12), 32), ("fc", 512, 128), ("fc", 128, 10))
    stack, flops, host_weights = [], 0.0, []
    for k, (kind, in_shape, out_size) in enumerate(shapes):
        if kind == "conv":
            indices, patches = conv_index_matrix(in_shape, (5, 5))
            in_size = in_shape[0] * 25 + 1
        else:
            indices, patches, in_size = None, 1, in_shape + 1
        w = (rng.uniform(-1, 1, (out_size, in_size)) / np.sqrt(in_size)).astype(np.float32)
        tile = InferenceTile(out_size, in_size, forward_io=io)
        tile.set_weights(torch.from_numpy(w))
        tile.cuda()
        tile.tile.set_seed(2000 + k)
        if indices is not None:
            tile.set_matrix_indices(indices)
        tile.drift_weights(86400.0)
        tile.compensate_in_tile(True)      # the drift-compensation factor rides on the ADC stage: no multiply of the output
        stack.append((kind, tile, patches, out_size))
        host_weights.append(w)
        flops += 2.0 * batch * patches * in_size * out_size
    x = torch.from_numpy(rng.uniform(0, 1, (batch, 1, 28, 28)).astype(np.float32)).cuda()

    def step():
        h = x
        for kind, tile, patches, out_size in stack:
            if kind == "conv":
                side = int(round(patches ** 0.5))
                y = tile.forward_indexed(h, torch.empty(h.size(0), out_size, side, side, device="cuda"), is_test=True)
                h = F.max_pool2d(torch.tanh(y), 2)
            else:
                h = tile.forward(h.reshape(h.size(0), -1), is_test=True, bias=True)     # the tile adds the bias column
                if out_size != 10:
                    h = torch.tanh(h)
        return h

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps

    cpu = None
    if not args.no_cpu_baseline:
        from indexed_oracle import IndexedOracle
        from oracle_lib import OracleTile

        sample = 16
        meta = dv.AnalogTileParameter()
        meta.forward_io = io
        t0 = time.perf_counter()
        h = x[:sample].cpu().numpy()
        for (kind, tile, patches, out_size), w in zip(stack, host_weights):
            orc = OracleTile(w.shape[1], w.shape[0], meta._config(dv.IdealResistiveDeviceParameter()))
            orc.set_weights(w)
            if kind == "conv":
                side = int(round(patches ** 0.5))
                in_shape = h.shape[1:]
                idx, _ = conv_index_matrix(in_shape, (5, 5))
                y = IndexedOracle(orc, idx.numpy(), patches).forward(h).reshape(sample, out_size, side, side)
                h = F.max_pool2d(torch.tanh(torch.from_numpy(y)), 2).numpy()
            else:
                flat = np.concatenate([h.reshape(sample, -1), np.ones((sample, 1), np.float32)], axis=1)
                h = orc.forward(np.ascontiguousarray(flat))
                if out_size != 10:
                    h = np.tanh(h)
        dt = time.perf_counter() - t0
        cpu = {"value": sample / dt, "unit": "images/s", "cores": 1, "kind": "port",
               "sample": "forward of %d images through the oracle tiles and the numpy index gather "
                         "(weights as set, without the PCM perturbation)" % sample}
    out = {
        "metric": "noisy inference forward of a LeNet5-shaped stack of PCM tiles, images/s, 1 MI355X",
        "value": batch / (ms_per_step * 1e-3), "unit": "images/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms_per_step, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"storage": args.storage, "workload": "config4: conv 1->16 5x5 (tile 26 x 16, 576 patches), conv 16->32 5x5 (tile 401 x 32, 64 "
                               "patches), fc 513 x 128, fc 129 x 10, batch 512 images 28 x 28, PCM programming noise + "
                               "drift to 1 day + global drift compensation, 8-bit IO, abs-max noise management",
                   "batch": batch},
        "useful_tflops": flops / (ms_per_step * 1e-3) / 1e12,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out))
    return 0


def bench_config6(args) -> int:
    """Supplementary configuration 6: one 3 x 3 convolution 48 -> 48 on 128 images of 34 x 34 (1024 patches per image,
    131072 in all) as an analog training tile of 433 x 48 (SoftBounds, IO of configuration 2) through the indexed
    interface: too wide for the fused convolution kernel, so the patches are gathered by the init kernels and the
    contraction runs on the large-tile kernel.  A step = forward + backward + update of the 128 images; the calls are
    also timed one by one, with their kernels (HIP events on the tile's stream)."""
    import numpy as np
    import torch

    from aihwkit_amd.benchmark_configs import config2, conv_index_matrix
    from aihwkit_amd.rpu_base import tiles

    torch.cuda.set_device(0)
    c_in, c_out, side, n = 48, 48, 34, 128
    rng = np.random.default_rng(0)
    indices, patches = conv_index_matrix((c_in, side, side), (3, 3))
    out_side = side - 2
    x_size = c_in * 9 + 1
    meta, dev = config2(noise=True)
    host = meta.create_array(x_size, c_out, dev)
    host.set_weights(torch.from_numpy(rng.uniform(-0.1, 0.1, (c_out, x_size)).astype(np.float32)))
    tile = tiles.CudaAnalogTile(host)
    tile.set_learning_rate(0.01)
    tile.set_matrix_indices(indices)
    x = torch.from_numpy(rng.uniform(0, 1, (n, c_in, side, side)).astype(np.float32)).cuda()
    g = torch.from_numpy(rng.normal(0, 0.01, (n, c_out, out_side, out_side)).astype(np.float32)).cuda()
    y = torch.empty(n, c_out, out_side, out_side, device="cuda")
    dx = torch.empty_like(x)
    calls = (("forward", lambda: tile.forward_indexed(x, y)), ("backward", lambda: tile.backward_indexed(g, dx)),
             ("update", lambda: tile.update_indexed(x, g)))

    def step():
        for _name, fn in calls:
            fn()

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    per_call = {}
    for name, fn in calls:
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            fn()
        torch.cuda.synchronize()
        tile.set_profiling(True)
        fn()
        kernels = [(k, round(ms, 5)) for k, ms in tile.get_profile()]
        tile.set_profiling(False)
        per_call[name] = {"ms_per_call": (time.perf_counter() - t0) * 1e3 / (args.steps + 1), "kernels_ms": kernels}
    flops = 2.0 * n * patches * x_size * c_out
    out = {
        "metric": "patches/s through forward + backward + update of one wide convolution tile, 1 MI355X (supplementary)",
        "value": n * patches / (ms_per_step * 1e-3), "unit": "patches/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms_per_step, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"storage": args.storage, "workload": "config6 (supplementary): conv 48->48 3x3 on 128 images 34 x 34 = 131072 patches, tile "
                               "433 x 48 SoftBounds (dtod + ctoc), BL 31, UM+UBLM, 7/9-bit IO, iterative BM, indexed "
                               "interface", "patches": n * patches},
        "calls": per_call,
        "forward_useful_tflops": flops / (per_call["forward"]["ms_per_call"] * 1e-3) / 1e12,
        "cpu_baseline": None,
    }
    print(json.dumps(out))
    return 0


if __name__ == "__main__":
    sys.exit(main())
