"""Benchmark of the mapped-convolution hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--interp bilinear|nearest]

A step is one forward + backward (grad_input, grad_weight, grad_bias) of a
MappedConvolution at the headline configuration: B=8, 64->64 channels, 256x512
equirectangular input, 3x3 latitude-distorted sample map, fp32, synthetic data
resident in HBM.  Prints ONE JSON line: Mpix/s (B*OH*OW per step / time), the
roofline position of the dominant kernel (timed with events on the launch stream
inside the timed region) and the reference CPU implementation timed on this
host's cores on a bounded sample of the same workload.
"""
import argparse
import json
import os
import statistics
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

from mappedconvolutions_amd import _C  # noqa: E402
from mappedconvolutions_amd.util import synthetic  # noqa: E402

B, CI, CO, H, W, K = 8, 64, 64, 256, 512, 9
# Dense peak of the unit the timed calls' dominant kernels multiply on: six bf16 matrix
# instructions per fp32 product.
PEAK_SPLIT_TFLOPS = 2500.0 / 6
GEMM_FLOP = 2.0 * B * H * W * CO * CI * K  # one of the three products

TRAFFIC_PROFILE = os.path.join(ROOT, "profiles", "conv_fwd_bwd_headline_hbm_traffic.txt")


def recorded_traffic():
    """Kernel name and bytes crossing the L2 boundary per launch, per timed C-ABI call, from the
    committed counter summary (FETCH_SIZE / WRITE_SIZE passes of this script, scaled by copy
    dispatches of known size; bench_traffic_summary.py writes it).  Counters
    cannot be read from inside the process, so these are recorded figures: they are dropped when
    a kernel source has changed since the counter run."""
    import re
    from bench_traffic_summary import source_lines
    table = {}
    try:
        text = open(TRAFFIC_PROFILE).read()
    except OSError:
        return {}, False
    lines = text.splitlines()
    fresh = set(source_lines()) == {line for line in lines if line.startswith("@source ")}
    for line in lines:
        m = re.match(r'@traffic label=(\w+) kernel="([^"]+)" read_bytes=(\d+) written_bytes=(\d+)',
                     line)
        if m:
            table[m.group(1)] = (m.group(2), int(m.group(3)) + int(m.group(4)))
    return table, fresh


def make_inputs(device, batch=B):
    g = torch.Generator().manual_seed(0)
    x = torch.randn(batch, CI, H, W, generator=g)
    gy = torch.randn(batch, CO, H, W, generator=g)
    w = torch.randn(CO, CI, K, generator=g) * (2.0 / (CI * K)) ** 0.5
    b = torch.zeros(CO)
    smap = synthetic.latitude_map(H, W, 1)
    return [t.to(device) for t in (x, gy, w, b, smap)]


def step(x, gy, w, b, smap, interp):
    y = _C.mapped_conv_forward(x, smap, w, b, K, interp)
    grads = _C.mapped_conv_backward(gy, smap, x, w, b, K, interp)
    return y, grads


def cpu_baseline(interp):
    """Reference CPU implementation (oracle/_ref, built from the reference's own
    sources) on a B=1 slice of the workload; falls back to the C port."""
    from oracle import reference
    x, gy, w, b, smap = make_inputs("cpu", batch=1)
    if reference.available():
        mod, kind = reference.module("_mapped_convolution"), "reference"
    else:
        from oracle import ops as mod
        kind = "port"
    def once():
        t0 = time.perf_counter()
        mod.mapped_conv_forward(x, smap, w, b, K, interp)
        mod.mapped_conv_backward(gy, smap, x, w, b, K, interp)
        return time.perf_counter() - t0

    warm = once()
    reps = int(min(40, max(3, 12.0 / max(warm, 1e-3))))  # about 12 s of CPU work
    times = [once() for _ in range(reps)]
    t = statistics.median(times)
    return {"value": round(H * W / t / 1e6, 4), "unit": "Mpix/s", "cores": torch.get_num_threads(),
            "kind": kind,
            "sample": "B=1 slice (1 of 8 images; the reference loops over the batch, so cost is "
                      "linear in B), forward+backward, 1 warm-up + median of %d, %.2f s each"
                      % (reps, t)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=30,
                    help="untimed steps first; the GPU needs some 50 ms of work to reach its clock "
                         "(3 steps measured 2.5 %% slower than 30 or 100)")
    ap.add_argument("--interp", default="bilinear", choices=["bilinear", "nearest"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--map-plan-cache", action="store_true",
                    help="not the headline configuration: keep the backward's plan of the sample "
                         "map (transposed map, pair masks) across steps instead of rebuilding "
                         "it in every call as the reference's kernels decode the map every call")
    ap.add_argument("--calibration-copy", action="store_true",
                    help="before the warm-up, run three plain copy kernels over the input "
                         "(reads and writes B*Ci*H*W*4 bytes each) so that a counter run of this "
                         "command holds a dispatch of known traffic to scale FETCH_SIZE/WRITE_SIZE by")
    args = ap.parse_args()
    if args.gpus != 1:
        sys.exit("bench.py measures one GPU: this build has no multi-GPU path (--gpus must be 1)")
    if not torch.cuda.is_available():
        sys.exit("bench.py needs a GPU")
    interp = 1 if args.interp == "bilinear" else 0
    _C.enable_map_plan_cache(args.map_plan_cache)
    dev = torch.device("cuda:0")
    inputs = make_inputs(dev)

    if args.calibration_copy:
        dst = torch.empty_like(inputs[0])
        for _ in range(3):
            torch.mul(inputs[0], 1.0, out=dst)  # one elementwise kernel: 1 read + 1 write per element
        torch.cuda.synchronize()
        del dst

    for _ in range(args.warmup):
        step(*inputs, interp)
    torch.cuda.synchronize()
    _C.profile_pool = _C.make_event_pool(3 * args.steps, dev)
    torch.cuda.synchronize()
    _C.profile_events = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step(*inputs, interp)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    events, _C.profile_events = _C.profile_events, None

    # per C-ABI call: its dominant kernel alone (events recorded by the library around
    # that launch, on the launch stream)
    per_kernel = {}
    for label, k0, k1 in events:
        per_kernel.setdefault(label, []).append(k0.elapsed_time(k1))
    kernel_ms = {k: sum(v) / len(v) for k, v in per_kernel.items()}
    dominant = max(kernel_ms, key=kernel_ms.get)
    achieved = GEMM_FLOP / (kernel_ms[dominant] * 1e-3) / 1e12
    peak = PEAK_SPLIT_TFLOPS

    ms = elapsed / args.steps * 1e3
    # (the recorded counter runs cover the bilinear headline workload without a plan cache)
    recorded, fresh = recorded_traffic() if interp == 1 and not args.map_plan_cache else ({}, False)
    out = {
        "metric": "Mapped-conv fwd+bwd Mpix/s (B8,C64,256x512,3x3); % HBM/MFMA roofline",
        "value": round(B * H * W / (ms * 1e-3) / 1e6, 3),
        "unit": "Mpix/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "synthetic",
        "config": {"workload": "MappedConvolution fwd+bwd B8 Ci64 Co64 256x512 K9 latitude map, "
                               + args.interp, "interpolation": args.interp,
                   "map_plan_cache": bool(args.map_plan_cache)},
        "roofline": {"bound": "mfma", "kernel": recorded.get(dominant, (dominant, None))[0],
                     "achieved": round(achieved, 3), "peak": round(peak, 1),
                     "unit": "TFLOP/s", "frac": round(achieved / peak, 4),
                     "traffic": recorded[dominant][1] if fresh and dominant in recorded else None,
                     "traffic_unit": "bytes per launch",
                     "traffic_source": "profiles/conv_fwd_bwd_headline_hbm_traffic.txt"
                                       if fresh and dominant in recorded else
                                       "none: no counter run of this kernel source is recorded"},
        "kernel_ms": {k: round(v, 4) for k, v in kernel_ms.items()},
    }
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline(interp)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
