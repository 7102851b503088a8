#!/usr/bin/env python3
"""Benchmark of the fused CP4 Conv2d hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload C3] [--no-cpu]
                    [--settle-ms MS] [--shape PASS,N,C,H,W,pad,T,Y,R [--stride S]]
                    [--filter-variant V]

A step is one launch of the workload's pass (default: the forward pass of the
ResNet-stage workload N=32, C=K=256, 56x56, 3x3, R=32) on synthetic inputs that
are already resident in HBM.  Prints ONE JSON line:

  value        whole-job throughput = algorithmic bytes * K / wall time of the K
               steps (host clock, device synchronised on both sides), in GB/s
  roofline     the same K launches timed with HIP events on the launch stream:
               achieved GB/s = algorithmic bytes / mean launch duration, against
               the 8 TB/s HBM peak.  The headline loop re-launches on ONE buffer set,
               like the reference's PROFCOUNT loop; at C3 that set (206 MB) is
               smaller than the part's 256 MB memory-side cache, so `frac` is the
               cache-resident figure ("regime").  `cold` is the same event-timed
               loop rotating over --cold-sets distinct x / y sets (footprint well
               beyond the cache): every launch streams from and to HBM, which is
               what a training step sees.
  cpu_baseline the CPU oracle's unfused factor-by-factor computation of the same
               workload timed on this box's host cores (a reported baseline)
  passes       mean event-timed microseconds and GB/s of all five workloads

Before the W warm-up launches the headline workload runs untimed for
--settle-ms milliseconds (default 150): a launch takes ~45 us, and for the first
~30 ms of back-to-back launches the device's power management is still
settling (kernel durations rise by 10-20 % and come back down), so a short
run would time that transient instead of the steady state a training loop sees.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
FACTORS = ("FK", "FC", "FH", "FW")

# HBM bytes per launch of the dominant kernel from rocprofv3 --pmc FETCH_SIZE /
# WRITE_SIZE runs, scaled by the plain copy kernel's reading (profiles/), keyed by the
# workload AND the plan the counters were taken on (variant, strip rows, workgroups): a
# launch that runs another plan reports null rather than another kernel's bytes.
MEASURED_TRAFFIC = {
    # fwd_pipe_kernel<3,4,2,4,false,2> (results streamed): 107.1 MB fetched + 102.9 MB written
    ("C3", "mfma_bf16x3_pipe", 8, 224): 209.9e6,
}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--workload", default="C3")
    ap.add_argument("--shape", default=None, metavar="PASS,N,C,H,W,pad,T,Y,R",
                    help="time an ad-hoc shape instead of a named workload, e.g. "
                         "forward,8,64,224,224,1,64,3,16 (uniform inputs; no CPU leg, no table)")
    ap.add_argument("--stride", type=int, default=0,
                    help="with --shape: the same layer with this stride and the framework's "
                         "\"same\" padding (out = ceil(in / stride)); times all three passes "
                         "of the strided entry points and prints their figures")
    ap.add_argument("--settle-ms", type=float, default=150.0,
                    help="untimed back-to-back launches of the headline workload for this "
                         "long before the warm-up, so clocks are at their steady state")
    ap.add_argument("--cold-sets", type=int, default=4,
                    help="distinct x / y buffer sets of the rotating (HBM-streaming) leg of a "
                         "forward workload; 0 skips the leg")
    ap.add_argument("--cold-only", action="store_true",
                    help="run only the rotating leg (profiling: every launch of the process "
                         "then streams from and to HBM); prints that leg's figures")
    ap.add_argument("--filter-variant", type=int, default=-1,
                    help="backward-filter workloads: run this variant (0 general, 1 four launches, "
                         "2 three launches) instead of the library's choice")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-passes", action="store_true", help="skip the five-workload table")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run only the plain copy kernel on the workload's input size "
                         "(hardware-counter and bandwidth calibration)")
    args = ap.parse_args()
    if args.gpus != 1:
        sys.exit("bench.py: this path is built and measured on ONE GPU; --gpus must be 1 "
                 "(the passes shard over the batch with one small all-reduce of the factor "
                 "gradients; that is designed, not built)")

    import torch

    import paralleltnnlayers_amd as cp4
    from paralleltnnlayers_amd.configs import WORKLOADS, algorithmic_bytes, make_inputs

    cp4.lib()  # fail loudly if the HIP library is missing
    if not torch.cuda.is_available():
        sys.exit("bench.py: no GPU visible")
    torch.cuda.set_device(0)

    def device_inputs(w):
        a = make_inputs(w, seed=0)
        return a, {k: torch.from_numpy(v).cuda() for k, v in a.items()}

    def timed(w, d, warmup, steps, settle_ms=0.0):
        """(event-timed mean us, wall seconds of the same `steps` launches)."""
        f = [d[k] for k in FACTORS]
        if w.pass_ == "forward":
            out = torch.empty((w.N, w.T, w.H, w.W), device="cuda")
            run = lambda wu, k: cp4.time_forward(d["x"], *f, out, w.pad, wu, k)
        elif w.pass_ == "backward_data":
            out = torch.empty((w.N, w.C, w.H, w.W), device="cuda")
            run = lambda wu, k: cp4.time_backward_data(d["dy"], *f, out, w.pad, wu, k)
        else:
            s = cp4.capi.shape_for(d["x"].shape, *f, w.pad)
            ws = torch.empty(cp4.backward_filter_workspace_bytes(s) // 4 + 1, device="cuda")
            run = lambda wu, k: cp4.time_backward_filter(d["x"], d["dy"], *f, w.pad, wu, k,
                                                         workspace=ws)
        t_settle = time.perf_counter()
        while (time.perf_counter() - t_settle) * 1e3 < settle_ms:
            run(0, 500)
        run(warmup, 1)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        us = run(0, steps)          # K launches between one HIP event pair on the stream
        torch.cuda.synchronize()
        return us, time.perf_counter() - t0

    w = WORKLOADS[args.workload]
    if args.shape:
        from paralleltnnlayers_amd.configs import Workload
        f = args.shape.split(",")
        N, C, H, W_, pad, T, Y, R = (int(v) for v in f[1:])
        w = Workload("adhoc", f[0], N, C, H, W_, pad, T, Y, Y, R, "uniform")
        args.no_cpu = args.no_passes = True
    if args.stride:
        assert args.shape, "--stride goes with --shape"
        gen = torch.Generator(device="cuda").manual_seed(0)
        x = torch.rand((w.N, w.C, w.H, w.W), device="cuda", generator=gen)
        f = [torch.randn((d, w.R), device="cuda", generator=gen) * (w.R * w.C) ** -0.5
             for d in (w.T, w.C, w.Y, w.X)]
        s = cp4.capi.shape_for(x.shape, *f, 0)
        g = cp4.geometry(s, args.stride, "same")
        y = torch.empty((w.N, w.T, g.out_h, g.out_w), device="cuda")
        dy = torch.randn(y.shape, device="cuda", generator=gen)
        dx = torch.empty_like(x)
        ws = torch.empty(cp4.backward_ex_workspace_bytes(s, g) + 512, device="cuda",
                         dtype=torch.uint8)
        ws = ws[(-ws.data_ptr()) % 256:]
        legs = {"forward": lambda: cp4.conv2d_forward_ex(x, *f, g, out=y),
                "backward_data": lambda: cp4.conv2d_backward_data_ex(dy, (w.H, w.W), *f, g, out=dx,
                                                                     workspace=ws),
                "backward_filter": lambda: cp4.conv2d_backward_filter_ex(x, dy, *f, g, workspace=ws)}
        nb = 4 * (x.numel() + y.numel())
        res = {}
        for name, fn in legs.items():
            t0 = time.perf_counter()
            while (time.perf_counter() - t0) * 1e3 < args.settle_ms:
                fn()
            for _ in range(args.warmup):
                fn()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(args.steps):
                fn()
            e1.record()
            torch.cuda.synchronize()
            us = e0.elapsed_time(e1) * 1e3 / args.steps
            res[name] = {"us": round(us, 2), "GB/s": round(nb / us / 1e3, 1),
                         "hbm_frac": round(nb / us / 1e3 / HBM_PEAK_GBS, 4)}
        cp4.device_status()
        print(json.dumps({"workload": "%s stride %d, out %dx%d" % (args.shape, args.stride, g.out_h,
                                                                  g.out_w),
                          "algorithmic_bytes": nb, "passes": res}))
        return
    if args.calibrate_copy:
        n = w.N * w.C * w.H * w.W
        src = torch.randn(n, device="cuda")
        dst = torch.empty_like(src)
        us = cp4.time_copy(dst, src, warmup=args.warmup, profcount=args.steps)
        print(json.dumps({"kernel": "copy_f32x4_kernel", "bytes_read": 4 * n, "bytes_written": 4 * n,
                          "us_per_launch": round(us, 2),
                          "GB/s": round(8 * n / us / 1e3, 1)}))
        return
    host, d = device_inputs(w)
    nbytes = algorithmic_bytes(w)
    if args.cold_only:
        assert w.pass_ == "forward" and args.cold_sets > 0
        f = [d[k] for k in FACTORS]
        xs = [d["x"]] + [d["x"].clone() for _ in range(args.cold_sets - 1)]
        ys = [torch.empty((w.N, w.T, w.H, w.W), device="cuda") for _ in xs]
        t_settle = time.perf_counter()
        while (time.perf_counter() - t_settle) * 1e3 < args.settle_ms:
            cp4.time_forward_sets(xs, *f, ys, w.pad, 0, 200)
        cus = cp4.time_forward_sets(xs, *f, ys, w.pad, args.warmup, args.steps)
        print(json.dumps({"workload": w.name, "sets": len(xs), "us_per_launch": round(cus, 2),
                          "GB/s": round(nbytes / cus / 1e3, 1),
                          "hbm_frac": round(nbytes / cus / 1e3 / HBM_PEAK_GBS, 4)}))
        return
    shape = cp4.capi.shape_for((w.N, w.C, w.H, w.W), *[d[k] for k in FACTORS], w.pad)
    if args.filter_variant >= 0:
        assert w.pass_ == "backward_filter", "--filter-variant goes with a backward-filter workload"
        cp4.set_tuned_filter_choice(shape, args.filter_variant)
    plan = cp4.plan_query(shape, w.pass_)
    us, wall = timed(w, d, args.warmup, args.steps, args.settle_ms)
    value = nbytes * args.steps / wall / 1e9
    achieved = nbytes / us / 1e3

    cold = None
    if w.pass_ == "forward" and args.cold_sets > 0:
        f = [d[k] for k in FACTORS]
        xs = [d["x"]] + [d["x"].clone() for _ in range(args.cold_sets - 1)]
        ys = [torch.empty((w.N, w.T, w.H, w.W), device="cuda") for _ in xs]
        cp4.time_forward_sets(xs, *f, ys, w.pad, args.warmup, max(args.steps // 4, 1))
        cus = cp4.time_forward_sets(xs, *f, ys, w.pad, args.warmup, args.steps)
        cold = {"us": round(cus, 2), "achieved": round(nbytes / cus / 1e3, 1),
                "frac": round(nbytes / cus / 1e3 / HBM_PEAK_GBS, 4), "sets": len(xs),
                "footprint_bytes": len(xs) * 4 * (d["x"].numel() + ys[0].numel())}
        del xs, ys

    out = {
        "metric": "CP4 conv2d %s achieved HBM GB/s (algorithmic bytes / time), 1 GPU" % w.pass_,
        "value": round(value, 1), "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(wall / args.steps * 1e3, 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "synthetic",
        "config": {"workload": "%s %s fp32 NCHW N=%d C=%d K=%d H=W=%d %dx%d pad=%d R=%d"
                               % (w.name, w.pass_, w.N, w.C, w.T, w.H, w.Y, w.X, w.pad, w.R),
                   "algorithmic_bytes": nbytes, "us_per_launch": round(us, 2), "plan": plan},
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                     "traffic": MEASURED_TRAFFIC.get((w.name, plan["variant"], plan["strip_rows"],
                                                      plan["workgroups"])),
                     "regime": "one buffer set re-launched (%.0f MB working set; the part's "
                               "memory-side cache holds 256 MB)" % (nbytes / 1e6),
                     "cold": cold},
    }

    if not args.no_passes:
        passes = {}
        for name, ww in WORKLOADS.items():
            if name == w.name:
                t = us
            else:
                _, dd = device_inputs(ww)
                t, _ = timed(ww, dd, 5, 200, args.settle_ms)
                del dd
            b = algorithmic_bytes(ww)
            passes[name] = {"pass": ww.pass_, "us": round(t, 2),
                            "GB/s": round(b / t / 1e3, 1),
                            "hbm_frac": round(b / t / 1e3 / HBM_PEAK_GBS, 4)}
        out["passes"] = passes

    if not args.no_cpu:
        from oracle import cp4_oracle
        fa = [host[k] for k in FACTORS]
        fn = {"forward": lambda: cp4_oracle.forward(host["x"], *fa, w.pad),
              "backward_data": lambda: cp4_oracle.backward_data(host["dy"], *fa, w.pad),
              "backward_filter": lambda: cp4_oracle.backward_filter(host["x"], host["dy"], *fa,
                                                                    w.pad)}[w.pass_]
        fn()  # warm-up
        best, reps, t_start = None, 0, time.perf_counter()
        while reps < 5 and time.perf_counter() - t_start < 20.0:
            t0 = time.perf_counter()
            fn()
            dt = time.perf_counter() - t0
            best = dt if best is None else min(best, dt)
            reps += 1
        out["cpu_baseline"] = {
            "value": round(nbytes / best / 1e9, 3), "unit": "GB/s",
            "cores": cp4_oracle.num_threads(), "kind": "port",
            "sample": "full %s workload, best of %d runs, %.1f ms each (OpenMP unfused "
                      "factor-by-factor oracle)" % (w.name, reps, best * 1e3)}

    print(json.dumps(out))


if __name__ == "__main__":
    main()
