"""Benchmark: SeeML LoRA update steps on one MI355X through the gfx950 backend.

A "step" is one TrainImpl iteration of the compiled plan (update_engine.cc:
736-753): step scalars, device-resident batch staged into the plan's I/O
slots, the train program replayed as one hipGraph, the loss read back and
checked. Inputs are resident in HBM before timing starts.

Default workload: BASELINE configs[3] (C4, the d_model-2048 decoder the
north-star target is stated on: V32000, 16 layers, 16x128 heads, seq 1024 x
8, SwiGLU 5504, LoRA r16 on q/k/v/o). --config selects c1..c5.

Emits ONE JSON line (rank 0) with, besides the driver's fields:
  roofline      the dominant kernel — the (opcode, shape, tile) group with
                the largest share of step time — its launches timed inside
                the train graph by device wall-clock stamp nodes over the
                timed steps: algorithmic FLOPs (or bytes) of one launch /
                mean launch time, vs MI355X peak; `traffic` is
                the HBM bytes per launch from the committed rocprofv3 PMC
                summary for that kernel (profiles/), when one matches
  cpu_baseline  the reference's own executor kernels (oracle/_ref, built
                from the reference sources) timed on this host's cores and on
                one thread: steps-lo/hi slopes (C1-C3) or the per-kernel-group
                model (C4/C5), oracle/cpu_baseline.py
  ms_per_step_slope  the reference bench's own step timing: the slope
                between steps-4 and steps-12 runs, median of 3
  kernels       per-opcode time split, dense-GEMM MFMA utilisation and the
                HBM throughput of the bandwidth-bound kernels
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "see-ml_amd"))

PEAK_FP32_MFMA_TFLOPS = 157.3
# fp32 products as the tile GEMMs form them: six bf16 products each
PEAK_GEMM_TFLOPS = round(2516.6 / 6, 1)
PEAK_HBM_GBPS = 8000.0


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def cpu_baseline(w, plan, cores):
    """The reference's own executor kernels (oracle/_ref, compiled from the
    reference sources) timed on this host's cores and on one thread, as
    oracle/cpu_baseline.py describes: whole-step steps-lo/hi slopes for C1-C3,
    the per-kernel-group model (each distinct instruction group timed on a
    bounded sample of its work, times its multiplicity) for C4/C5 and for
    every one-thread figure."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import cpu_baseline as cb
    import oracle
    from seeml_amd import planner

    if not oracle.ref_available():
        raise RuntimeError("oracle/_ref is not built (the reference sources were absent)")
    if w.name in cb.STEP_SLOPE and plan.blob is None:  # released after upload
        plan = planner.compile_update(w.model, w.cfg)
    return cb.measure(w, plan, cores)


def measured_traffic(kernel: str):
    """HBM bytes per launch of `kernel` from a committed rocprofv3 PMC
    summary (profiles/*.md carrying a line
    `traffic: kernel="<kernel>" bytes_per_launch=<B>`), else (None, None)."""
    import glob
    import re
    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*.md"))):
        for line in open(path):
            m = re.search(r'traffic: kernel="([^"]+)" bytes_per_launch=(\d+)', line)
            if m and m.group(1) == kernel:
                return int(m.group(2)), os.path.relpath(path, ROOT)
    return None, None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--config", default="c4")
    ap.add_argument("--no-autotune", action="store_true")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--profile-reps", type=int, default=3)
    ap.add_argument("--slope-lo", type=int, default=4)
    ap.add_argument("--slope-hi", type=int, default=12)
    args = ap.parse_args()

    if args.gpus != 1:
        print(f"bench.py: this build runs on exactly one GPU; --gpus {args.gpus} is not "
              "supported (the multi-GPU design is described, not built)", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    from seeml_amd import DeviceUpdateEngine, PROGRAM_TRAIN, configs, planner, workmodel

    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)

    w = configs.make(args.config)
    t0 = time.perf_counter()
    plan = planner.compile_update(w.model, w.cfg)
    log(f"plan {w.name}: {len(plan.train)} train instrs, arena {plan.header['arena_size'] / 1e9:.2f} GB, "
        f"rodata {plan.header['rodata_size'] / 1e9:.2f} GB ({time.perf_counter() - t0:.1f}s)")
    e = DeviceUpdateEngine(plan.blob)
    plan.blob = None  # the device holds its copy; free the host bytes
    log("engine open")
    if not args.no_autotune:
        t0 = time.perf_counter()
        e.autotune(16)
        log(f"autotuned GEMM tiles ({time.perf_counter() - t0:.1f}s)")

    dev = torch.device("cuda:0")
    batches = []
    for s in range(2):
        x, y = configs.batch(w, s)
        batches.append((torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)))
    torch.cuda.synchronize()

    losses = []
    for s in range(args.warmup):
        xb, yb = batches[s % 2]
        losses.append(e.train_step(xb, yb))
    log(f"warmup done, loss {losses[-1] if losses else float('nan'):.6f}")

    # Per-instruction breakdown (eager replay with events, before the timed
    # region) picks the dominant kernel: the (opcode, shape, tile) group with
    # the largest share of the step.
    ms = e.profile(PROGRAM_TRAIN, reps=args.profile_reps)
    variants = [e.gemm_choice(PROGRAM_TRAIN, i) for i in range(len(plan.train))]
    launches = [e.launch_work(PROGRAM_TRAIN, i) for i in range(len(plan.train))]
    summ = workmodel.summarize(plan.train, list(ms), PEAK_GEMM_TFLOPS, PEAK_HBM_GBPS,
                               variants=variants, launches=launches)
    rows = summ["rows"]
    groups = {}
    for i, r in enumerate(rows):
        tile = variants[i]
        g = groups.setdefault((r["op"], tuple(r["shape"]), tile), [0.0, []])
        g[0] += r["ms"]
        g[1].append(i)
    (dom_op, dom_shape, dom_tile), (dom_total, dom_idx) = max(groups.items(), key=lambda kv: kv[1][0])
    log("top (op, shape, tile) groups by step share:")
    for (op, shape, tile), (tot, idx) in sorted(groups.items(), key=lambda kv: -kv[1][0])[:40]:
        r0 = rows[idx[0]]
        if tot <= 0.0:  # fused into another launch: no time of its own
            rate = "      -"
        elif r0["flops"]:
            rate = f"{r0['flops'] * len(idx) / (tot * 1e-3) / 1e12:7.1f} TFLOP/s"
        else:
            rate = f"{r0['bytes'] * len(idx) / (tot * 1e-3) / 1e9:7.0f} GB/s"
        log(f"  {tot:8.3f} ms  x{len(idx):<4d} {op:15s} {'x'.join(map(str, shape)):22s} {tile:28s} {rate}")
    dom_row = rows[dom_idx[0]]
    # Its launches get event-record nodes in the train graph, timed live in
    # every timed step on the engine stream.
    e.mark_timed(PROGRAM_TRAIN, dom_idx)
    e.build(PROGRAM_TRAIN)
    xb, yb = batches[0]
    losses.append(e.train_step(xb, yb))  # first replay of the rebuilt graph, untimed

    e.marked_times(PROGRAM_TRAIN)  # restarts the device-side sums: the timed steps' alone
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for s in range(args.steps):
        xb, yb = batches[s % 2]
        losses.append(e.train_step(xb, yb))  # returns after the step's loss read (synchronized)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    # each marked launch's mean over the K timed steps, summed on the device
    launch_ms = [e.marked_times(PROGRAM_TRAIN)]
    ms_per_step = dt / args.steps * 1e3
    tokens_per_s = w.cfg.batch * args.steps / dt
    log(f"timed {args.steps} steps: {ms_per_step:.3f} ms/step, {tokens_per_s:.1f} tok/s")

    # The reference bench's method (tool/seeml_bench.cc:288-310): per-step
    # time = the slope between a steps-lo and a steps-hi run, median of 3
    # (reported beside the contract's K-step figure; outside its timing).
    e.mark_timed(PROGRAM_TRAIN, [])
    losses.append(e.train_step(*batches[0]))  # the unsplit graph's first replay, untimed
    slopes = []
    lo, hi = args.slope_lo, args.slope_hi
    for _ in range(3 if hi > lo else 0):
        walls = []
        for n in (lo, hi):
            torch.cuda.synchronize()
            t1 = time.perf_counter()
            for s in range(n):
                xb, yb = batches[s % 2]
                losses.append(e.train_step(xb, yb))
            torch.cuda.synchronize()
            walls.append(time.perf_counter() - t1)
        slopes.append((walls[1] - walls[0]) / (hi - lo) * 1e3)
    slope_ms = float(np.median(slopes)) if slopes else None
    if slope_ms:
        log(f"steps-{lo}/{hi} slope: {slope_ms:.3f} ms/step (median of 3)")

    dom_ms = float(np.mean(np.concatenate(launch_ms)))
    if dom_row["cls"] == "mfma" or (dom_row["cls"] == "attn" and dom_row["flops"]):
        achieved = dom_row["flops"] / (dom_ms * 1e-3) / 1e12
        peak = PEAK_GEMM_TFLOPS if dom_row["cls"] == "mfma" else PEAK_FP32_MFMA_TFLOPS
        roof = dict(bound="mfma", achieved=round(achieved, 3), peak=peak,
                    unit="TFLOP/s", frac=round(achieved / peak, 4))
    else:
        achieved = dom_row["bytes"] / (dom_ms * 1e-3) / 1e9
        roof = dict(bound="hbm", achieved=round(achieved, 1), peak=PEAK_HBM_GBPS, unit="GB/s",
                    frac=round(achieved / PEAK_HBM_GBPS, 4))
    kernel = f"{dom_op} {'x'.join(map(str, dom_shape))}" + (f" {dom_tile}" if dom_tile else "")
    traffic, traffic_src = measured_traffic(kernel)
    roof.update(kernel=kernel, launches_per_step=len(dom_idx),
                step_share=round(dom_total / summ["total_ms"], 4),
                launch_ms=round(dom_ms, 4),
                timing=f"device wall-clock stamp nodes around its {len(dom_idx)} launches per "
                       f"step inside the train graph, summed on the device over the "
                       f"{args.steps} timed steps",
                traffic=traffic, traffic_source=traffic_src,
                algorithmic=(f"{dom_row['flops']} FLOP" if roof["bound"] == "mfma"
                             else f"{dom_row['bytes']} B"),
                algorithmic_bytes=dom_row["bytes"])
    by_op = {k: dict(count=v["count"], ms=round(v["ms"], 4),
                     share=round(v["ms"] / summ["total_ms"], 4)) for k, v in
             sorted(summ["by_op"].items(), key=lambda kv: -kv[1]["ms"])}

    cpu = None
    if not args.no_cpu_baseline:
        # This process's cores, capped at a GPU box's CPU share per GPU (16
        # threads per GPU, whatever the host reports); the host's own count
        # and this process's affinity are recorded beside it.
        affinity = len(os.sched_getaffinity(0))
        cores = min(16, affinity)
        log(f"cpu baseline on {cores} cores (host reports {os.cpu_count()}, affinity {affinity}) ...")
        try:
            cpu = cpu_baseline(w, plan, cores)
        except Exception as ex:  # reported, never fatal for the GPU figure
            cpu = dict(value=None, unit="tokens/s", cores=cores, kind="reference",
                       sample=f"unavailable: {ex}")
        cpu["host_cpus"] = os.cpu_count()
        cpu["affinity_cpus"] = affinity
        cpu["cores_note"] = ("threads capped at the GPU box's CPU share of 16 per GPU; "
                             "host_cpus is os.cpu_count() on the box")
    out = {
        "metric": "train tokens/sec per update step on 1 MI355X; GEMM MFMA util %; HBM GB/s",
        "value": round(tokens_per_s, 2),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "ms_per_step_slope": round(slope_ms, 4) if slope_ms else None,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded; weights/inputs generated, no dataset)",
        "config": {
            "workload": f"{w.name}: {w.description}",
            "global_batch": w.cfg.batch,
            "seq_len": w.seq or None,
            "parallelism": "none (1 GPU)",
            "train_instructions": len(plan.train),
            "autotuned": not args.no_autotune,
        },
        "gemm_dense_mfma_util": summ["gemm_dense_mfma_util"],
        "gemm_all_mfma_util": summ["gemm_all_mfma_util"],
        "hbm_kernels_gbps": summ["hbm_kernels_gbps"],
        "hbm_elementwise_gbps": summ["hbm_elementwise_gbps"],
        "hbm_skinny_gemm_gbps": summ["hbm_skinny_gemm_gbps"],
        "roofline": roof,
        "cpu_baseline": cpu,
        "kernels": by_op,
        "final_loss": losses[-1],
    }
    def plain(v):
        if isinstance(v, dict):
            return {k: plain(x) for k, x in v.items()}
        if isinstance(v, (list, tuple)):
            return [plain(x) for x in v]
        if hasattr(v, "item"):
            return v.item()
        return v
    print(json.dumps(plain(out)), flush=True)
    e.close()


if __name__ == "__main__":
    main()
