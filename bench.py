"""Fine training-step throughput on one MI355X (rays/s), with HBM roofline and the
CPU restatement timed beside it.

Workload: the plain fine step -- 256^3 float32 SDF grid (analytic perturbed sphere) +
256^3 x 12 float32 feature grid ~N(0, 0.1^2), rgbnet 42->192->192->192->3, 8192 rays per
step from the radius-3 sphere, stepsize 0.5 voxel, s = 256, forward + backward + Adam
(lr sdf 5e-3, k0 0.1, rgbnet 3e-3).  A pool of ray batches is generated once and kept
in HBM; each step takes the next batch.

  python bench.py [--gpus 1] [--steps K] [--warmup W] [--path fused|ops] [--no-cpu]

Prints one JSON line.
"""
import argparse
import gc
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

# Peak figures of an MI355X used for roofline fractions.
PEAK_HBM_GBS = 8000.0
PEAK_FP32_MFMA_TF = 157.3
PEAK_BF16_MFMA_TF = 2500.0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--prime", type=int, default=256,
                    help="ray batches whose reachable k0 pages are counted as touched before "
                         "timing (untimed, no training): the Adam sweep of a short run then "
                         "covers what a long run's would")
    ap.add_argument("--path", choices=["fused", "ops"], default="fused")
    ap.add_argument("--mlp", choices=["fp32", "fp32-mfma", "bf16"], default="fp32",
                    help="rgbnet arithmetic: fp32 = FP32 accuracy through three-way BF16 "
                         "splits (six BF16 MFMA products per pair); fp32-mfma = FP32 MFMAs; "
                         "bf16 = single BF16 MFMAs, bf16 activations")
    ap.add_argument("--rays", type=int, default=8192)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--serial-adam", action="store_true",
                    help="run the k0 Adam pass in order on the main stream (per-kernel timing)")
    ap.add_argument("--wgrad-blocks", type=int, default=None,
                    help="row blocks of rgbnet's weight-gradient passes on the third stream "
                         "(default: the trainer's; 0 = one per CU)")
    ap.add_argument("--bounds-now", action="store_true",
                    help="compute the empty-space bounds right before each forward on the "
                         "main stream (default: during the step before, on the second stream)")
    ap.add_argument("--bounds-at-start", action="store_true",
                    help="queue the next step's bounds at the start of the step, beside the "
                         "walk (default: behind the walk and the zero-gradient Adam pages)")
    ap.add_argument("--overlap-sdf-bwd", nargs="?", const="rgbnet", default=None,
                    choices=["rgbnet", "scatter"],
                    help="run phase 1 of the SDF backward on a stream of its own beside the "
                         "rgbnet backward (rgbnet, the flag alone) or beside the feature "
                         "scatter (scatter); default: in order on the main stream")
    ap.add_argument("--serial-wgrad", action="store_true",
                    help="run rgbnet's weight gradients and Adam pass in order on the main stream")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--mode", choices=["train", "coarse", "recompute", "precision", "serve",
                                       "kernels", "next_rows"],
                    default="train",
                    help="train: the plain fine step (the headline line); coarse: the plain "
                         "coarse step; recompute: 65536-ray fine step, per-ray recomputation "
                         "vs store-all; precision: BF16 rgbnet vs FP32 vs FP64; serve: the "
                         "render/SDF-query server vs sequential per-request rendering; "
                         "next_rows: ray pre-filter, regularisers, mesh extraction")
    ap.add_argument("--requests", type=int, default=300)
    ap.add_argument("--rate", type=float, default=50.0)
    ap.add_argument("--kernel-steps", type=int, default=5,
                    help="untimed steps after the timed region whose kernels are timed one by "
                         "one with HIP events (per-kernel HBM GB/s); 0 skips them")
    ap.add_argument("--serve-requests", type=int, default=120,
                    help="requests of the serving run reported in the default line (0 skips it)")
    ap.add_argument("--serve-rate", type=float, default=200.0,
                    help="Poisson arrival rate of that run (req/s), above what one GPU serves, so "
                         "the throughputs of the two schedulers are compared at saturation")
    ap.add_argument("--seeds", type=int, default=10)
    ap.add_argument("--psnr-steps", type=int, default=200)
    return ap.parse_args()


def step_bytes(cfg, counts):
    """Algorithmic HBM bytes of one fine step (read/write of every grid element by Adam
    and the gradient clear, ray I/O, and the trilinear corner traffic of the gathers and
    scatters), from the per-step sample counts."""
    R, C = cfg.R, cfg.feat_dim
    n_e = R ** 3 * (1 + C)
    if not all(k in counts for k in ("m0", "m1b", "m2")):
        return None
    m0, m1b, m2 = counts["m0"], counts["m1b"], counts["m2"]
    return (32 * n_e + 60 * cfg.n_rays + m0 * 7 * 8 * 4 + m2 * 8 * C * 4 + m1b * 7 * 8 * 8
            + m2 * 8 * C * 8)


def host_cpus():
    """CPUs this process may run on (the cgroup/affinity share of the host, which on a
    shared GPU host is smaller than os.cpu_count()), capped by OMP_NUM_THREADS when the
    environment sets it."""
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    omp = os.environ.get("OMP_NUM_THREADS", "")
    if omp.isdigit() and int(omp) > 0:
        n = min(n, int(omp))
    return max(1, n)


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(cfg, threads, steps=3):
    """The reference's step restated in PyTorch on the CPU (the oracle: lib/cuda ops
    transcribed to torch CPU, F.grid_sample, nn.Linear, index_add_ for segment_coo,
    utils.Adam) on the same fine workload: one warm-up step, then the median of `steps`
    timed steps, all host threads this process may use."""
    import torch
    from oracle import torch_ref as tr
    from voxurf_amd import scene
    torch.set_num_threads(threads)
    st = tr.make_state(cfg)
    o, d, v = scene.rays(cfg.n_rays, seed=cfg.seed)
    tg = scene.targets(cfg.n_rays, seed=cfg.seed)
    opt = {}
    tr.train_step(st, opt, o, d, v, tg, cfg, 1)  # warm-up (allocates optimiser state)
    times = []
    for i in range(steps):
        t0 = time.perf_counter()
        tr.train_step(st, opt, o, d, v, tg, cfg, 2 + i)
        times.append(time.perf_counter() - t0)
    times.sort()
    dt = times[len(times) // 2]
    return dict(value=cfg.n_rays / dt, unit="rays/s", cores=threads, kind="port",
                cpu_model=cpu_model(), host_cpus_visible=os.cpu_count(),
                sample=f"full fine steps (8192 rays, 256^3 grids, fwd+bwd+Adam) of the "
                       f"PyTorch-CPU restatement of the reference step: median of {steps} "
                       f"after 1 warm-up ({', '.join(f'{t:.2f}' for t in times)} s), "
                       f"{threads} threads")


# The roofline kernel: the rgbnet 192 x 192 hidden layers' weight gradient
# (k_mlp_wgrad<6, false>, FP32 MFMA), the largest share of kernel time in the step's
# rocprofv3 kernel trace.
ROOF_KEY = "wgrad192"

# Algorithmic bytes (or FLOPs) per unit of each timed kernel, and the unit's count key:
# SURVEY's per-sample / per-element figures (C feature channels, pages of P elements).
def _kernel_units(cfg, c):
    C = cfg.feat_dim
    from voxurf_amd import _lib
    P = int(_lib.lib().vx_adam_page_elems())
    return {
        "fused_fwd": ("hbm", 224.0 * c["m0_processed"], "224 B (7 trilinear lookups x 8 corners x "
                      "4 B) per processed sample"),
        "gather": ("hbm", 8.0 * C * 4 * c["m2"], f"{8 * C * 4} B (8 corners x {C} channels x 4 B) "
                   "per survivor"),
        "feat_bwd": ("hbm", 8.0 * C * 8 * c["m2"], f"{8 * C * 8} B (8 corners x {C} channels, "
                     "read + write) per survivor"),
        "fused_bwd": ("hbm", 448.0 * c["m1b"], "448 B (7 x 8 corners, read + write) per "
                      "walk-range sample; phase 2 of the SDF backward (stencil adjoints and "
                      "the brick scatter), on the main stream"),
        "bwd_alpha": ("hbm", 52.0 * c["m1b"], "52 B (the slot's two float4 read, its "
                      "adjoints and bricks written) per walk-range sample; phase 1 of the SDF "
                      "backward (alpha adjoints, brick binning), beside the rgbnet backward"),
        "adam_k0_phase1": ("hbm", 24.0 * P * c.get("k0_swept_pages", 0), "24 B (p, m, v read "
                           "and written) per element of the swept zero-gradient pages"),
        "adam_k0_phase2": ("hbm", 32.0 * P * c.get("k0_live_pages", 0), "32 B (p, g, m, v read; "
                           "p, m, v written; g cleared) per element of the flagged pages"),
        "adam_sdf": ("hbm", 32.0 * P * c.get("sdf_live_pages", 0), "32 B per element of the "
                     "flagged SDF pages (phase 2)"),
        "layer192_fwd": ("mfma", 2.0 * 192 * 192 * c["m2"], "2 x 192 x 192 FLOP per survivor row"),
        "wgrad192": ("mfma", 2.0 * 192 * 192 * c["m2"], "2 x 192 x 192 FLOP per survivor row"),
    }


def roofline_of(trainer, events, rows):
    """The roofline object of the hidden layers' weight-gradient kernel from its in-step
    launches (two per step): the device wall-clock span of each launch's row-block pass
    (first workgroup start to last workgroup end, the span a kernel trace reports), and
    the HIP events around it on its stream, which also count the wait for CUs that the
    kernels of the other streams hold; and the steps' survivor rows."""
    launches = sum(k for _, _, k in events)
    ev_us = 1e3 * sum(a.elapsed_time(b) for a, b, _ in events) / launches
    dur = events.durations_us() if hasattr(events, "durations_us") else []
    us = sum(dur) / len(dur) if dur else ev_us
    flops = 2.0 * 192 * 192 * sum(rows) / len(rows)
    tf = flops / (us * 1e-6) / 1e12
    prec = trainer.mlp_prec
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "rgbnet_wgrad_traffic.json")
    if os.path.exists(tpath):
        with open(tpath) as f:
            traffic = json.load(f)["hbm_bytes_per_launch"]
    kernel = {
        0: "k_mlp_wgrad<6, false>: FP32 MFMAs (v_mfma_f32_32x32x2f32)",
        1: "k_mlp_wgrad<6, true>: BF16 activations, FP32 MFMAs",
        2: "k_mlp_wgrad_split<6>: FP32 accuracy from three-way BF16 splits of both operands, "
           "six v_mfma_f32_32x32x16_bf16 per 16-deep step",
    }[prec]
    out = {"bound": "mfma",
           "kernel": kernel + "; rgbnet 192x192 hidden-layer weight gradient dW = dY^T X over "
                              "the step's survivor rows",
           "us_per_launch": us, "events_us_per_launch": ev_us, "launches_timed": launches,
           "algorithmic_flops": flops, "achieved": tf, "peak": PEAK_FP32_MFMA_TF,
           "unit": "TFLOP/s", "frac": tf / PEAK_FP32_MFMA_TF, "traffic": traffic,
           "timing": ("device wall-clock span of each launch of the row-block pass (its "
                      "reduction excluded) over the timed steps, with the other streams' "
                      "kernels running beside it; events_us_per_launch: HIP events around the "
                      "same launches on their stream") if dur else
                     "HIP events on the weight-gradient stream around each launch of the "
                     "row-block pass (its reduction excluded), over the timed steps"}
    if prec == 2:
        # the BF16 matrix-core work it issues: six BF16 products per FP32 product
        out["bf16_instruction_frac"] = 6 * tf / PEAK_BF16_MFMA_TF
    return out


def kernel_table(trainer, cfg, run_step, n_steps):
    """Untimed steps with every listed kernel timed by HIP events on its stream; returns
    per kernel the average duration, algorithmic bytes (FLOPs) per launch and the achieved
    rate against the HBM (FP32 matrix) peak.  The rgbnet weight gradients run in stream
    order in these steps (on the main stream, not beside the SDF backward and the next
    forward), so their figures are those of the kernel alone; the k0 Adam halves stay on
    the second stream as in the timed steps."""
    import torch
    keys = ["fused_fwd", "gather", "feat_bwd", "bwd_alpha", "fused_bwd", "adam_k0_phase1",
            "adam_k0_phase2", "adam_sdf", "layer192_fwd", "wgrad192"]
    acc = {k: [0.0, 0.0, 0] for k in keys}
    desc = {}
    overlap_wgrad = trainer.overlap_wgrad
    trainer.overlap_wgrad = False
    from voxurf_amd.mlp_hip import LaunchTiming
    for i in range(n_steps):
        trainer.kernel_timing = {k: [] for k in keys}
        trainer.kernel_timing[ROOF_KEY] = LaunchTiming(trainer.dev, 8)
        run_step(i)
        trainer.wait_pending()
        c = trainer.step_counts(cfg.n_rays)
        units = _kernel_units(cfg, c)
        for k in keys:
            tl = trainer.kernel_timing[k]
            # the weight-gradient pass: its device wall-clock spans when it has them
            dur = tl.durations_us() if hasattr(tl, "durations_us") else []
            if dur:
                acc[k][0] += sum(dur) * 1e-3
            for e0, e1, n in tl:
                if not dur:
                    acc[k][0] += e0.elapsed_time(e1)
                acc[k][1] += units[k][1] * n
                acc[k][2] += n
            desc[k] = units[k][2]
    trainer.kernel_timing = None
    trainer.overlap_wgrad = overlap_wgrad
    out = {}
    for k in keys:
        ms, work, n = acc[k]
        if n == 0:
            continue
        bound = _kernel_units(cfg, {"m0_processed": 0, "m2": 0, "m1b": 0})[k][0]
        rate = work / (ms * 1e-3)
        if bound == "hbm":
            out[k] = {"bound": "hbm", "us": 1e3 * ms / n, "bytes_per_launch": work / n,
                      "GBs": rate / 1e9, "frac": rate / 1e9 / PEAK_HBM_GBS, "unit": desc[k]}
        else:
            out[k] = {"bound": "mfma", "us": 1e3 * ms / n, "flops_per_launch": work / n,
                      "TFs": rate / 1e12, "frac": rate / 1e12 / PEAK_FP32_MFMA_TF, "unit": desc[k]}
    return out


def serving_summary(n_req, rate):
    """The render server on 4 resident 256^3 scenes at a saturating Poisson load:
    p50/p99 latency and rays/s of continuous batching against sequential per-request
    rendering in 8192-ray chunks (run.py:123-126), and whether every result is identical."""
    import types
    import studies
    r = studies.serve(types.SimpleNamespace(requests=n_req, rate=rate))
    b, q = r["continuous_batching"], r["sequential_8192_chunks"]
    return {"requests": n_req, "rate_per_s": rate, "total_rays": r["total_rays"],
            "batched": {k: b[k] for k in ("p50_ms", "p99_ms", "rays_per_s")},
            "sequential": {k: q[k] for k in ("p50_ms", "p99_ms", "rays_per_s")},
            "throughput_ratio": b["rays_per_s"] / q["rays_per_s"],
            "identical_results": r["identical_results"], "workload": r["config"]["workload"]}


def _stage(what):
    """One progress line on stderr (stdout carries only the result line)."""
    print(f"bench: {what}", file=sys.stderr, flush=True)


def kernel_sources():
    """Hash of the sources of the step's kernels, by which counters measured on them are told from
    older ones."""
    import hashlib
    h = hashlib.sha256()
    for name in ("common.h", "fine.h", "voxel.h", "fused.hip", "mlp.hip", "optim.hip",
                 "render_utils.hip"):
        with open(os.path.join(ROOT, "voxurf_amd", "csrc", name), "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build measures one GPU; --gpus must be 1 "
                                   "(multi-GPU sharding is a design note only)"}))
        sys.exit(2)
    if args.mode != "train":
        import studies
        res = getattr(studies, args.mode)(args)
        print(json.dumps(res))
        return
    import torch
    from voxurf_amd import scene
    from voxurf_amd.fused import FusedFineTrainer
    from voxurf_amd.model import Trainer, VoxurfFine

    _stage("scene and trainer")
    cfg = scene.FINE
    if args.rays != cfg.n_rays:
        import dataclasses
        cfg = dataclasses.replace(cfg, n_rays=args.rays)
    dev = torch.device("cuda:0")
    mlp_dtype = torch.bfloat16 if args.mlp == "bf16" else torch.float32

    n_pool = 16
    pool = []
    for i in range(n_pool):
        o, d, v = scene.rays(cfg.n_rays, seed=100 + i)
        pool.append((o.to(dev), d.to(dev), v.to(dev), scene.targets(cfg.n_rays, seed=100 + i).to(dev)))

    sdf = scene.sdf_grid(cfg.R).to(dev)
    k0 = scene.feature_grid(cfg.R, cfg.feat_dim).to(dev)
    mlp = scene.mlp_params(cfg.mlp_in, cfg.mlp_width, cfg.mlp_depth)
    if args.path == "fused":
        trainer = FusedFineTrainer(cfg, sdf, k0, mlp, device=dev, mlp_dtype=mlp_dtype)
        trainer.overlap_adam = not args.serial_adam
        trainer.overlap_wgrad = not args.serial_wgrad
        trainer.overlap_sdf_bwd = {None: False, "rgbnet": True,
                                   "scatter": "scatter"}[args.overlap_sdf_bwd]
        trainer.bounds_ahead = not args.bounds_now
        trainer.bounds_behind_walk = not args.bounds_at_start
        if args.wgrad_blocks is not None:
            trainer.wgrad_blocks = args.wgrad_blocks
        trainer.rgbnet.f32_split = args.mlp != "fp32-mfma"
    else:
        model = VoxurfFine(cfg, sdf, k0, mlp, mlp_dtype=mlp_dtype).to(dev)
        model.rgbnet.f32_split = args.mlp != "fp32-mfma"
        trainer = Trainer(model, cfg)
    del sdf, k0

    def run(i, **kw):
        o, d, v, t = pool[i % n_pool]
        return trainer.step(o, d, v, t, **kw)

    if args.path == "fused" and args.prime > 0:
        for b0 in range(0, args.prime, 16):
            batches = []
            for s in range(b0, min(args.prime, b0 + 16)):
                o, d, v = scene.rays(cfg.n_rays, seed=10000 + s)
                batches.append((o.to(dev), d.to(dev), v.to(dev)))
            trainer.prime_touched(batches)
    if args.path == "fused":
        # the timed batches' own walk ranges size the slots before the timed region (a
        # step whose walk ranges overflow the slots walks again with larger ones)
        trainer.prime_touched([b[:3] for b in pool])
    fused = args.path == "fused"
    if fused:
        # the roofline kernel's launches are timed on their own stream (two event records
        # per step, on the third stream); the warm-up steps run the same code
        trainer.kernel_timing = {ROOF_KEY: []}
    # The objects created so far (torch's modules, the scene, the trainer) leave the
    # collector's generations: a full collection over them takes tens of milliseconds of
    # host time, which would otherwise land inside a short timed region now and then.
    # Done before the warm-up steps: the GPU idles meanwhile and its clocks drop, and the
    # warm-up steps, not the timed ones, then bring them back up.
    gc.collect()
    gc.freeze()
    _stage(f"{args.warmup} warm-up steps")
    for i in range(args.warmup):
        run(i)
    torch.cuda.synchronize()
    _stage(f"{args.steps} timed steps")
    if fused:
        from voxurf_amd.mlp_hip import LaunchTiming
        trainer.kernel_timing = {ROOF_KEY: LaunchTiming(dev, 4 * args.steps + 8)}
    rows = []
    stream = torch.cuda.current_stream()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps + 1)]
    retries0 = dict(trainer.retries) if fused else None
    host_s = []
    wait0 = trainer.host_wait_s if fused else 0.0
    t0 = time.perf_counter()
    ev[0].record(stream)
    for i in range(args.steps):
        th = time.perf_counter()
        run(args.warmup + i)
        host_s.append(time.perf_counter() - th)
        if fused:
            rows.append(trainer.m)
        if i == args.steps - 1 and fused:
            # the last step's k0 update (second stream) and rgbnet weight gradients and
            # Adam pass (third stream) may still be running: the timed region ends when
            # every one of them has finished
            trainer.wait_pending()
        ev[i + 1].record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    per = [ev[i].elapsed_time(ev[i + 1]) for i in range(args.steps)]
    slowest = sorted(range(args.steps), key=lambda i: -per[i])[:3]
    slowest = [[i, per[i]] for i in slowest]
    retries = None if not fused else {k: trainer.retries[k] - retries0[k] for k in retries0}
    per.sort()
    ms = sum(per) / len(per)

    roofline = kernels = None
    if fused:
        roofline = roofline_of(trainer, trainer.kernel_timing[ROOF_KEY], rows)
        trainer.kernel_timing = None
        if args.kernel_steps > 0:
            _stage(f"kernel table ({args.kernel_steps} steps)")
            kernels = kernel_table(trainer, cfg, lambda i: run(args.warmup + args.steps + i),
                                   args.kernel_steps)
            # the same kernel alone (weight gradients in stream order)
            if ROOF_KEY in kernels:
                roofline["alone"] = {"us_per_launch": kernels[ROOF_KEY]["us"],
                                     "achieved": kernels[ROOF_KEY]["TFs"],
                                     "frac": kernels[ROOF_KEY]["frac"]}
        counts = trainer.step_counts(cfg.n_rays)
    else:
        run(args.warmup + args.steps, profile=True)
        torch.cuda.synchronize()
        counts = trainer.last_counts
    sb = step_bytes(cfg, counts)
    step_traffic = None
    tpath = os.path.join(ROOT, "profiles", "step_traffic.json")
    if fused and args.mlp == "fp32" and os.path.exists(tpath):
        with open(tpath) as f:
            st = json.load(f)
        step_traffic = {k: st[k] for k in ("hbm_read_bytes_per_step", "hbm_write_bytes_per_step",
                                            "hbm_bytes_per_step", "source")}
        # bytes counted on other kernels than these say nothing about this step time
        current = st.get("kernel_sources") == kernel_sources()
        step_traffic["of_these_kernels"] = current
        rate = st["hbm_bytes_per_step"] / (ms * 1e-3) / 1e9 if current else None
        step_traffic["achieved_GBs"] = rate
        step_traffic["frac"] = rate / PEAK_HBM_GBS if current else None

    res = {
        "metric": "fine train-step rays/s at 256^3",
        "value": cfg.n_rays / (ms * 1e-3),
        "unit": "rays/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "p50_ms": per[len(per) // 2],
        "p99_ms": per[min(len(per) - 1, int(round(0.99 * (len(per) - 1))))],
        # the three slowest timed steps ([index, ms]) and the steps that ran again inside
        # the timed region (walk ranges past the slots, survivors past the row buffers)
        "slowest_steps": slowest,
        "retries_timed": retries,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32 (rgbnet bf16)" if args.mlp == "bf16" else "f32",
        "data": "synthetic (seeded analytic SDF scene, random-init features and rgbnet)",
        "config": {"workload": "plain fine step: 256^3 SDF + 256^3x12 features, rgbnet "
                               "42-192x3-3, 8192 rays, stepsize 0.5, s=256, fwd+bwd+Adam",
                   "rays_per_step": cfg.n_rays, "path": args.path, "mlp": args.mlp},
        "roofline": roofline,
        "kernels": kernels,
        # physical HBM bytes of one step (PMC FETCH_SIZE + WRITE_SIZE over every kernel of
        # a step, calibrated against a copy kernel) over the step time
        "step_traffic": step_traffic,
        # the SURVEY byte formula over the step time: it charges the dense Adam sweep and
        # every in-box sample's lookups, work this path skips exactly (untouched pages,
        # samples past each walk's end), so it is an effective rate, not HBM traffic
        "step_roofline_effective": None if sb is None else {
            "algorithmic_bytes": sb, "achieved_GBs": sb / (ms * 1e-3) / 1e9,
            "frac": sb / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS},
        "samples": counts,
        "k0_pages": None if not fused else {
            "total": trainer.n_pages, "touched": trainer.touched_pages(),
            "primed_batches": args.prime, "sdf_total": trainer.n_sdf_pages,
            "sdf_touched": trainer.sdf_touched_pages()},
        "wall_s": wall,
        # host time per timed step (Python and the launches, and its waits for the survivor
        # count of the step's own walk): when launch time nears ms_per_step the GPU idles
        "host": {"ms_per_step": 1e3 * sum(host_s) / len(host_s),
                 "wait_ms_per_step": 1e3 * ((trainer.host_wait_s if fused else 0.0) - wait0)
                                     / len(host_s)},
    }
    if not args.no_cpu:
        threads = args.cpu_threads or host_cpus()
        _stage(f"CPU baseline ({threads} threads)")
        res["cpu_baseline"] = cpu_baseline(cfg, threads)
    if fused and args.serve_requests > 0:
        del trainer, pool
        torch.cuda.empty_cache()
        _stage(f"serving ({args.serve_requests} requests)")
        res["serving"] = serving_summary(args.serve_requests, args.serve_rate)
    print(json.dumps(res))


if __name__ == "__main__":
    main()
