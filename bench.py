#!/usr/bin/env python3
"""Benchmark of the quaternion Conv2D / Dense hot path on one MI355X.

A step is one pass of the hot path over one batch of synthetic input, resident in HBM: forward,
input gradient and filter gradient of one quaternion operator (or one forward+backward of the
quaternion ResNet-50).  The default run measures every configuration (Dense fp32; 1x1 and 3x3 fp32; the
four fp16 shapes under both fp16 policies; each in both product modes; the ResNet-50) and prints one
full JSON record per configuration as a line of its own (`{"record": ...}`), then -- LAST -- the one
short JSON line of the contract (under 1800 characters): headline (`value`, `roofline`, `cpu_baseline`)
= the largest convolution configuration -- 3x3, fp16 tensors, N=128, 128->128 quaternion channels,
28x28, full16 policy --, `per_config` as workload -> policy -> mode -> [ms per step, TFLOP/s] and `c5`
= the ResNet-50's images/s.  `--workload NAME` runs one configuration alone (used for profiling).

Throughput is real-equivalent: 16 real multiply-adds per quaternion multiply-add whichever product
formulation runs; the factorized (8-product) kernels execute half of them and the kernels on bf16 parts six times as many
(on instructions of sixteen times the rate), which `executed_frac` reports next to the real-equivalent `frac`.
"""
import argparse
import ctypes
import json
import os
import re
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "quaternion conv TFLOP/s (real-equiv, % MFMA peak) + q-ResNet-50 fwd+bwd img/s"
PEAK_TFLOPS = {"f32": 157.3, "f16": 2500.0}  # MI355X dense MFMA peaks
PEAK_HBM_GBS = 8000.0

CONVS = {
    # name: (n, ci, co, h, w, k, padding, dtype)
    "c2_pw_f32": (32, 64, 64, 56, 56, 1, "VALID", "f32"),
    "c3_k3_f32": (64, 64, 64, 56, 56, 3, "SAME", "f32"),
    "c4_k3_f16_128_28": (128, 128, 128, 28, 28, 3, "SAME", "f16"),
    "c4_k3_f16_256_14": (128, 256, 256, 14, 14, 3, "SAME", "f16"),
    "c4_pw_f16_128_28": (128, 128, 128, 28, 28, 1, "VALID", "f16"),
    "c4_pw_f16_256_14": (128, 256, 256, 14, 14, 1, "VALID", "f16"),
}
# grouped convolutions (run by name only, not part of the default table): name: (..., groups)
GROUPED = {
    "x_depthwise_k3_f16_128_28": (32, 128, 128, 28, 28, 3, "SAME", "f16", 128),
    "x_depthwise_k3_f16_256_14": (64, 256, 256, 14, 14, 3, "SAME", "f16", 256),
    "x_groups32_k3_f16_128_28": (32, 128, 128, 28, 28, 3, "SAME", "f16", 32),
    # (..., groups, stride, dilation): shapes that run as rewritten problems
    "x_smallbatch_k3_f16_512_7": (1, 512, 512, 7, 7, 3, "SAME", "f16", 1, 1, 1),       # reduction slices
    "x_atrous_k3_d12_f16_512_64_33": (8, 512, 64, 33, 33, 3, "SAME", "f16", 1, 1, 12),  # dilation phases
    "x_stride3_k3_f16_128_28": (32, 128, 128, 28, 28, 3, "SAME", "f16", 1, 3, 1),       # filter gradient by tap classes
    "x_patch_k16_s16_f16_16_192_224": (16, 16, 192, 224, 224, 16, "VALID", "f16", 1, 16, 1),  # patches as channels
}
DENSE = {"c1_dense_f32": (32, 128, 128, "f32")}  # name: (n, in, out, dtype)
RESNET = "c5_qresnet50"  # quaternion ResNet-50 forward+backward, N=64, 224x224, fp16 full16 policy
HEADLINE = "c4_k3_f16_128_28"
PASSES = ("fwd", "bwd_data", "bwd_weights")
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "hbm_traffic.md")


def executed_share(kernel_name):
    """Executed / real-equivalent arithmetic of a kernel: the factorized (8-product) kernels run half the
    multiplications.  The product mode asks for a formulation; where the 16-product kernel is the faster one
    the library runs that in either mode, so the share is read off the kernel that actually ran.  Kernels on three bf16
    parts a value run six products for one."""
    return (0.5 if "_p8_" in kernel_name else 1.0) * (6.0 if on_bf16_parts(kernel_name) else 1.0)


def on_bf16_parts(kernel_name):
    """fp32 passes whose products are made by the bf16 matrix instructions: their roof is those instructions' peak."""
    return "f32mfmax3" in kernel_name or "f32mfmagemm" in kernel_name


def measured_traffic():
    """Counter figures per launch from the rocprofv3 --pmc summaries, keyed by (workload, kernel variant name):
    rows `| workload | kernel | fetched bytes | written bytes | MFMA busy |` of profiles/hbm_traffic.md
    -> {"bytes": fetched + written, "mfma_busy": fraction or None}."""
    table = {}
    num = r"[0-9.e+]+"
    try:
        with open(TRAFFIC_FILE) as f:
            for line in f:
                cells = [c.strip().strip("`") for c in line.strip().strip("|").split("|")]
                if len(cells) in (4, 5) and re.fullmatch(num, cells[2]) and re.fullmatch(num, cells[3]):
                    busy = None
                    if len(cells) == 5 and re.fullmatch(num, cells[4].rstrip(" %")):
                        busy = float(cells[4].rstrip(" %")) / 100.0
                    table[(cells[0], cells[1])] = {"bytes": float(cells[2]) + float(cells[3]), "mfma_busy": busy}
    except OSError:
        pass
    return table


def host_info():
    """What the CPU baselines ran on: CPU model, the threads used, torch's version and its oneDNN."""
    import torch
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        threads = int(os.environ.get("OMP_NUM_THREADS", "0"))
    except ValueError:
        threads = 0
    if threads <= 0:
        threads = min(os.cpu_count() or 1, 16)  # a one-GPU box's share of its host is 16 cores
    return {"cpu_model": model, "threads": threads, "torch": torch.__version__,
            "onednn": bool(torch.backends.mkldnn.is_available())}


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="all", choices=["all"] + sorted(CONVS) + sorted(GROUPED) + sorted(DENSE) + [RESNET])
    ap.add_argument("--mode", type=int, default=0, choices=[0, 8, 16],
                    help="product formulation; 0 = from UPSTRIDE_MEMORY_OPTIMIZED like the reference (default 8)")
    ap.add_argument("--policy", default=None, help="UPSTRIDE_CONV_FP16_POLICY for fp16 workloads (default full16)")
    ap.add_argument("--batch", type=int, default=64, help="images per step of the ResNet workload")
    ap.add_argument("--torch-bn", action="store_true",
                    help="ResNet workload: torch.nn.BatchNorm2d + ReLU (MIOpen) instead of the library's batch-norm kernels")
    ap.add_argument("--pack-in-forward", action="store_true",
                    help="c5_qresnet50: every layer packs its changed filter in its own forward call (on the caller's "
                         "stream) instead of all layers ahead of the forward pass on the second stream")
    ap.add_argument("--frozen-filters", action="store_true",
                    help="ResNet workload: the filters do not change between steps, so no step packs them again")
    ap.add_argument("--no-graph", action="store_true", help="time the eager steps only (no HIP graph replay)")
    ap.add_argument("--channels-last", action="store_true",
                    help="one convolution workload on channels-last activations [4N, H, W, C] (needs --workload)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also launch a plain 256 MiB device copy (untimed), the yardstick for HBM byte counters")
    ap.add_argument("--cpu-seconds", type=float, default=12.0, help="CPU time budget of the cpu_baseline leg")
    return ap.parse_args()


def make_context(mode, policy):
    import phoenix_core_amd as phx
    env = {"UPSTRIDE_CONV_FP16_POLICY": policy}
    if mode == 16:
        env["UPSTRIDE_MEMORY_OPTIMIZED"] = "1"
    return phx.Context(env)


def default_mode(args):
    import phoenix_core_amd as phx
    if args.mode:
        return args.mode
    return 16 if phx.Context().memory_optimized else 8


def _median_time(step, seconds, least, most):
    step()  # warm-up (primitive creation)
    times = []
    t_end = time.perf_counter() + seconds
    while len(times) < least or (time.perf_counter() < t_end and len(times) < most):
        t0 = time.perf_counter()
        step()
        times.append(time.perf_counter() - t0)
    times.sort()
    return times[len(times) // 2], len(times)


def cpu_baseline_conv(cfg, mode, seconds, images=None):
    """The reference's CPU algorithm (lane decomposition + scalar oneDNN convolutions through
    torch's CPU backend) on a bounded sample of the same workload: `images` of its N images."""
    import torch
    import oracle
    from oracle import torch_cpu_path as tcp
    n, ci, co, h, w, k, padding, _ = cfg
    host = host_info()
    torch.set_num_threads(host["threads"])
    n_s = images or max(1, n // 8)
    g = oracle.make_geom(n_s, ci, co, h, w, k, k, 1, 1, padding)
    gen = torch.Generator().manual_seed(0x5EED)
    x = torch.randn(4 * n_s, ci, h, w, generator=gen)
    wt = torch.randn(4, co, ci, k, k, generator=gen) * (2.0 / (ci * k * k)) ** 0.5
    gr = torch.randn(4 * n_s, co, g.ho, g.wo, generator=gen)
    name = "factorized" if mode == 8 else "generic"
    flops = 3 * 2 * 16 * n_s * co * ci * g.ho * g.wo * k * k

    def step():
        tcp.conv2d_fwd(g, x, wt, None, name)
        tcp.conv2d_bwd(g, x, wt, gr, name)

    med, runs = _median_time(step, seconds, 3, 50)
    return {
        "value": flops / med / 1e12, "unit": "TFLOP/s", "cores": host["threads"], "cpu_model": host["cpu_model"],
        "kind": "port",
        "sample": "%d/%d images, fwd+bwd, %s path, torch %s CPU (oneDNN) convs, fp32, "
                  "median of %d" % (n_s, n, name, host["torch"], runs),
        "ms_per_step_sample": med * 1e3,
    }


def cpu_baseline_dense(cfg, mode, seconds):
    """The reference's CPU Dense path (lane decomposition + 8 or 16 scalar matmuls, src/dense.hpp:77-180, 252-377
    over src/backend/onednn/dense.hpp:53-93) with the matmuls by torch's CPU backend, whole workload, all threads;
    the single-threaded C restatement of the same algorithm is timed beside it."""
    import numpy as np
    import torch
    import oracle
    from oracle import torch_cpu_path as tcp
    n, ni, no, _ = cfg
    host = host_info()
    torch.set_num_threads(host["threads"])
    r = np.random.default_rng(0x5EED + 1)
    x = r.standard_normal((4 * n, ni)).astype(np.float32)
    lim = (6.0 / (ni + no)) ** 0.5
    w = r.uniform(-lim, lim, (4, ni, no)).astype(np.float32)
    b = np.zeros((4, no), np.float32)
    gr = r.standard_normal((4 * n, no)).astype(np.float32)
    name = "factorized" if mode == 8 else "generic"
    tx, tw, tb, tg = (torch.from_numpy(a) for a in (x, w, b, gr))

    def step():
        tcp.dense_fwd(tx, tw, tb, name)
        tcp.dense_bwd(tx, tw, tg, name)

    def step_c():
        oracle.dense_fwd(x, w, b, name, dtype=np.float32)
        oracle.dense_bwd(x, w, gr, name, dtype=np.float32)

    med, runs = _median_time(step, min(seconds, 2.0), 5, 500)
    med_c, _ = _median_time(step_c, min(seconds, 1.0), 5, 200)
    flops = 3 * 2.0 * 16 * n * ni * no
    return {"value": flops / med / 1e12, "unit": "TFLOP/s", "cores": host["threads"], "cpu_model": host["cpu_model"],
            "kind": "port",
            "sample": "whole workload, fwd+dgrad+wgrad, %s path, scalar matmuls by torch %s CPU (oneDNN), fp32, "
                      "median of %d" % (name, host["torch"], runs),
            "ms_per_step_sample": med * 1e3,
            "c_restatement_one_thread_ms": med_c * 1e3}


class _Timed:
    """Runs `step` (which makes ncalls library calls) and returns wall-clock milliseconds per step and, per call
    slot, the mean HIP-event duration of its dominant kernel.  Three passes of `steps` steps each: eager without
    the library's event timer (its event records sit between the kernels), eager with it (kernel durations), and --
    where `outputs` is given and graphs are not switched off -- the step replayed from a HIP graph, trusted only if
    every checked replay reproduces the eager outputs bit for bit.  One rule for `ms_per_step`: the verified replay
    where there is one, the eager figure otherwise (both are kept in the record)."""

    def __init__(self, step, ncalls, steps, warmup, outputs=None, use_graph=True):
        import torch
        from phoenix_core_amd import capi
        for _ in range(warmup):
            step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            step()
        torch.cuda.synchronize()
        self.ms_per_step_eager = (time.perf_counter() - t0) / steps * 1e3
        capi.profile_enable(ncalls * steps)
        torch.cuda.synchronize()
        for _ in range(steps):
            step()
        torch.cuda.synchronize()
        ms = capi.profile_collect(ncalls * steps)
        capi.profile_enable(0)
        self.kernel_ms = [sum(ms[i::ncalls]) / max(1, len(ms[i::ncalls])) for i in range(ncalls)]
        self.ms_per_step = self.ms_per_step_eager
        self.graph = {"used": False, "note": "not attempted"}
        if outputs is not None and use_graph:
            self.graph = self._replay(step, steps, warmup, outputs)
            if self.graph["used"]:
                self.ms_per_step = self.graph["ms_per_step"]
            self.graph["reported"] = "hip_graph_replay" if self.graph["used"] else "eager"

    @staticmethod
    def _replay(step, steps, warmup, outputs):
        import torch
        from phoenix_core_amd import capi
        try:
            capi.init()
            want = [t.clone() for t in outputs()]
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                step()
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                step()
            for _ in range(3):
                for t in outputs():
                    t.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                if not all(torch.equal(a, b) for a, b in zip(outputs(), want)):
                    return {"used": False, "note": "a replay did not reproduce the eager outputs"}
                step()  # eager work of the program between the replays
                torch.cuda.synchronize()
            for _ in range(max(warmup, 3)):
                graph.replay()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(steps):
                graph.replay()
            torch.cuda.synchronize()
            return {"used": True, "ms_per_step": (time.perf_counter() - t0) / steps * 1e3, "replays_checked": 3,
                    "note": "every checked replay reproduced the eager outputs bit for bit"}
        except Exception as exc:  # capture is an optimisation: any failure leaves the eager figure standing
            return {"used": False, "note": "capture or replay failed: %s" % (str(exc)[:200],)}


def roofline_of(pass_name, kernel, flops, nbytes, kernel_ms, compute, counters):
    """Roofline record of one kernel launch.  `bound` names the roof that applies by arithmetic
    intensity (algorithmic FLOPs / algorithmic bytes against the ridge peak_flops / peak_bandwidth) and
    `frac` is algorithmic work over that roof.  `regime` is what the counters of the committed rocprofv3
    run of this kernel variant say it is held by: "mfma" when the matrix pipe is busy at least half the
    time, "hbm" when the measured traffic moves at half of peak bandwidth or more, otherwise "issue/latency";
    null when the variant has no counter row."""
    peak = PEAK_TFLOPS["f16" if on_bf16_parts(kernel) else compute]  # (bf16 instructions run at the fp16 rate)
    tflops = flops / (kernel_ms * 1e-3) / 1e12
    gbs = nbytes / (kernel_ms * 1e-3) / 1e9
    share = executed_share(kernel)
    ridge = peak * 1e12 / (PEAK_HBM_GBS * 1e9)
    ai = flops / nbytes
    bound = "hbm" if ai < ridge else "mfma"
    frac_mfma, frac_hbm = tflops / peak, gbs / PEAK_HBM_GBS
    traffic = counters["bytes"] if counters else None
    busy = counters["mfma_busy"] if counters else None
    out = {"bound": bound, "pass": pass_name, "kernel": kernel, "kernel_ms": kernel_ms}
    if bound == "mfma":
        out.update({"achieved": tflops, "peak": peak, "unit": "TFLOP/s", "frac": frac_mfma})
    else:
        out.update({"achieved": gbs, "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": frac_hbm})
    regime = None
    if counters:
        traffic_frac = traffic / (kernel_ms * 1e-3) / 1e9 / PEAK_HBM_GBS
        if busy is not None and busy >= 0.5:
            regime = "mfma"
        elif traffic_frac >= 0.5:
            regime = "hbm"
        elif busy is not None:
            regime = "issue/latency"
    out.update({
        "executed_frac": frac_mfma * share,  # executed FLOPs / MFMA peak (the factorized kernels run half)
        "real_equiv_tflops": tflops, "frac_of_mfma_peak": frac_mfma, "algorithmic_gb_s": gbs, "frac_of_hbm_peak": frac_hbm,
        "arithmetic_intensity": ai, "ridge": ridge, "regime": regime, "mfma_busy": busy,
        "algorithmic_bytes": nbytes, "algorithmic_flops": flops,
        "traffic": traffic,
    })
    if traffic is None:
        out["traffic_note"] = "no rocprofv3 --pmc summary under profiles/ for this kernel variant on this workload"
    return out


def run_conv(name, mode, policy, args, traffic_table):
    """fwd + input gradient + filter gradient of one convolution configuration through the C ABI."""
    import torch
    import phoenix_core_amd as phx
    from phoenix_core_amd import capi
    n, ci, co, h, w, k, padding, dt = (CONVS.get(name) or GROUPED[name])[:8]
    groups = GROUPED[name][8] if name in GROUPED else 1
    stride, dilation = GROUPED[name][9:11] if name in GROUPED and len(GROUPED[name]) > 9 else (1, 1)
    if dt == "f32":
        policy = "fp32"
    ctx = make_context(mode, policy)
    dtype = torch.float32 if dt == "f32" else torch.float16
    dev = torch.device("cuda:0")
    torch.manual_seed(0x5EED + sorted(list(CONVS) + list(GROUPED)).index(name))
    scale = 1.0 if dt == "f32" else 0.5
    cl = bool(getattr(args, "channels_last", False))
    x = (scale * torch.randn((4 * n, h, w, ci) if cl else (4 * n, ci, h, w), device=dev)).to(dtype)
    wt = (scale * torch.randn(4, co, ci // groups, k, k, device=dev) * (2.0 / (ci // groups * k * k)) ** 0.5).to(dtype)
    desc = phx.Conv2DDescriptor(x.shape, wt.shape, stride, dilation, padding, groups=groups, dtype=dtype, context=ctx,
                                data_format="NHWC" if cl else "NCHW")
    gr = (scale * torch.randn(desc.output_shape, device=dev)).to(dtype)
    ho, wo = desc.output_shape[1:3] if cl else desc.output_shape[2:]
    y = torch.empty(desc.output_shape, dtype=dtype, device=dev)
    dx = torch.empty_like(x)
    dw = torch.empty_like(wt)
    L = capi.lib()
    sizes = [desc.workspace_bytes(p) for p in (capi.PHX_PASS_FWD, capi.PHX_PASS_BWD_DATA, capi.PHX_PASS_BWD_WEIGHTS)]
    ws = torch.empty(max(sizes + [1]), dtype=torch.uint8, device=dev)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    d = ctypes.byref(desc.c)
    names = {}

    def step():
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)  # (the capture stream during a graph capture)
        capi.check(L.phx_qconv2d_fwd(d, stream, P(x), P(wt), None, P(y), P(ws), sizes[0]), "fwd")
        names.setdefault("fwd", capi.last_kernel_name())
        capi.check(L.phx_qconv2d_bwd_data(d, stream, P(gr), P(wt), P(dx), P(ws), sizes[1]), "bwd_data")
        names.setdefault("bwd_data", capi.last_kernel_name())
        capi.check(L.phx_qconv2d_bwd_weights(d, stream, P(x), P(gr), P(dw), P(ws), sizes[2]), "bwd_weights")
        names.setdefault("bwd_weights", capi.last_kernel_name())

    if args.copy_calibration:
        src = torch.empty(64 << 20, dtype=torch.float32, device=dev).normal_()
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)  # reads 256 MiB, writes 256 MiB
        del src, dst
    t = _Timed(step, 3, args.steps, args.warmup, outputs=lambda: (y, dx, dw), use_graph=not args.no_graph)
    flops_pass = 2.0 * 16 * n * co * (ci // groups) * ho * wo * k * k
    esize = 4 if dt == "f32" else 2
    # algorithmic bytes of a pass: read the activations (or the gradient), read the filters, write the result
    bytes_pass = {
        "fwd": esize * (x.numel() + wt.numel() + y.numel()),
        "bwd_data": esize * (gr.numel() + wt.numel() + dx.numel()),
        "bwd_weights": esize * (x.numel() + gr.numel() + dw.numel()),
    }
    per_pass = dict(zip(PASSES, t.kernel_ms))
    # (fp32 arithmetic on fp16 tensors runs on the fp16 matrix instructions, whose products of fp16 values are exact)
    compute = {p: "f32" if "_f32mfma" in names[p] else dt for p in PASSES}
    roofs = {p: roofline_of(p, names[p], flops_pass, bytes_pass[p], per_pass[p], compute[p],
                            traffic_table.get((name, names[p]))) for p in PASSES}
    dominant = max(per_pass, key=per_pass.get)
    value = 3 * flops_pass / (t.ms_per_step * 1e-3) / 1e12
    del x, wt, gr, y, dx, dw, ws
    torch.cuda.empty_cache()
    return {
        "workload": "%s: quaternion conv %dx%d stride %d%s, N=%d (4N=%d rows), %d->%d q-channels%s, %dx%d, "
                    "fwd+input-grad+filter-grad%s" % (name, k, k, stride, " dilation %d" % dilation if dilation > 1 else "", n, 4 * n, ci, co,
                                                      " in %d groups" % groups if groups > 1 else "", h, w,
                                                      ", channels-last activations" if cl else ""),
        "data_format": "NHWC" if cl else "NCHW",
        "n": n, "product_mode": mode, "fp16_policy": policy, "padding": padding, "dtype": dt,
        "value": value, "unit": "TFLOP/s", "ms_per_step": t.ms_per_step, "ms_per_step_eager": t.ms_per_step_eager,
        "hip_graph": t.graph, "images_per_s": n / (t.ms_per_step * 1e-3),
        "kernel_ms": per_pass, "kernels": names,
        "real_equiv_tflops": {p: roofs[p]["real_equiv_tflops"] for p in PASSES},
        "frac_of_mfma_peak": {p: roofs[p]["frac_of_mfma_peak"] for p in PASSES},
        "executed_frac": {p: roofs[p]["executed_frac"] for p in PASSES},
        "frac_of_hbm_peak": {p: roofs[p]["frac_of_hbm_peak"] for p in PASSES},
        "roofline": roofs[dominant],
        "unprofiled_kernels": sorted({names[p] for p in PASSES if (name, names[p]) not in traffic_table}),
    }


def run_dense(name, mode, args, traffic_table):
    """fwd + input gradient + filter gradient of the Dense configuration through the C ABI."""
    import torch
    import phoenix_core_amd as phx
    from phoenix_core_amd import capi
    n, ni, no, dt = DENSE[name]
    ctx = make_context(mode, "fp32")
    dev = torch.device("cuda:0")
    torch.manual_seed(0x5EED + 1)
    x = torch.randn(4 * n, ni, device=dev)
    lim = (6.0 / (ni + no)) ** 0.5
    wt = torch.empty(4, ni, no, device=dev).uniform_(-lim, lim)
    b = torch.zeros(4, no, device=dev)
    desc = phx.DenseDescriptor(x.shape, wt.shape, use_bias=True, context=ctx)
    gr = torch.randn(desc.output_shape, device=dev)
    y, dx, dw = torch.empty_like(gr), torch.empty_like(x), torch.empty_like(wt)
    L = capi.lib()
    sizes = [desc.workspace_bytes(p) for p in (capi.PHX_PASS_FWD, capi.PHX_PASS_BWD_DATA, capi.PHX_PASS_BWD_WEIGHTS)]
    ws = torch.empty(max(sizes + [1]), dtype=torch.uint8, device=dev)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    d = ctypes.byref(desc.c)
    names = {}

    def step():
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)  # (the capture stream during a graph capture)
        capi.check(L.phx_qdense_fwd(d, stream, P(x), P(wt), P(b), P(y), P(ws), sizes[0]), "fwd")
        names.setdefault("fwd", capi.last_kernel_name())
        capi.check(L.phx_qdense_bwd_data(d, stream, P(gr), P(wt), P(dx), P(ws), sizes[1]), "bwd_data")
        names.setdefault("bwd_data", capi.last_kernel_name())
        capi.check(L.phx_qdense_bwd_weights(d, stream, P(x), P(gr), P(dw), P(ws), sizes[2]), "bwd_weights")
        names.setdefault("bwd_weights", capi.last_kernel_name())

    t = _Timed(step, 3, args.steps, args.warmup, outputs=lambda: (y, dx, dw), use_graph=not args.no_graph)
    flops_pass = 2.0 * 16 * n * ni * no
    bytes_pass = {"fwd": 4 * (x.numel() + wt.numel() + b.numel() + y.numel()),
                  "bwd_data": 4 * (gr.numel() + wt.numel() + dx.numel()),
                  "bwd_weights": 4 * (x.numel() + gr.numel() + dw.numel())}
    per_pass = dict(zip(PASSES, t.kernel_ms))
    roofs = {p: roofline_of(p, names[p], flops_pass, bytes_pass[p], per_pass[p], "f32", traffic_table.get((name, names[p])))
             for p in PASSES}
    dominant = max(per_pass, key=per_pass.get)
    out = {
        "workload": "%s: quaternion Dense, N=%d (4N=%d rows), %d->%d quaternion units, bias, "
                    "fwd+input-grad+filter-grad" % (name, n, 4 * n, ni, no),
        "product_mode": mode, "fp16_policy": "fp32", "dtype": dt,
        "value": 3 * flops_pass / (t.ms_per_step * 1e-3) / 1e12, "unit": "TFLOP/s", "ms_per_step": t.ms_per_step,
        "ms_per_step_eager": t.ms_per_step_eager, "hip_graph": t.graph,
        "kernel_ms": per_pass, "kernels": names,
        "real_equiv_tflops": {p: roofs[p]["real_equiv_tflops"] for p in PASSES},
        "roofline": roofs[dominant],
        "unprofiled_kernels": sorted({names[p] for p in PASSES if (name, names[p]) not in traffic_table}),
        "note": "16.8 MFLOP per pass: a handful of kernel launches of a few microseconds each, launch-latency bound",
    }
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline_dense(DENSE[name], mode, args.cpu_seconds)
    return out


def resnet_flops(n):
    """Real-equivalent forward FLOPs of the 53 convolutions + head (2*16*N*Co*Ci*Ho*Wo*Kh*Kw each)."""
    total, size = 0.0, 224

    def conv(ci, co, k, s, hin):
        ho = (hin + s - 1) // s
        return 2.0 * 16 * n * co * ci * ho * ho * k * k, ho
    f, size = conv(3, 16, 7, 2, size)
    total += f
    size = (size + 1) // 2  # max-pool
    cin = 16
    for width, cout, count, stride in ((16, 64, 3, 1), (32, 128, 4, 2), (64, 256, 6, 2), (128, 512, 3, 2)):
        for i in range(count):
            s = stride if i == 0 else 1
            total += conv(cin, width, 1, 1, size)[0]
            f, out = conv(width, width, 3, s, size)
            total += f + conv(width, cout, 1, 1, out)[0]
            if s != 1 or cin != cout:
                total += conv(cin, cout, 1, s, size)[0]
            size, cin = out, cout
    return total + 2.0 * 16 * n * 250 * 512


def _graphed_step(step, eager_loss, args):
    """The same step captured into a HIP graph (torch.cuda.graph) and replayed: the ~330 kernel launches of a step
    then cost one graph launch.  The capture is trusted only if every one of three checked replays -- with eager
    steps and synchronisations between them -- reproduces the eager loss exactly (the step is deterministic and
    nothing it reads changes between steps); otherwise the eager timing stands."""
    import torch
    from phoenix_core_amd import capi
    try:
        capi.init()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                step()  # sizes the scratch buffer of the capture stream, fills the plan cache
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            graph_loss = step()
        losses = []
        for _ in range(3):
            graph_loss.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            losses.append(float(graph_loss))
            step()  # eager work of the program between the replays
            torch.cuda.synchronize()
        if any(v != eager_loss for v in losses):
            return {"used": False, "note": "replays gave losses %s, the eager step %r" % (losses, eager_loss)}
        for _ in range(max(args.warmup, 3)):
            graph.replay()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            graph.replay()
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) / args.steps * 1e3
        return {"used": True, "ms_per_step": ms, "replays_checked": len(losses),
                "note": "every checked replay reproduced the eager loss exactly"}
    except Exception as exc:  # capture is an optimisation: any failure leaves the eager figure standing
        return {"used": False, "note": "capture or replay failed: %s" % (str(exc)[:200],)}


def run_resnet(mode, policy, args):
    import torch
    import phoenix_core_amd as phx
    ctx = make_context(mode, policy)
    n = args.batch
    dev = torch.device("cuda:0")
    torch.manual_seed(0x5EED + 5)
    model = phx.QResNet50(1000, dtype=torch.float16, context=ctx, fused_bn=not args.torch_bn).to(dev).train()
    images = torch.randn(n, 3, 224, 224, device=dev).half()
    labels = torch.randint(0, 1000, (n,), device=dev)
    last = {}

    convs = [m for m in model.modules() if isinstance(m, phx.QConv2d)]

    def step():
        model.zero_grad(set_to_none=True)
        packed = None
        if not args.frozen_filters:
            # a training step follows an optimizer update: every layer packs its filter anew (once, for the forward
            # pass and the input gradient together); with frozen filters the packed images of the first step stay valid
            for m in convs:
                m.invalidate_packed_filters()
            if not args.pack_in_forward:
                # ... all of them here, on the library's second stream, instead of each in front of its convolution
                packed = phx.repack_filters(model)
        loss = torch.nn.functional.cross_entropy(model(images).float(), labels)
        loss.backward()
        if packed is not None:
            torch.cuda.current_stream().wait_event(packed)
        return loss.detach()

    t = _Timed(lambda: last.__setitem__("loss", step()), 3 * 54, args.steps, max(args.warmup, 3))
    eager_ms, eager_loss = t.ms_per_step, float(last["loss"])
    graph = _graphed_step(step, eager_loss, args) if not args.no_graph else {"used": False, "note": "--no-graph"}
    ms_per_step = graph["ms_per_step"] if graph["used"] else eager_ms
    fwd_flops = resnet_flops(n)
    out = {
        "workload": "%s: quaternion ResNet-50 forward+backward (no optimizer step, as the metric names), "
                    "N=%d real images (4N=%d quaternion rows after the real-input stem), 224x224, 53 quaternion convs + "
                    "quaternion dense head; batch-norm (with the ReLU behind it) and the stem's max-pool by %s, residual add, "
                    "average pool and cross-entropy by PyTorch; the step %s"
                    % (RESNET, n, 4 * n, "torch.nn.BatchNorm2d (MIOpen) and torch.nn.MaxPool2d" if args.torch_bn else
                       "the library's streaming kernels (include/phx_bn.h, include/phx_pool.h)",
                       "is captured once into a HIP graph and replayed" if graph["used"] else "runs eagerly"),
        "product_mode": mode, "fp16_policy": policy, "batch_norm": "torch" if args.torch_bn else "library", "dtype": "f16",
        "filters": "frozen (packed once, before the timed steps)" if args.frozen_filters else
                   "packed once per step and layer, for the forward pass and the input gradient together, " +
                   ("by each layer in its forward call" if args.pack_in_forward else
                    "all at the top of the step on the library's second stream"),
        "value": n / (ms_per_step * 1e-3), "unit": "img/s", "images_per_s": n / (ms_per_step * 1e-3),
        "ms_per_step": ms_per_step, "ms_per_step_eager": eager_ms, "images_per_s_eager": n / (eager_ms * 1e-3),
        "hip_graph": graph,
        "real_equiv_tflops": 3 * fwd_flops / (ms_per_step * 1e-3) / 1e12,
        "frac_of_mfma_peak": 3 * fwd_flops / (ms_per_step * 1e-3) / 1e12 / PEAK_TFLOPS["f16"],
        "quaternion_kernel_ms_per_step": sum(t.kernel_ms), "loss": eager_loss,
    }
    del model, images, labels, last
    torch.cuda.empty_cache()
    return out


def sig(v, digits=4):
    """Floats rounded to `digits` significant digits, recursively (the contract's line has to stay short)."""
    if isinstance(v, float):
        if v != v or abs(v) == float("inf"):
            return None
        r = float("%.*g" % (digits, v))
        return int(r) if abs(r) >= 10 ** (digits - 1) else r  # (no digits behind the point are significant there)
    if isinstance(v, dict):
        return {k: sig(x, digits) for k, x in v.items()}
    if isinstance(v, (list, tuple)):
        return [sig(x, digits) for x in v]
    return v


LINE_LIMIT = 1800  # characters; the driver keeps the last 2000 of the output for parsing


def line(head, args, extra=None):
    """The contract's JSON line around one workload record: the keys the contract names, a trimmed `roofline`
    and `cpu_baseline`, and whatever short `extra` the caller adds; the full record goes out on a line before it."""
    out = {
        "metric": METRIC, "value": head["value"], "unit": head["unit"], "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": head["ms_per_step"], "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": head["dtype"], "data": "synthetic",
        "config": {k: head[k] for k in ("workload", "product_mode", "fp16_policy", "padding", "batch_norm") if k in head},
    }
    out["config"]["workload"] = out["config"]["workload"].split(", fwd+")[0].replace(" (4N=%d rows)" % (4 * head.get("n", 0)), "")[:120]
    if "roofline" in head:
        keep = ("bound", "pass", "kernel", "kernel_ms", "achieved", "peak", "unit", "frac", "executed_frac",
                "algorithmic_bytes", "traffic", "regime")
        out["roofline"] = {k: head["roofline"].get(k) for k in keep}
    if "cpu_baseline" in head:
        keep = ("value", "unit", "cores", "cpu_model", "kind", "sample", "ms_per_step_sample")
        out["cpu_baseline"] = {k: head["cpu_baseline"].get(k) for k in keep}
        out["cpu_baseline"]["cpu_model"] = str(out["cpu_baseline"]["cpu_model"])[:40]
    if extra:
        out.update(extra)
    out = sig(out)
    text = json.dumps(out, separators=(",", ":"))
    if len(text) > LINE_LIMIT and "per_config" in out:  # keep the headline parseable whatever the table's size
        out["per_config"] = sig(out["per_config"], 2)
        text = json.dumps(out, separators=(",", ":"))
        if len(text) > LINE_LIMIT:
            out["per_config"] = "see the record lines above"
            text = json.dumps(out, separators=(",", ":"))
    return text


def emit(record, name, key=None):
    """One full record as a line of its own, ahead of the contract's line."""
    print(json.dumps({"record": name if key is None else "%s/%s" % (name, key), **sig(record, 6)}), flush=True)


def main():
    args = parse()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path (--gpus %d refused)" % args.gpus,
              file=sys.stderr)
        return 2
    if args.channels_last and args.workload not in CONVS:
        print("--channels-last takes one convolution workload (--workload c2_.. / c3_.. / c4_..)", file=sys.stderr)
        return 2
    import phoenix_core_amd  # noqa: F401  (fails loudly when the HIP library is missing)
    mode = default_mode(args)
    policy = args.policy or "full16"
    traffic = measured_traffic()

    if args.workload == RESNET:
        head = run_resnet(mode, policy, args)
        emit(head, RESNET)
        print(line(head, args, {"c5": {"images_per_s": head["images_per_s"], "ms_per_step": head["ms_per_step"]}}))
        return 0
    if args.workload in DENSE:
        head = run_dense(args.workload, mode, args, traffic)
        emit(head, args.workload)
        print(line(head, args))
        return 0
    if args.workload in CONVS or args.workload in GROUPED:
        head = run_conv(args.workload, mode, policy, args, traffic)
        if not args.no_cpu_baseline and args.workload in CONVS:  # (the CPU restatement has no grouped form)
            head["cpu_baseline"] = cpu_baseline_conv(CONVS[args.workload], mode, args.cpu_seconds)
        emit(head, args.workload)
        print(line(head, args))
        return 0

    # default: every configuration as a record line of its own, the headline's short line last
    short, stale = {}, set()

    def note(name, pol, m, rec):
        emit(rec, name, "%s_mode%d" % (pol, m))
        short.setdefault(name, {}).setdefault(pol, {})[str(m)] = sig([rec["ms_per_step"], rec["value"]], 3)
        stale.update("%s:%s" % (name, k) for k in rec.get("unprofiled_kernels", ()))

    sampled = {"c4_pw_f16_128_28": 4, "c2_pw_f32": 8, "c3_k3_f32": 4}  # images of the 1-2 s CPU samples
    c5 = {}
    for m in (mode, 24 - mode):
        c5[m] = run_resnet(m, "full16", args)
        emit(c5[m], RESNET, "full16_mode%d" % m)
    for name in sorted(DENSE):
        for m in (8, 16):
            note(name, "fp32", m, run_dense(name, m, args, traffic))
    # the longest-running records last: the tail of the output is what a log keeps
    order = [n for n in sorted(CONVS) if "pw" in n and CONVS[n][7] == "f16"] + \
            [n for n in sorted(CONVS) if "k3" in n and CONVS[n][7] == "f16"] + \
            [n for n in sorted(CONVS) if CONVS[n][7] == "f32"]
    head = None
    for pol_pick in ("full16", "backward32", "fp32"):
        for name in order:
            if (CONVS[name][7] == "f32") != (pol_pick == "fp32"):
                continue
            for m in (8, 16):
                rec = run_conv(name, m, pol_pick, args, traffic)
                if name in sampled and m == mode and pol_pick in ("full16", "fp32") and not args.no_cpu_baseline:
                    rec["cpu_baseline"] = cpu_baseline_conv(CONVS[name], m, 1.5, images=sampled[name])
                if name == HEADLINE and m == mode and pol_pick == policy:
                    head = rec
                    if not args.no_cpu_baseline:
                        head["cpu_baseline"] = cpu_baseline_conv(CONVS[HEADLINE], mode, args.cpu_seconds)
                note(name, pol_pick, m, rec)
    if head is None:  # a policy outside the table was asked for
        head = run_conv(HEADLINE, mode, policy, args, traffic)
        if not args.no_cpu_baseline:
            head["cpu_baseline"] = cpu_baseline_conv(CONVS[HEADLINE], mode, args.cpu_seconds)
        emit(head, HEADLINE, "%s_mode%d" % (policy, mode))
    print(json.dumps({"record": "stale_profiles", "note": "kernel variants that ran without a row in "
                      "profiles/hbm_traffic.md", "kernels": sorted(stale)}), flush=True)
    extra = {"c5": {"images_per_s": c5[mode]["images_per_s"], "ms_per_step": c5[mode]["ms_per_step"],
                    "images_per_s_other_mode": c5[24 - mode]["images_per_s"]},
             "per_config": short, "stale_profiles": len(stale)}
    print(line(head, args, extra))
    return 0


if __name__ == "__main__":
    sys.exit(main())
