"""Causal self-attention fwd+bwd throughput on one MI355X.

Workload (the headline): one GPT-2 124M training
micro-step's attention, 12 layers, each forward + backward at B=16, T=256,
H=12, head_dim=64, fp32, packed qkv [B, T, 3C]. One "step" runs the 12
forwards in layer order then the 12 backwards in reverse order, through the
C ABI (gpt_amd/libgpt_hip_attn.so), with every input already resident in HBM.

Timing: W warm-up steps, then untimed steps until the GPU has been busy for
--settle-ms (250 ms; its clocks rise over the first ~30 ms of load after
idle, see SETTLE_MS), then exactly K timed steps between two events.

value = algorithmic FLOPs / GPU time, FLOPs = 12 * 7 * B * H * d * T * (T+1)
(QK^T and PV forward; S recompute, dP, dV, dK, dQ backward; causal pairs
including the diagonal; exp and masking not counted).

Also reported:
  kernels       per-kernel average durations and algorithmic TFLOP/s over a
                second pass of the same steps, from the library's launch timer
                (gpt_hip_attn_timing_*: each head_dim-64 kernel launched by
                hipExtLaunchKernelGGL with an event pair that the dispatch's
                own start and end set); kernel_ms_per_step = their sum per
                step (the rest of ms_per_step is the gaps between kernels)
  roofline      the dominant kernel (most GPU time): algorithmic FLOPs per
                launch / its average launch duration, against 157.3 TFLOP/s;
                `traffic` = its measured HBM bytes per launch, read from
                profiles/<kernel>_c3_traffic.json when that file matches the
                kernel (written by --traffic from two rocprofv3 --pmc runs,
                FETCH_SIZE and WRITE_SIZE, each scaled by the same counter's
                reading for a plain device copy of known size)
  cpu_baseline  the reference's own CPUBackend attention (compiled from its
                sources into oracle/_ref, -O3) on a bounded sample of the
                same workload, one thread, on this host

Usage:
  python bench.py [--gpus 1] [--steps K] [--warmup W]       the metric line
  python bench.py --no-cpu --bwd-path 2                     same workload with the fp32-atomic
                                                            dQ backward (for profiling)
  python bench.py --prefix-sweep [--no-cpu]                 BASELINE config 5(b): forward at B=1
                                                            for every prefix T=1..256 (the reference's
                                                            generation loop without a KV cache); one
                                                            JSON line of its own
  python bench.py --configs [--no-cpu]                      BASELINE configs 1, 2, 4 and 5(a): one JSON
                                                            line each (GPU time, TFLOP/s, % peak,
                                                            per-kernel times; CPU baseline on 1 core
                                                            and on N threads, with the errors of the
                                                            GPU outputs on its sampled (b, h))
  python bench.py --ops [--no-cpu]                          the GPT-2 124M ops around attention
                                                            (gpt_amd/libgpt_hip_ops.so) at the C3
                                                            shapes, each against its roofline; one
                                                            JSON line of its own
  python bench.py --copy-calibration                        256 MiB device copy x5
                                                            (run under --pmc)
  python bench.py --traffic KERNEL FETCH.csv WRITE.csv COPY_FETCH.csv COPY_WRITE.csv
      turns rocprofv3 counter_collection CSVs into profiles/KERNEL_c3_traffic.json
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "causal attn fwd+bwd TFLOP/s & % fp32 MFMA peak, GPT-2 124M shape, 1 GPU"
PEAK_FP32_MFMA_TFLOPS = 157.3
LAYERS, B, T, C, H = 12, 16, 256, 768, 12
D_HEAD = C // H
CONFIG_SEED = 1237  # 1234 + config index 3
# The GPU's clocks rise over the first ~30 ms of sustained load after idle:
# in a kernel trace of this workload the fused backward takes 60.9 us per
# launch over the first 5 steps and 52.3 us from step 30 on, the forward
# 28.5 -> 24.2 us. The timed steps start once the GPU has been busy this long.
SETTLE_MS = 250.0


def settle(step, ms):
    """Runs `step` untimed, in groups of 5 with a synchronize after each,
    until `ms` milliseconds have passed; returns (steps run, ms taken)."""
    import torch

    t0 = time.perf_counter()
    n = 0
    while (time.perf_counter() - t0) * 1e3 < ms:
        for _ in range(5):
            step()
        n += 5
        torch.cuda.synchronize()
    return n, (time.perf_counter() - t0) * 1e3


def attn_flops(b, t, h, d, fwd=True, bwd=True):
    pairs = b * h * d * t * (t + 1)
    return (2 * pairs if fwd else 0) + (5 * pairs if bwd else 0)


# Algorithmic FLOPs of one launch of each head_dim-64 kernel, in units of
# B*H*d*T(T+1) (= 2 FLOPs x d per causal pair): forward QK^T + PV = 2;
# two-launch backward: dK/dV kernel S + dP + dV + dK = 4, dQ kernel dS K = 1;
# fused backward (T <= 256, one launch) all five = 5. The D-row kernel does no
# matrix work (bandwidth-bound: reads dO and O).
KERNEL_FLOP_UNITS = {"fwd": 2, "bwd_dkdv": 4, "bwd_dq": 1, "bwd_fused": 5, "bwd_rowdot": 0}
KERNEL_SYMBOL = {"fwd": "fwd_qs_d64_kernel", "bwd_dkdv": "bwd_dkdv_d64_kernel", "bwd_dq": "bwd_dq_d64_kernel",
                 "bwd_fused": "bwd_fused_d64_kernel", "bwd_rowdot": "bwd_rowdot_d64_kernel"}
COPY_BYTES = 256 << 20


def copy_calibration():
    """A plain device-to-device copy of COPY_BYTES, five times (for --pmc runs)."""
    import torch

    x = torch.ones(COPY_BYTES // 4, device="cuda")
    y = torch.empty_like(x)
    for _ in range(5):
        y.copy_(x)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes": COPY_BYTES, "launches": 5}))


def _counter_per_dispatch(path, counter, kernel_substr):
    import csv

    vals = [float(r["Counter_Value"]) for r in csv.DictReader(open(path))
            if r["Counter_Name"] == counter and kernel_substr in r["Kernel_Name"]]
    if not vals:
        names = sorted({r["Kernel_Name"] for r in csv.DictReader(open(path))})
        raise SystemExit(f"{path}: no {counter} rows for kernels matching {kernel_substr!r}; kernels: {names}")
    return sum(vals) / len(vals), len(vals)


def write_traffic(kernel, fetch_csv, write_csv, copy_fetch_csv, copy_write_csv):
    """HBM bytes per launch of `kernel` from FETCH_SIZE / WRITE_SIZE (KiB per
    dispatch), each scaled by expected / measured for the copy kernel."""
    sym = KERNEL_SYMBOL[kernel]
    f_kib, nf = _counter_per_dispatch(fetch_csv, "FETCH_SIZE", sym)
    w_kib, nw = _counter_per_dispatch(write_csv, "WRITE_SIZE", sym)
    cf_kib, _ = _counter_per_dispatch(copy_fetch_csv, "FETCH_SIZE", "copy")
    cw_kib, _ = _counter_per_dispatch(copy_write_csv, "WRITE_SIZE", "copy")
    f_scale = COPY_BYTES / (cf_kib * 1024)
    w_scale = COPY_BYTES / (cw_kib * 1024)
    fetch = f_kib * 1024 * f_scale
    write = w_kib * 1024 * w_scale
    out = {"kernel": sym, "workload": "one C3 layer: B=16 T=256 H=12 d=64",
           "fetch_bytes_per_launch": round(fetch), "write_bytes_per_launch": round(write),
           "hbm_bytes_per_launch": round(fetch + write),
           "fetch_kib_raw": f_kib, "write_kib_raw": w_kib, "dispatches": [nf, nw],
           "copy_scale": {"fetch": f_scale, "write": w_scale, "copy_bytes": COPY_BYTES}}
    path = os.path.join(ROOT, "profiles", f"{kernel}_c3_traffic.json")
    with open(path, "w") as fh:
        json.dump(out, fh, indent=1)
    print(json.dumps(out))


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--copy-calibration", action="store_true")
    ap.add_argument("--traffic", nargs=5, metavar=("KERNEL", "FETCH", "WRITE", "COPY_FETCH", "COPY_WRITE"))
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--settle-ms", type=float, default=SETTLE_MS,
                    help="after the warm-up steps, keep running untimed steps until the GPU has been busy "
                         "this long, so that the timed steps run at settled clocks (0: off)")
    ap.add_argument("--cpu-layers", type=int, default=12,
                    help="layers of the workload timed on the CPU baseline sample")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--prefix-sweep", action="store_true",
                    help="time BASELINE config 5(b) (forward, B=1, T=1..256) instead of the headline")
    ap.add_argument("--configs", action="store_true",
                    help="time BASELINE configs 1, 2, 4 and 5(a), one JSON line each")
    ap.add_argument("--only", default="", help="with --configs: a comma-separated subset, e.g. C4,C5a")
    ap.add_argument("--ops", action="store_true",
                    help="time the GPT-2 ops around attention (libgpt_hip_ops.so) instead of the headline")
    ap.add_argument("--bwd-path", type=int, default=0, choices=(0, 2, 3),
                    help="backward variant for profiling (gpt_hip_attn_set_path): 0 default (one fused "
                         "launch at T <= 256), 2 fp32-atomic dQ, 3 two-launch (dK/dV + dS tiles, then dQ)")
    return ap.parse_args()


def cpu_baseline(layers: int):
    """Reference CPUBackend attention fwd+bwd on `layers` layers of the same
    workload (B=16, T=256): once on 1 thread (the reference as written), once
    on N = min(B, 16, cpu_count) threads, one batch element per thread calling
    the unchanged function with B=1 on that element's slice (its batch loop is
    independent per element). value = the N-thread rate; value_1core beside."""
    import threading

    import numpy as np

    from gpt_amd import synth
    from oracle import pyoracle

    impl, kind = ("ref_fast", "reference") if pyoracle.ref_available(fast=True) else ("oracle", "port")
    scales = synth.layer_scales(LAYERS, CONFIG_SEED)
    data = []
    for layer in range(layers):
        seed = CONFIG_SEED + layer
        data.append((synth.qkv(B, T, C, seed, scale=float(scales[layer])), synth.grad_out(B, T, C, seed)))

    def run(x, g):
        y, lse = pyoracle.forward(x, H, impl)
        pyoracle.backward(x, y, lse, g, H, impl)
        assert np.isfinite(y).all()

    t0 = time.perf_counter()
    for x, g in data:
        run(x, g)
    t1 = time.perf_counter() - t0
    n_thr = max(1, min(B, 16, os.cpu_count() or 1))
    t0 = time.perf_counter()
    for x, g in data:
        for b0 in range(0, B, n_thr):
            ths = [threading.Thread(target=run, args=(np.ascontiguousarray(x[b:b + 1]), np.ascontiguousarray(g[b:b + 1])))
                   for b in range(b0, min(B, b0 + n_thr))]
            for th in ths:
                th.start()
            for th in ths:
                th.join()
    tn = time.perf_counter() - t0
    flops = layers * attn_flops(B, T, H, D_HEAD)
    lib = "oracle/_ref/libref_cpu_attn_fast.so, -O3 -march=x86-64-v3" if kind == "reference" else "oracle/liboracle_attn.so"
    return {
        "value": round(flops / tn / 1e12, 6),
        "unit": "TFLOP/s",
        "cores": n_thr,
        "value_1core": round(flops / t1 / 1e12, 6),
        "nproc": os.cpu_count(),
        "cpu_model": _cpu_model(),
        "kind": kind,
        "sample": f"{layers} of the 12 layers (B=16,T=256,H=12,d=64) fwd+bwd: {t1:.2f} s on 1 thread, "
                  f"{tn:.2f} s on {n_thr} threads (one batch element each) ({lib})",
    }


PREFIX_SEED = 1239  # 1234 + config index 5


def prefix_sweep(args):
    """BASELINE config 5(b): y, lse for qkv[:, :T] at B=1, every T in 1..256,
    each prefix its own contiguous [1, T, 3C] tensor (the reference's inference
    loop re-sizes its activations every token, infer.cpp:117, gpt.cpp:399-424).
    value = total forward FLOPs of the sweep / summed GPU time, where each T's
    time is the median of `reps` event-timed calls on resident inputs (each rep
    is queued behind a GPU spin, so the host's launch latency is not timed)."""
    import numpy as np
    import torch

    import gpt_amd
    from gpt_amd import synth

    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()
    Tmax, reps = 256, 7
    x = synth.qkv(1, Tmax, C, PREFIX_SEED)
    xs = [torch.from_numpy(np.ascontiguousarray(x[:, :t])).to(dev) for t in range(1, Tmax + 1)]
    ys = [torch.empty(1, t, C, device=dev) for t in range(1, Tmax + 1)]
    ls = [torch.empty(1, t, H, device=dev) for t in range(1, Tmax + 1)]
    for t in range(1, Tmax + 1):  # warm every shape once
        gpt_amd.device_flash_attention_forward(ys[t - 1], ls[t - 1], xs[t - 1], 1, t, C, H, stream)
    torch.cuda.synchronize()
    ev = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(reps)]
          for _ in range(Tmax)]
    for r in range(reps):
        # queue the rep behind a ~10 ms GPU spin, so the events time the GPU
        # only, not the host's per-call launch latency
        torch.cuda._sleep(20_000_000)
        for t in range(1, Tmax + 1):
            e0, e1 = ev[t - 1][r]
            e0.record(stream)
            gpt_amd.device_flash_attention_forward(ys[t - 1], ls[t - 1], xs[t - 1], 1, t, C, H, stream)
            e1.record(stream)
    # the same timing around a one-element fill kernel: the per-call floor of
    # this method (event packets, dispatch, kernel start-up) on this GPU
    tiny = torch.empty(1, device=dev)
    fl = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(64)]
    torch.cuda._sleep(20_000_000)
    for e0, e1 in fl:
        e0.record(stream)
        tiny.fill_(1.0)
        e1.record(stream)
    torch.cuda.synchronize()
    per_t_us = [float(np.median([a.elapsed_time(b) for a, b in ev[t]])) * 1e3 for t in range(Tmax)]
    floor_us = float(np.median([a.elapsed_time(b) for a, b in fl])) * 1e3
    total_us = sum(per_t_us)
    flops = sum(attn_flops(1, t, H, D_HEAD, bwd=False) for t in range(1, Tmax + 1))
    out = {
        "metric": "causal attn forward prefix sweep TFLOP/s, B=1 T=1..256 (generation without KV cache), 1 GPU",
        "value": round(flops / (total_us * 1e-6) / 1e12, 4),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "higher_is_better": True,
        "dtype": "fp32",
        "data": "synthetic (splitmix64 Box-Muller; Q/K/V ~ N(0,1))",
        "config": {"workload": "BASELINE config 5(b): forward, B=1, every prefix T=1..256, H=12 d=64",
                   "flops": flops, "reps_per_T": reps},
        "sweep_ms": round(total_us / 1e3, 4),
        "us_at_T": {str(t): round(per_t_us[t - 1], 2) for t in (1, 2, 32, 33, 64, 128, 200, 256)},
        "fill_kernel_floor_us": round(floor_us, 2),
    }
    if not args.no_cpu:
        from oracle import pyoracle

        impl, kind = ("ref_fast", "reference") if pyoracle.ref_available(fast=True) else ("oracle", "port")
        t0 = time.perf_counter()
        for t in range(1, Tmax + 1):
            pyoracle.forward(np.ascontiguousarray(x[:, :t]), H, impl)
        cpu_s = time.perf_counter() - t0
        out["cpu_baseline"] = {"value": round(flops / cpu_s / 1e12, 6), "unit": "TFLOP/s", "cores": 1, "kind": kind,
                               "sample": f"the whole sweep, {cpu_s:.2f} s on 1 thread"}
    print(json.dumps(out), flush=True)


# BASELINE configs other than the headline (3) and the prefix sweep (5b):
# (name, B, T, backward, seed = 1234 + config index, GPU reps, CPU sample as
# (batch elements, heads per element)). The CPU sample is bounded to a few
# seconds of one core: the whole config for C1 and C2, 2 of the 12 heads of
# every batch element for C4, 1 head of each of the 2 batch elements for C5a.
CONFIG_LIST = [
    ("C1", 1, 256, False, 1235, 50, (1, 12)),
    ("C2", 8, 256, True, 1236, 30, (8, 12)),
    ("C4", 8, 1024, True, 1238, 20, (8, 2)),
    ("C5a", 2, 4096, True, 1239, 5, (2, 1)),
]


def _cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _cpu_leg(x, g, H, bwd, sample, gpu_out):
    """The reference CPU backend (oracle/_ref, -O3; the C restatement if that
    is not built) on `sample` = (n_b, n_h): heads 0, H-1, ... of the first n_b
    batch elements, each element's heads as one call with B=1 on a compacted
    qkv (the unchanged function on a smaller tensor). Timed on 1 thread, then
    on N = min(n_b, 16, cpu_count) threads (one batch element each: the
    reference's batch loop is independent per element, so the results are
    identical). The GPU outputs on the same (b, h) are compared with the CPU
    ones (norm-wise and elementwise, tests/tolerances.py's metrics)."""
    import threading

    import numpy as np

    from oracle import pyoracle

    impl, kind = ("ref_fast", "reference") if pyoracle.ref_available(fast=True) else ("oracle", "port")
    B, T, W = x.shape
    C = W // 3
    d = C // H
    n_b, n_h = sample
    heads = sorted({round(i * (H - 1) / max(1, n_h - 1)) for i in range(n_h)}) if n_h < H else list(range(H))
    cols_h = np.concatenate([np.arange(h * d, (h + 1) * d) for h in heads])
    cols_qkv = np.concatenate([cols_h, C + cols_h, 2 * C + cols_h])
    items = [(b, np.ascontiguousarray(x[b:b + 1, :, cols_qkv]), np.ascontiguousarray(g[b:b + 1, :, cols_h]))
             for b in range(n_b)]
    Hs = len(heads)
    res = [None] * n_b

    def work(k):
        b, xs, gs = items[k]
        y, lse = pyoracle.forward(xs, Hs, impl)
        gx = D = None
        if bwd:
            gx, D = pyoracle.backward(xs, y, lse, gs, Hs, impl)
        res[k] = (y, lse, gx, D)

    t0 = time.perf_counter()
    for k in range(n_b):
        work(k)
    t1 = time.perf_counter() - t0
    n_thr = max(1, min(n_b, 16, os.cpu_count() or 1))
    t0 = time.perf_counter()
    for k0 in range(0, n_b, n_thr):
        ths = [threading.Thread(target=work, args=(k,)) for k in range(k0, min(n_b, k0 + n_thr))]
        for th in ths:
            th.start()
        for th in ths:
            th.join()
    tn = time.perf_counter() - t0
    flops = n_b * Hs * d * T * (T + 1) * (7 if bwd else 2)

    def errs(a, r, rtol):
        a = a.astype(np.float64)
        r = r.astype(np.float64)
        m = np.abs(r).max()
        return {"rel": float(np.abs(a - r).max() / m), "elem_excess": float((np.abs(a - r) - rtol * np.abs(r)).max() / m)}

    ygpu, lgpu, gxgpu, Dgpu = gpu_out
    e = {}
    for k, (b, _, _) in enumerate(items):
        y, lse, gx, D = res[k]
        cur = {"O": errs(ygpu[b:b + 1, :, cols_h], y, 1e-5), "LSE": errs(lgpu[b:b + 1, :, heads], lse, 1e-5)}
        if bwd:
            for nm, off in (("dQ", 0), ("dK", 1), ("dV", 2)):
                sel = slice(off * Hs * d, (off + 1) * Hs * d)
                cur[nm] = errs(gxgpu[b:b + 1, :, off * C + cols_h], gx[..., sel], 1e-4)
            cur["D"] = errs(Dgpu[b:b + 1, :, heads], D, 1e-4)
        for nm, v in cur.items():
            if nm not in e:
                e[nm] = v
            else:
                e[nm] = {kk: max(e[nm][kk], v[kk]) for kk in v}
    return {
        "value_1core": round(flops / t1 / 1e12, 6),
        "value_ncore": round(flops / tn / 1e12, 6),
        "unit": "TFLOP/s",
        "cores": [1, n_thr],
        "nproc": os.cpu_count(),
        "cpu_model": _cpu_model(),
        "kind": kind,
        "sample": f"{n_b} batch element(s) x heads {heads} of B={B} T={T} H={H}, "
                  f"{'fwd+bwd' if bwd else 'fwd'}: {t1:.2f} s on 1 thread, {tn:.2f} s on {n_thr}",
        "gpu_vs_cpu_on_sample": {k: {kk: float(f"{vv:.3e}") for kk, vv in v.items()} for k, v in e.items()},
    }


def configs_bench(args):
    """BASELINE configs 1, 2, 4 and 5(a) (BASELINE.md "Results"): per config,
    the forward (C1) or forward + backward through the C ABI on resident
    inputs, K calls back to back between two events (after 3 warm-up calls
    and the clock-settling calls of settle()),
    value = algorithmic FLOPs / time per call; per-kernel averages from the
    library's launch timer in a second pass; the CPU baseline leg on a
    bounded sample, with the GPU outputs' errors on it."""
    import numpy as np
    import torch

    import gpt_amd
    from gpt_amd import synth

    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()
    if args.bwd_path:
        gpt_amd.set_path(args.bwd_path)
    only = set(args.only.split(",")) if args.only else None
    for name, Bc, Tc, bwd, seed, reps, sample in CONFIG_LIST:
        if only and name not in only:
            continue
        x = synth.qkv(Bc, Tc, C, seed)
        g = synth.grad_out(Bc, Tc, C, seed)
        xd, gd = torch.from_numpy(x).to(dev), torch.from_numpy(g).to(dev)
        y = torch.empty(Bc, Tc, C, device=dev)
        lse = torch.empty(Bc, Tc, H, device=dev)
        gx = torch.empty(Bc, Tc, 3 * C, device=dev)
        Dd = torch.empty(Bc, Tc, H, device=dev)

        def call():
            gpt_amd.device_flash_attention_forward(y, lse, xd, Bc, Tc, C, H, stream)
            if bwd:
                gpt_amd.device_flash_attention_backward(gx, Dd, lse, gd, y, xd, Bc, Tc, C, H, stream)

        for _ in range(3):
            call()
        torch.cuda.synchronize()
        settle_steps, settle_ms = settle(call, args.settle_ms)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(reps):
            call()
        e1.record(stream)
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / reps
        gpt_amd.timing_enable(True)
        for _ in range(reps):
            call()
        torch.cuda.synchronize()
        per_kernel = gpt_amd.timing_read()
        gpt_amd.timing_enable(False)
        flops = attn_flops(Bc, Tc, H, D_HEAD, bwd=bwd)
        tf = flops / (ms * 1e-3) / 1e12
        out = {
            "metric": f"causal attn {'fwd+bwd' if bwd else 'fwd'} TFLOP/s & % fp32 MFMA peak, "
                      f"BASELINE config {name[1:]}, 1 GPU",
            "value": round(tf, 3),
            "unit": "TFLOP/s",
            "n_gpus": 1,
            "higher_is_better": True,
            "dtype": "fp32",
            "data": "synthetic (splitmix64 Box-Muller; Q/K/V ~ N(0,1), dO ~ N(0,1e-3))",
            "config": {"workload": f"BASELINE config {name[1:]}: causal {'fwd+bwd' if bwd else 'fwd'}, "
                                   f"B={Bc} T={Tc} H={H} d={D_HEAD}", "flops_per_call": flops, "reps": reps},
            "ms_per_call": round(ms, 5),
            "settle": {"calls": settle_steps, "ms": round(settle_ms, 1)},
            **({"bwd_path": args.bwd_path} if args.bwd_path else {}),
            "pct_fp32_mfma_peak": round(100 * tf / PEAK_FP32_MFMA_TFLOPS, 2),
            "kernels": {k: {"avg_us": round(1e3 * t / n, 3), "launches": n} for k, (t, n) in per_kernel.items()
                        if n > 0},
        }
        if not args.no_cpu:
            torch.cuda.synchronize()
            gpu_out = (y.cpu().numpy(), lse.cpu().numpy(), gx.cpu().numpy() if bwd else None,
                       Dd.cpu().numpy() if bwd else None)
            out["cpu_baseline"] = _cpu_leg(x, g, H, bwd, sample, gpu_out)
        print(json.dumps(out), flush=True)


# GPT-2 124M around the attention path at the C3 shapes (B=16, T=256): d_model
# 768, d_ffn 3072, vocabulary 50257 padded to 50304, 12 layers, max_seq_len 256
# (reference src/train/train.cpp:63-70; weights gpt.cpp:38-84; the call
# sequence of GPT::forward / GPT::backward, gpt.cpp:431-641, and the
# optimizer step, gpt.cpp:643-676).
F_FFN, VOCAB, VOCAB_P = 3072, 50257, 50304
PEAK_HBM_GBS = 8000.0


def ops_bench(args):
    """Each op of one GPT-2 124M training step other than attention, at the
    step's shapes, through gpt_amd.ops (the C ABI of libgpt_hip_ops.so), with
    resident device inputs: median of `reps` event-timed calls on the current
    stream. HBM-bound ops are scored by algorithmic bytes (each operand read
    or written once) against 8 TB/s, GEMM ops by 2 M N K FLOPs per product
    against the fp32 MFMA peak. `per_step` is how many calls of that shape one
    training step makes; `step_ms` = sum of per_step x time over these ops and
    the attention op pair (12 layers, timed here too), i.e. a whole step's GPU
    time when the calls run back to back."""
    import numpy as np
    import torch

    import gpt_amd
    from gpt_amd import ops

    dev = torch.device("cuda:0")
    st = torch.cuda.current_stream()
    M, Cm = B * T, C
    rng = np.random.default_rng(1240)
    n_params = (VOCAB_P * Cm + T * Cm  # wte, wpe (max_seq_len 256, train.cpp:64)
                + LAYERS * (2 * Cm + 3 * Cm * Cm + 3 * Cm + Cm * Cm + Cm + 2 * Cm + 2 * Cm * F_FFN + F_FFN + Cm)
                + 2 * Cm)

    def randn(*shape, scale=1.0):
        return torch.randn(*shape, device=dev) * scale

    tok = torch.from_numpy(rng.integers(0, VOCAB, size=M).astype(np.int32)).to(dev)
    n_unique = int(np.unique(tok.cpu().numpy()).size)
    f4 = 4
    cases = []  # (name, per_step, bound, work, fn)

    wte, wpe = randn(VOCAB_P, Cm, scale=0.02), randn(T, Cm, scale=0.02)
    y = torch.empty(M, Cm, device=dev)
    cases.append(("embedding_forward", 1, "hbm", f4 * (2 * M * Cm + T * Cm + M),
                  lambda: ops.device_embedding_forward(y, wte, wpe, tok, B, T, Cm, VOCAB_P, st)))
    gwte, gwpe, gy = torch.zeros(VOCAB_P, Cm, device=dev), torch.zeros(T, Cm, device=dev), randn(M, Cm)
    cases.append(("embedding_backward", 1, "hbm", f4 * (M * Cm + M + 2 * n_unique * Cm + 2 * T * Cm),
                  lambda: ops.device_embedding_backward(gwte, gwpe, gy, tok, B, T, Cm, VOCAB_P, st)))

    x, res, lny = randn(M, Cm), randn(M, Cm), torch.empty(M, Cm, device=dev)
    gam, bet = 1 + randn(Cm, scale=0.1), randn(Cm, scale=0.1)
    mu, var = torch.empty(M, device=dev), torch.empty(M, device=dev)
    cases.append(("layernorm_residual_forward", 2 * LAYERS + 1, "hbm", f4 * (4 * M * Cm + 2 * Cm + 2 * M),
                  lambda: ops.device_layernorm_residual_fused_forward(lny, mu, var, x, res, gam, bet, B, T, Cm, st)))
    lgx, gres, ggam, gbet = torch.empty(M, Cm, device=dev), randn(M, Cm), torch.zeros(Cm, device=dev), \
        torch.zeros(Cm, device=dev)
    cases.append(("layernorm_residual_backward", 2 * LAYERS + 1, "hbm", f4 * (4 * M * Cm + 2 * M + 5 * Cm),
                  lambda: ops.device_layernorm_residual_fused_backward(lgx, ggam, gbet, gy, gres, x, mu, var, gam,
                                                                       B, T, Cm, st)))

    for tag, k_in, n_out, act in (("qkv", Cm, 3 * Cm, False), ("attn_proj", Cm, Cm, False),
                                  ("ffn_up", Cm, F_FFN, True), ("ffn_down", F_FFN, Cm, False)):
        xi, w, bb = randn(M, k_in), randn(k_in, n_out, scale=k_in ** -0.5), randn(n_out, scale=0.1)
        yo, ao = torch.empty(M, n_out, device=dev), torch.empty(M, n_out, device=dev) if act else None
        cases.append((f"linear_forward_{tag}", LAYERS, "mfma", 2 * M * k_in * n_out,
                      lambda xi=xi, w=w, bb=bb, yo=yo, ao=ao, k_in=k_in, n_out=n_out, act=act:
                      ops.device_linear_activation_fused_forward(yo, ao, xi, w, bb, act, B, T, k_in, n_out, st)))
        gyo, gxi = randn(M, n_out), torch.empty(M, k_in, device=dev)
        gw, gb = torch.zeros(k_in, n_out, device=dev), torch.zeros(n_out, device=dev)
        cases.append((f"linear_backward_{tag}", LAYERS, "mfma", 4 * M * k_in * n_out,
                      lambda gxi=gxi, gw=gw, gb=gb, gyo=gyo, xi=xi, w=w, k_in=k_in, n_out=n_out:
                      ops.device_linear_backward(gxi, gw, gb, gyo, xi, w, B, T, k_in, n_out, st)))
    ga, gyf, xf = torch.empty(M, F_FFN, device=dev), randn(M, F_FFN), randn(M, F_FFN)
    cases.append(("activation_backward", LAYERS, "hbm", f4 * 3 * M * F_FFN,
                  lambda: ops.device_activation_backward(ga, gyf, xf, B, T, F_FFN, st)))

    logits, probs = torch.empty(M, VOCAB_P, device=dev), torch.empty(M, VOCAB_P, device=dev)
    cases.append(("unembedding_forward", 1, "mfma", 2 * M * Cm * VOCAB_P,
                  lambda: ops.device_unembedding_forward(logits, x, wte, B, T, Cm, VOCAB_P, st)))
    cases.append(("softmax_forward", 1, "hbm", f4 * 2 * M * VOCAB_P,
                  lambda: ops.device_softmax_forward(probs, logits, B, T, VOCAB, VOCAB_P, st)))
    gl = torch.zeros(M, VOCAB_P, device=dev)
    cases.append(("cross_entropy_softmax_backward", 1, "hbm", f4 * (2 * M * VOCAB + M),
                  lambda: ops.device_cross_entropy_softmax_fused_backward(gl, probs, tok, B, T, VOCAB, VOCAB_P, st)))
    loss = torch.empty(1, device=dev)
    cases.append(("cross_entropy_loss", 1, "hbm", f4 * 2 * M,
                  lambda: ops.device_cross_entropy_loss(loss, probs, tok, B, T, VOCAB_P, st)))
    gxu = torch.empty(M, Cm, device=dev)
    cases.append(("unembedding_backward", 1, "mfma", 4 * M * Cm * VOCAB_P,
                  lambda: ops.device_unembedding_backward(gxu, gwte, gl, x, wte, B, T, Cm, VOCAB_P, st)))

    prm, grd = randn(n_params, scale=0.02), randn(n_params, scale=1e-3)
    m1, v1 = torch.zeros(n_params, device=dev), torch.zeros(n_params, device=dev)
    cases.append(("adamw_step", 1, "hbm", f4 * 7 * n_params,
                  lambda: ops.device_adamw_step(prm, grd, m1, v1, n_params, 6e-4, 0.9, 0.95, 1e-8, 0.1, 1, st)))
    cases.append(("scale_and_clip_grad", 1, "hbm", f4 * n_params,  # nothing to clip: one read
                  lambda: ops.device_scale_and_clip_grad(grd, n_params, 1e9, 1, st)))

    # the attention op pair of one layer, for the step total
    qkv = randn(B, T, 3 * Cm)
    ya, la = torch.empty(B, T, Cm, device=dev), torch.empty(B, T, H, device=dev)
    gqkv, Dc, dya = torch.empty(B, T, 3 * Cm, device=dev), torch.empty(B, T, H, device=dev), randn(B, T, Cm)
    cases.append(("attention_forward", LAYERS, "mfma", attn_flops(B, T, H, D_HEAD, bwd=False),
                  lambda: gpt_amd.device_flash_attention_forward(ya, la, qkv, B, T, Cm, H, st)))
    cases.append(("attention_backward", LAYERS, "mfma", attn_flops(B, T, H, D_HEAD, fwd=False),
                  lambda: gpt_amd.device_flash_attention_backward(gqkv, Dc, la, dya, ya, qkv, B, T, Cm, H, st)))

    reps = max(5, args.steps // 2)
    res_ops = {}
    step_ms = 0.0
    for name, per_step, bound, work, fn in cases:
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        torch.cuda._sleep(5_000_000)  # queue the reps behind a GPU spin: time the GPU, not the launches
        ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(reps)]
        for e0, e1 in ev:
            e0.record(st)
            fn()
            e1.record(st)
        torch.cuda.synchronize()
        us = float(np.median([a.elapsed_time(b) for a, b in ev])) * 1e3
        if bound == "hbm":
            ach, peak, unit = work / (us * 1e-6) / 1e9, PEAK_HBM_GBS, "GB/s"
        else:
            ach, peak, unit = work / (us * 1e-6) / 1e12, PEAK_FP32_MFMA_TFLOPS, "TFLOP/s"
        res_ops[name] = {"us": round(us, 2), "per_step": per_step, "bound": bound,
                         ("bytes" if bound == "hbm" else "flops"): work, "achieved": round(ach, 2), "unit": unit,
                         "frac": round(ach / peak, 4)}
        step_ms += per_step * us / 1e3
    out = {
        "metric": "GPT-2 124M training-step ops on one MI355X: per-op GPU time vs roofline, B=16 T=256",
        "n_gpus": 1,
        "dtype": "fp32",
        "data": "synthetic (torch.randn / uniform token ids)",
        "config": {"workload": "every IGPTBackend compute op of one GPT-2 124M step at B=16 T=256 "
                               "(12 layers, d_model 768, d_ffn 3072, vocab 50257 padded to 50304)",
                   "params": n_params, "reps": reps},
        "ops": res_ops,
        "step_ms": round(step_ms, 3),
        "peaks": {"hbm_GBs": PEAK_HBM_GBS, "fp32_mfma_TFLOPs": PEAK_FP32_MFMA_TFLOPS},
    }
    if not args.no_cpu:
        out["cpu_baseline"] = ops_cpu_baseline(res_ops)
    print(json.dumps(out), flush=True)


def ops_cpu_baseline(res_ops):
    """The reference CPUBackend ops (oracle/_ref, -O3, one thread) on bounded
    samples of the same shapes (a few rows each, the rest of the shape as in
    the step); each op's time is scaled to the step's rows, and `step_s` is
    the whole step at that rate."""
    import numpy as np

    from oracle import pyoracle, pyops

    impl, kind = ("ref_fast", "reference") if pyoracle.ref_available(fast=True) else ("oracle", "port")
    rng = np.random.default_rng(7)
    Cm = C

    def rnd(*shape, s=1.0):
        return (rng.standard_normal(shape) * s).astype(np.float32)

    per_op = {}

    def timed(name, rows, fn, scale_rows):
        t0 = time.perf_counter()
        fn()
        dt = time.perf_counter() - t0
        per_op[name] = {"sample_rows": rows, "s_at_step_shape": round(dt * scale_rows / rows, 4)}

    Mfull = B * T
    r = 64
    tok = rng.integers(0, VOCAB, size=r).astype(np.int32)
    wte, wpe = rnd(VOCAB_P, Cm, s=0.02), rnd(T, Cm, s=0.02)
    timed("embedding_forward", r, lambda: pyops.embedding_forward(np.zeros((r, Cm), np.float32), wte, wpe, tok, 1, r,
                                                                   Cm, impl), Mfull)
    gw = np.zeros_like(wte)
    timed("embedding_backward", r, lambda: pyops.embedding_backward(gw, np.zeros((T, Cm), np.float32),
                                                                     rnd(r, Cm), tok, 1, r, Cm, impl), Mfull)
    r = 512
    x, res = rnd(r, Cm), rnd(r, Cm)
    g_, b_ = rnd(Cm), rnd(Cm)
    mu, var = np.zeros(r, np.float32), np.zeros(r, np.float32)
    timed("layernorm_residual_forward", r, lambda: pyops.layernorm_forward(np.zeros((r, Cm), np.float32), mu, var, x,
                                                                            res, g_, b_, 1, r, Cm, impl), Mfull)
    timed("layernorm_residual_backward", r, lambda: pyops.layernorm_backward(
        np.zeros((r, Cm), np.float32), np.zeros(Cm, np.float32), np.zeros(Cm, np.float32), rnd(r, Cm), rnd(r, Cm), x,
        mu, var, g_, 1, r, Cm, impl), Mfull)
    r = 8
    for tag, k_in, n_out, act in (("qkv", Cm, 3 * Cm, False), ("attn_proj", Cm, Cm, False),
                                  ("ffn_up", Cm, F_FFN, True), ("ffn_down", F_FFN, Cm, False)):
        xi, w, bb = rnd(r, k_in), rnd(k_in, n_out, s=0.03), rnd(n_out)
        timed(f"linear_forward_{tag}", r, lambda: pyops.linear_forward(
            np.zeros((r, n_out), np.float32), np.zeros((r, n_out), np.float32), xi, w, bb, act, 1, r, k_in, n_out,
            impl), Mfull)
        timed(f"linear_backward_{tag}", r, lambda: pyops.linear_backward(
            np.zeros((r, k_in), np.float32), np.zeros((k_in, n_out), np.float32), np.zeros(n_out, np.float32),
            rnd(r, n_out), xi, w, 1, r, k_in, n_out, impl), Mfull)
    r = 256
    timed("activation_backward", r, lambda: pyops.activation_backward(np.zeros((r, F_FFN), np.float32), rnd(r, F_FFN),
                                                                       rnd(r, F_FFN), 1, r, F_FFN, impl), Mfull)
    r = 2
    xu = rnd(r, Cm)
    timed("unembedding_forward", r, lambda: pyops.unembedding_forward(np.zeros((r, VOCAB_P), np.float32), xu, wte, 1,
                                                                       r, Cm, VOCAB_P, impl), Mfull)
    timed("unembedding_backward", r, lambda: pyops.unembedding_backward(
        np.zeros((r, Cm), np.float32), np.zeros_like(wte), rnd(r, VOCAB_P, s=1e-4), xu, wte, 1, r, Cm, VOCAB_P, impl),
        Mfull)
    r = 64
    lg = rnd(r, VOCAB_P, s=3.0)
    pr = np.zeros_like(lg)
    labels = rng.integers(0, VOCAB, size=r).astype(np.int32)
    timed("softmax_forward", r, lambda: pyops.softmax_forward(pr, lg, 1, r, VOCAB, VOCAB_P, impl), Mfull)
    timed("cross_entropy_softmax_backward", r, lambda: pyops.ce_backward(np.zeros_like(lg), pr, labels, 1, r, VOCAB,
                                                                          VOCAB_P, impl), Mfull)
    timed("cross_entropy_loss", r, lambda: pyops.ce_loss(pr, labels, 1, r, VOCAB_P, impl), Mfull)
    n = 1 << 22
    p_, g2 = rnd(n, s=0.02), rnd(n, s=1e-3)
    n_params = res_ops["adamw_step"]["bytes"] // 28
    timed("adamw_step", n, lambda: pyops.adamw(p_, g2, np.zeros(n, np.float32), np.zeros(n, np.float32), n, 6e-4, 0.9,
                                               0.95, 1e-8, 0.1, 1, impl), n_params)
    timed("scale_and_clip_grad", n, lambda: pyops.scale_clip(g2, n, 1e9, 1, impl), n_params)
    step_s = sum(res_ops[k]["per_step"] * v["s_at_step_shape"] for k, v in per_op.items())
    gpu_ms = sum(v["per_step"] * v["us"] for k, v in res_ops.items() if k in per_op) / 1e3
    return {"value": round(step_s, 3), "unit": "s per step (these ops, attention excluded)", "cores": 1,
            "kind": kind, "gpu_ms_same_ops": round(gpu_ms, 3),
            "sample": "each op on a few rows of its step shape (sample_rows), time scaled to the step's rows",
            "ops": per_op}


def main():
    args = parse()
    if args.traffic:
        write_traffic(*args.traffic)
        return
    if args.copy_calibration:
        copy_calibration()
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus {args.gpus}): the attention op "
              f"shards per (batch, head) with no communication; run with --gpus 1.", file=sys.stderr)
        sys.exit(2)
    if args.prefix_sweep:
        prefix_sweep(args)
        return
    if args.ops:
        ops_bench(args)
        return
    if args.configs:
        configs_bench(args)
        return

    import numpy as np
    import torch

    import gpt_amd
    from gpt_amd import synth

    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()
    if args.bwd_path:
        gpt_amd.set_path(args.bwd_path)
    scales = synth.layer_scales(LAYERS, CONFIG_SEED)

    # Per-layer buffers, as GPT::set_size lays them out (gpt.cpp:101-214).
    qkv, dout, y, lse, gx, Dc = [], [], [], [], [], []
    for layer in range(LAYERS):
        seed = CONFIG_SEED + layer
        qkv.append(torch.from_numpy(synth.qkv(B, T, C, seed, scale=float(scales[layer]))).to(dev))
        dout.append(torch.from_numpy(synth.grad_out(B, T, C, seed)).to(dev))
        y.append(torch.empty(B, T, C, device=dev))
        lse.append(torch.empty(B, T, H, device=dev))
        gx.append(torch.empty(B, T, 3 * C, device=dev))
        Dc.append(torch.empty(B, T, H, device=dev))
    torch.cuda.synchronize()

    def step():
        for layer in range(LAYERS):
            gpt_amd.device_flash_attention_forward(y[layer], lse[layer], qkv[layer], B, T, C, H, stream)
        for layer in reversed(range(LAYERS)):
            gpt_amd.device_flash_attention_backward(gx[layer], Dc[layer], lse[layer], dout[layer], y[layer],
                                                    qkv[layer], B, T, C, H, stream)

    gpt_amd.wait_timeouts()  # clear counts left by earlier work in this process
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    settle_steps, settle_ms = settle(step, args.settle_ms)

    # Timed region: exactly K steps between two events, nothing else recorded.
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    start.record(stream)
    for _ in range(args.steps):
        step()
    end.record(stream)
    torch.cuda.synchronize()
    total_ms = start.elapsed_time(end)

    # Breakdown pass: the same K steps again with the library's launch timer
    # (each kernel's own dispatch start and end timestamps). Kept out of the
    # timed region, whose step time alone is the metric.
    gpt_amd.timing_enable(True)
    torch.cuda.synchronize()
    for k in range(args.steps):
        step()
    torch.cuda.synchronize()
    per_kernel = gpt_amd.timing_read()
    gpt_amd.timing_enable(False)
    # A dQ wait that gave up at its spin limit computed from incomplete dS
    # tiles: the measured work would not be the op's, so the run fails.
    timeouts = gpt_amd.wait_timeouts()
    if timeouts:
        sys.exit(f"bench.py: {timeouts} dQ waits of the one-launch backward hit their spin limit")

    ms_per_step = total_ms / args.steps
    step_flops = LAYERS * attn_flops(B, T, H, D_HEAD)
    tflops = step_flops / (ms_per_step * 1e-3) / 1e12

    kernels = {k: {"avg_us": round(1e3 * ms / n, 3), "launches": n, "tflops": round(
                   KERNEL_FLOP_UNITS[k] * B * H * D_HEAD * T * (T + 1) / (ms / n * 1e-3) / 1e12, 3)}
               for k, (ms, n) in per_kernel.items() if n > 0 and k in KERNEL_FLOP_UNITS}
    dom = max((k for k in kernels if k in KERNEL_FLOP_UNITS), key=lambda k: per_kernel[k][0])
    dom_ms = per_kernel[dom][0] / per_kernel[dom][1]
    dom_flops = KERNEL_FLOP_UNITS[dom] * B * H * D_HEAD * T * (T + 1)
    dom_tf = dom_flops / (dom_ms * 1e-3) / 1e12
    traffic = None
    tpath = os.path.join(ROOT, "profiles", f"{dom}_c3_traffic.json")
    if os.path.exists(tpath):
        rec = json.load(open(tpath))
        if rec.get("kernel") == KERNEL_SYMBOL[dom]:
            traffic = rec.get("hbm_bytes_per_launch")

    out = {
        "metric": METRIC,
        "value": round(tflops, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "settle": {"steps": settle_steps, "ms": round(settle_ms, 1)},
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic (splitmix64 Box-Muller; Q/K/V ~ N(0,1)*U[0.5,2] per layer, dO ~ N(0,1e-3))",
        "config": {
            "workload": "GPT-2 124M attention micro-step: 12 layers x causal fwd+bwd, B=16 T=256 H=12 d=64",
            "layers": LAYERS, "batch": B, "seq_len": T, "heads": H, "head_dim": D_HEAD,
            "flops_per_step": step_flops,
            **({"bwd_path": args.bwd_path} if args.bwd_path else {}),
        },
        "pct_fp32_mfma_peak": round(100 * tflops / PEAK_FP32_MFMA_TFLOPS, 2),
        "kernels": kernels,
        "kernel_ms_per_step": round(sum(ms for ms, n in per_kernel.values()) / args.steps, 4),
        "roofline": {
            "kernel": KERNEL_SYMBOL[dom],
            "bound": "mfma",
            "achieved": round(dom_tf, 3),
            "peak": PEAK_FP32_MFMA_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(dom_tf / PEAK_FP32_MFMA_TFLOPS, 4),
            "traffic": traffic,
            "flops_per_launch": dom_flops,
            "avg_launch_us": round(dom_ms * 1e3, 3),
        },
    }
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(args.cpu_layers)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
