"""Benchmark of the MI355X TabICLv2 FP32 forward: cached-prediction test rows/s
and static-context build ms on one GPU.

Workload (N=1): the 50,000-train-row classifier: 50,000 x 64 features
N(0,1), 10 classes from a seeded linear map, seeded random-init FP32 weights
of the official architecture, written as an IRMODEL v1 artifact of the
official profile and loaded from it; the static context is built once and
held in HBM; 4,096 test rows are predicted in passes of 512 against the
cached ICL K/V.

A step is one prediction of the 4,096 test rows at Predictor::predict's
boundary: host x in, host logits out through irx_predictor_predict (H2D and
D2H included), its eight passes alternating between two HIP streams. After
untimed warmups each call is timed on its own; `value` is the test rows over
the nearest-rank p50 call time, reported with min/p95/p99/max/mean, the
samples and an FP64 output checksum (the reference's benchmark contract). The
same calls with inputs already in HBM are reported beside it. Kernel timing
runs in separate legs: the dominant kernel (ICL attention) is timed with HIP
events in steps whose passes run in order on one stream, where its launches
have the GPU to themselves. The build is timed separately (host FP32 inputs
to a resident context; nearest-rank p50 of five builds). The oracle (C
restatement of the reference CPU path) is timed on the host's cores on a
bounded sample of the same rows. Passes of 1, 8, 16 and 32 rows, where
streaming the cached K/V from HBM bounds the cross-attention, are timed after
the steps and reported with their HBM fraction. The same workload at
optimize="auto" (FP16 ICL cache, split-FP16 attention) and optimize="fast"
(FP8 ICL cache, FP16 attention products) is reported beside the FP32 line,
each with its accuracy gate.

Prints one JSON line.
"""

from __future__ import annotations

import argparse
import ctypes
import json
import os
import re
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

MFMA_FP32_PEAK_TFLOPS = 157.3
MFMA_FP16_PEAK_TFLOPS = 2500.0  # dense
CLASSES = 10
HBM_PEAK_GBPS = 8000.0
WORKLOAD = "clf-50k"
# Pass sizes of the HBM-bound sweep of the cross-attention, and passes timed each.
SMALL_PASSES = (1, 8, 16, 32)
SMALL_PASS_REPEATS = 10
# rocprofv3 FETCH_SIZE/WRITE_SIZE summary of the prediction-phase ICL attention
# launch on this workload, calibrated against a plain copy kernel.
TRAFFIC_PROFILE = os.path.join(ROOT, "profiles", "icl_attention_kernel_clf-50k.md")


def nearest_rank(values, percentile: int) -> float:
    """Nearest-rank percentile: sorted sample ceil(p N / 100), ranks from one
    (BenchmarkStats, src/benchmark.rs:26-49)."""
    v = sorted(values)
    return float(v[max(1, -(-len(v) * percentile // 100)) - 1])


def timed_calls(call, warmup: int, steps: int) -> list[float]:
    """Untimed warmups, then each call timed on its own (seconds); every call
    returns with its outputs written."""
    for _ in range(warmup):
        call()
    samples = []
    for _ in range(steps):
        t0 = time.perf_counter()
        call()
        samples.append(time.perf_counter() - t0)
    return samples


def latency_stats(seconds) -> dict:
    """min / p50 / p95 / p99 / max / mean in milliseconds of per-call durations."""
    ms = [1000.0 * t for t in seconds]
    return {"min_ms": min(ms), "p50_ms": nearest_rank(ms, 50), "p95_ms": nearest_rank(ms, 95),
            "p99_ms": nearest_rank(ms, 99), "max_ms": max(ms), "mean_ms": sum(ms) / len(ms), "calls": len(ms)}


def executor_from_model_file(task: str, weights: dict, device):
    """The model as the reference loads it: the seeded random-init weights
    written as an IRMODEL v1 artifact of the official profile (a temporary
    file), read back and uploaded through irx_weights_upload."""
    import tempfile

    from ironicl_amd import model_file, tabicl

    with tempfile.TemporaryDirectory() as tmp:
        path = os.path.join(tmp, f"{task}.irmodel")
        summary = model_file.write_model(path, task, weights)
        executor = tabicl.Executor.from_model_file(path, device)
        report = {"format": "IRMODEL v1", "bytes": os.path.getsize(path), "profile": summary.profile,
                  "source_sha256": summary.source_sha256, "tensors": summary.tensor_count,
                  "parameters": summary.parameter_count}
    return executor, report


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def host_facts() -> dict:
    facts = {"logical_cpus": os.cpu_count()}
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            if line.startswith("Model name:"):
                facts["cpu_model"] = line.split(":", 1)[1].strip()
        facts["avx512"] = "avx512f" in open("/proc/cpuinfo").read()
    except Exception:
        pass
    return facts


def profiled_traffic() -> int | None:
    """HBM bytes per launch of the dominant kernel, from the committed counter
    summary (two rocprofv3 --pmc passes scaled by the copy-kernel factors)."""
    try:
        text = open(TRAFFIC_PROFILE).read()
    except OSError:
        return None
    m = re.search(r"^traffic_bytes_per_launch = (\d+)$", text, re.M)
    return int(m.group(1)) if m else None


def attention_back_to_back(device, pairs: int, n: int, rows_list, layers: int = 12, rounds: int = 4) -> dict:
    """The whole KV-streaming cross-attention of a pass of few rows (the
    attention kernel and its split-K merge, as a pass issues them), launched
    back to back through irx_icl_attention_noalloc over `layers` K/V buffers
    of one ICL layer's shape ([pairs, n, 64] each; rotated, so every call
    streams its K/V from HBM past the 256 MB MALL) and timed with one pair of
    HIP events around rounds x layers calls: no event between the two
    launches of a call, so neither carries a timed launch's overhead."""
    from ironicl_amd import hip, hipmem

    rt = hipmem.runtime()
    kv = np.random.default_rng(11).standard_normal(pairs * n * 64, dtype=np.float32)
    ks = [hipmem.DeviceArray.from_host(kv) for _ in range(layers)]
    vs = [hipmem.DeviceArray.from_host(kv[::-1]) for _ in range(layers)]
    del kv
    e0, e1 = ctypes.c_void_p(), ctypes.c_void_p()
    hipmem._ok(rt.hipEventCreate(ctypes.byref(e0)), "hipEventCreate")
    hipmem._ok(rt.hipEventCreate(ctypes.byref(e1)), "hipEventCreate")
    out = {}
    try:
        for rows in rows_list:
            qd = hipmem.DeviceArray.from_host(
                (np.random.default_rng(rows).standard_normal((pairs, rows, 64)) * 0.5).astype(np.float32))
            od = hipmem.DeviceArray((pairs // 8, rows, 512))

            def call(i):
                hip.check(hip.lib().irx_icl_attention_noalloc(device.handle, qd.ptr, ks[i].ptr, vs[i].ptr, pairs, rows,
                                                              n, od.ptr, None))

            for i in range(layers):
                call(i)
            hipmem.synchronize()
            best = float("inf")
            for _ in range(3):
                hipmem._ok(rt.hipEventRecord(e0, None), "hipEventRecord")
                for _ in range(rounds):
                    for i in range(layers):
                        call(i)
                hipmem._ok(rt.hipEventRecord(e1, None), "hipEventRecord")
                hipmem._ok(rt.hipEventSynchronize(e1), "hipEventSynchronize")
                ms = ctypes.c_float()
                hipmem._ok(rt.hipEventElapsedTime(ctypes.byref(ms), e0, e1), "hipEventElapsedTime")
                best = min(best, ms.value / (rounds * layers))
            algo = 2.0 * pairs * n * 64 * 4 + 2.0 * pairs * rows * 64 * 4
            out[str(rows)] = {"ms_per_layer": best, "achieved_gbps": algo / (best * 1e-3) / 1e9,
                              "frac": algo / (best * 1e-3) / 1e9 / HBM_PEAK_GBPS}
            del qd, od
    finally:
        rt.hipEventDestroy(e0)
        rt.hipEventDestroy(e1)
        for a in ks + vs:
            a.free()
    return out


def predict_flops_per_row(n: int, h: int, width: int) -> float:
    """Algorithmic FLOPs of one test row's cached prediction against an
    N-row, H-feature context: column stage 3 H (12 D^2 + 4 M D), row stage
    36 L D^2 + 8 L^2 D + 16 L D + 48 D^2, ICL 12 (12 E^2 + 131,072) + 48 N E,
    decoder 2 E 1,024 + 2,048 width (D = M = 128, E = 512, L = H + 4)."""
    d, m, e, length = 128, 128, 512, h + 4
    column = 3 * h * (12 * d * d + 4 * m * d)
    row = 36 * length * d * d + 8 * length * length * d + 16 * length * d + 48 * d * d
    icl = 12 * (12 * e * e + 131072) + 12 * 4 * n * e
    return float(column + row + icl + 2 * e * 1024 + 2 * 1024 * width)


def cpu_baseline(weights, context_host, x_test, gpu_logits, threads: int, target_s: float) -> dict:
    """The oracle's cached prediction on the host cores, on a bounded sample of
    the workload's test rows (sized for about target_s seconds of CPU work), at
    the reference's default thread count and native-approximation math; then,
    on a third of that sample, all logical cores, and on a sixth, exact math as
    the control."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O

    O.set_threads(threads)
    m = O.OracleModel("classifier", weights, O.NATIVE)
    # Calls of about two seconds each (sized from the rate so far) over the
    # test rows in order, wrapping to the first row again when the CPU is fast
    # enough to finish them before target_s; parity is checked on the first
    # pass over the rows.
    n_test = x_test.shape[1]
    rows, dt, chunk, parts = 0, 0.0, 8, []
    while dt < target_s or not parts:
        start = rows % n_test
        take = min(chunk, n_test - start)
        t0 = time.perf_counter()
        out = m.predict_cached(context_host, np.ascontiguousarray(x_test[:, start:start + take]))
        dt += time.perf_counter() - t0
        if rows < n_test:
            parts.append(out)
        rows += take
        chunk = max(8, int(rows / dt * min(2.0, max(target_s - dt, 0.0))))
    logits = np.concatenate(parts, axis=1)
    unique = logits.shape[1]
    gpu = gpu_logits[:, :unique, : logits.shape[2]]
    cpu = logits[..., : gpu.shape[2]]
    excess = np.abs(gpu - cpu) - (1e-5 + 1e-4 * np.abs(cpu))

    def variant(model, workers, sample_rows):
        # A shorter sample of the same rows: the all-logical-cores variant and
        # the exact-math control of the reference's CPU path.
        O.set_threads(workers)
        t0 = time.perf_counter()
        out = model.predict_cached(context_host, np.ascontiguousarray(x_test[:, :sample_rows]))
        dt_v = time.perf_counter() - t0
        O.set_threads(threads)
        return {"value": sample_rows / dt_v, "cores": workers, "rows": sample_rows, "seconds": dt_v,
                "max_abs_diff_vs_gpu": float(np.abs(gpu_logits[:, :sample_rows, : out.shape[2]]
                                                    - out[..., : gpu.shape[2]]).max())}

    sample = max(8, min(unique, rows // 3))
    logical = os.cpu_count() or threads
    all_cores = variant(m, logical, sample)
    exact = variant(O.OracleModel("classifier", weights, O.EXACT), threads, max(8, sample // 2))
    n, h = context_host[2][0].shape[2], x_test.shape[2]
    per_row = predict_flops_per_row(n, h, CLASSES)
    all_cores["gflops"] = all_cores["value"] * per_row / 1e9
    exact["gflops"] = exact["value"] * per_row / 1e9
    return {
        "value": rows / dt,
        "unit": "rows/s",
        "gflops": rows / dt * per_row / 1e9,
        "flops_per_row": per_row,
        "cores": threads,
        "kind": "port",
        "sample": f"cached prediction of {rows} test rows ({min(rows, n_test)} distinct: the {n_test} test rows "
                  f"in order, from the first again once all ran) against the same 50k-row context, in calls of "
                  f"about 2 s, C restatement of the reference CPU path (native-approximation math, "
                  f"{threads} threads = ceil(logical/2) as the reference defaults)",
        "seconds": dt,
        "parity_rows": unique,
        "parity_max_abs_diff": float(np.abs(gpu - cpu).max()),
        "parity_ok": bool(excess.max() <= 0 and np.array_equal(gpu.argmax(-1), cpu.argmax(-1))),
        "all_logical_cores": all_cores,
        "exact_math_control": exact,
    }


def cpu_build_baseline(weights, x, y, threads: int, sample_rows: int = 2000) -> dict:
    """The oracle's static-context build (the reference CPU path's
    build_tensors_cpu) on the host cores, extrapolated to the workload's N: the
    build is timed at `sample_rows` training rows; its twelve ICL self-attentions
    (serial per estimator, as in the reference) are timed alone at that shape
    and scaled by N^2, the rest of the build by N."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O

    O.set_threads(threads)
    m = O.OracleModel("classifier", weights, O.NATIVE)
    n_full, n = x.shape[1], min(sample_rows, x.shape[1])
    t0 = time.perf_counter()
    m.build_context(np.ascontiguousarray(x[:, :n]), np.ascontiguousarray(y[:, :n]))
    build_s = time.perf_counter() - t0
    rng = np.random.default_rng(0)
    qkv = [rng.standard_normal((8, n, 64)).astype(np.float32) * 0.3 for _ in range(3)]
    t0 = time.perf_counter()
    O.attention(*qkv, math=O.NATIVE)
    att_s = 12 * (time.perf_counter() - t0)
    linear_s = max(build_s - att_s, 0.0)
    scale = n_full / n
    estimate = linear_s * scale + att_s * scale * scale
    return {"value_ms": 1000 * estimate, "kind": "port", "extrapolated": True, "cores": threads,
            "sample": f"oracle build (native math, {threads} threads) of the first {n} training rows: "
                      f"{build_s:.2f} s, of which the 12 serial ICL self-attentions {att_s:.2f} s (timed alone); "
                      f"extrapolated to {n_full:,} rows as the rest x N and the attentions x N^2",
            "sample_seconds": build_s}


def bench_fitted(executor, x, y, xt, args) -> dict:
    """TabICL preprocessing on the GPU and a fitted model predicting from raw
    features: the workload's rows as raw features with every fifth column
    log-normal, 8 ensemble members, none and power groups."""
    from ironicl_amd import hip, hipmem
    from ironicl_amd import preprocess as pp
    from ironicl_amd.fitted import FittedModel

    raw = np.array(x[0], dtype=np.float32)
    raw[:, ::5] = np.exp(raw[:, ::5])
    labels = y[0].astype(np.int64)
    query = np.array(xt[0], dtype=np.float32)
    query[:, ::5] = np.exp(query[:, ::5])
    opts = pp.PreprocessOptions()
    pp.Preprocessor.fit(opts, raw[:1000], labels[:1000], executor.device)  # warm-up
    t0 = time.perf_counter()
    p = pp.Preprocessor.fit(opts, raw, labels, executor.device)
    fit_ms = 1000 * (time.perf_counter() - t0)
    dev = hipmem.DeviceArray((p.member_count, query.shape[0], p.n_features_out))
    p.member_rows_device(query, dev.ptr)
    t0 = time.perf_counter()
    reps = 20
    for _ in range(reps):
        p.member_rows_device(query, dev.ptr)
    transform_s = (time.perf_counter() - t0) / reps
    log(f"preprocessing fit {fit_ms:.1f} ms, transform of {query.shape[0]} rows {1e3 * transform_s:.2f} ms")
    report = {
        "workload": f"{raw.shape[0]} x {raw.shape[1]} raw features (every fifth column log-normal), "
                    f"{p.member_count} members, groups {'+'.join(p.group_methods)}",
        "preprocess_fit_ms": fit_ms,
        "transform_rows_per_s": query.shape[0] / transform_s,
    }
    if not args.no_cpu:
        sys.path.insert(0, os.path.join(ROOT, "oracle"))
        import preprocess_oracle as PO
        sample = 8  # features
        t0 = time.perf_counter()
        PO.fit(raw.astype(np.float64), p.kept[:sample], p.group_methods, opts.outlier_threshold)
        cpu_s = (time.perf_counter() - t0) * len(p.kept) / sample
        report["cpu_baseline_fit"] = {"seconds": cpu_s, "cores": 1, "kind": "port",
                                      "sample": f"oracle (NumPy f64) fit of {sample} of {len(p.kept)} features, "
                                                f"scaled to all"}
    t0 = time.perf_counter()
    fm = FittedModel.fit(executor, raw, labels, opts)
    hipmem.synchronize()
    report["fit_s"] = time.perf_counter() - t0
    fm.predict_proba(query[:512])
    t0 = time.perf_counter()
    fm.predict_proba(query)
    report["predict_proba_rows_per_s"] = query.shape[0] / (time.perf_counter() - t0)
    log(f"fitted model: fit {report['fit_s']:.2f} s, predict_proba {report['predict_proba_rows_per_s']:.0f} rows/s")
    del fm
    return report


# The reduced-precision levels: optimize -> (ICL cache bytes per value, FP16
# products per FP32-equivalent product, gate on |logit - safe|
# (docs/experiments.md:406-423), wide and decode kernels).
LEVELS = {
    "auto": (2, 2, 1e-2, "icl_attention_split_kernel (FP16 cache, queries and probabilities split hi + lo into "
                         "one accumulator, 32x32x16 FP16 MFMA)",
             "icl_decode16_kernel (FP16 cache, 16x16x32 FP16 MFMA)"),
    "fast": (1, 1, 5e-2, "icl_attention_split_kernel<FP8> (E4M3 cache with per-dim scales, converted to FP16 after "
                         "the LDS read; FP16 queries and probabilities, 32x32x16 FP16 MFMA)",
             "icl_decode16_kernel<FP8> (E4M3 cache, 16x16x32 FP16 MFMA)"),
}


def bench_level(optimize, executor, x, y, q, dx, gpu_input, gpu_logits, args) -> dict:
    """A reduced-precision optimize level on the same workload: "auto" (FP16
    ICL cache, split-FP16 attention products) or "fast" (FP8 ICL cache, FP16
    products). Build ms (nearest-rank p50), rows/s over the p50 of per-call
    times from host buffers (two streams), the attention
    launch's rate (single-stream steps), the small passes' HBM rate, and the
    level's accuracy gate against the "safe" logits of the main run (max
    |logit| difference, labels that differ where safe's top-2 margin exceeds
    twice the gate)."""
    from ironicl_amd import hip, hipmem

    elem, products, gate, wide_name, decode_name = LEVELS[optimize]
    ms = []
    ctx = executor.build_context(x, y, optimize=optimize)
    for _ in range(max(1, args.build_repeats)):
        del ctx
        hipmem.synchronize()
        t0 = time.perf_counter()
        ctx = executor.build_context(x, y, optimize=optimize)
        hipmem.synchronize()
        ms.append(1000 * (time.perf_counter() - t0))
    ctx.set_pass_rows(args.pass_rows)
    b = x.shape[0]
    dl = hipmem.DeviceArray((b, q, executor.width))

    def step():
        hip.check(hip.lib().irx_predictor_predict_device(ctx.handle, dx.ptr, q, dl.ptr, None))

    xh = np.ascontiguousarray(gpu_input, np.float32)
    lh = np.zeros((b, q, executor.width), np.float32)
    no_progress = hip.PROGRESS()

    def host_call():
        hip.check(hip.lib().irx_predictor_predict(ctx.handle, hip.fptr(xh), q, hip.fptr(lh), None, no_progress,
                                                  None))

    samples = timed_calls(host_call, args.warmup, args.steps)
    stats = latency_stats(samples)
    logits = lh.copy()
    step()
    ctx.set_streams(1)
    step()
    hip.profile_enable(["icl_attention"])
    for _ in range(args.steps):
        step()
    hipmem.synchronize()
    att = hip.profile_read("icl_attention")
    hip.profile_enable(False)
    # Small passes: HBM-bound over the cache's K and V of one layer.
    small = {}
    n = x.shape[1]
    kv_bytes = 2.0 * b * 8 * n * 64 * elem
    ctx.set_pass_rows(max(SMALL_PASSES))
    for qb in SMALL_PASSES:
        def small_step():
            hip.check(hip.lib().irx_predictor_predict_device(ctx.handle, dx.ptr, qb, dl.ptr, None))

        small_step()
        hipmem.synchronize()
        hip.profile_enable(["icl_attention"])
        for _ in range(SMALL_PASS_REPEATS):
            small_step()
        hipmem.synchronize()
        st = hip.profile_read("icl_attention")
        hip.profile_enable(False)
        lm = st["milliseconds"] / max(st["launches"], 1)
        algo = kv_bytes + 2.0 * b * 8 * qb * 64 * 4
        small[str(qb)] = {"avg_launch_ms": lm, "bytes_per_launch": algo,
                          "achieved_gbps": algo / (lm * 1e-3) / 1e9,
                          "frac": algo / (lm * 1e-3) / 1e9 / HBM_PEAK_GBPS}
    ctx.set_pass_rows(args.pass_rows)
    ctx.set_streams(2)
    launch_ms = att["milliseconds"] / max(att["launches"], 1)
    flops = att["flops"] / max(att["launches"], 1)
    safe = gpu_logits[..., :CLASSES]
    got = logits[..., :CLASSES]
    top2 = np.sort(safe, axis=-1)[..., -2:]
    decided = (top2[..., 1] - top2[..., 0]) > 2 * gate
    report = {
        "rows_per_s": q / (stats["p50_ms"] * 1e-3),
        "latency_ms": stats,
        "build_ms": nearest_rank(ms, 50),
        "attention": {
            "kernel": wide_name,
            "avg_launch_ms": launch_ms,
            "algorithmic_tflops": flops / (launch_ms * 1e-3) / 1e12,
            "fp16_products_per_product": products,
            "fp16_mfma_frac": products * flops / (launch_ms * 1e-3) / 1e12 / MFMA_FP16_PEAK_TFLOPS,
        },
        "small_pass_hbm": {"kernel": decode_name, "by_pass_rows": small},
        "gate_vs_safe": {"max_abs_logit_diff": float(np.abs(got - safe).max()),
                         "tolerance": gate,
                         "labels_differing_beyond_near_ties": int((got.argmax(-1) != safe.argmax(-1))[decided].sum())},
    }
    log(f"{optimize}: build {report['build_ms']:.1f} ms, {report['rows_per_s']:.0f} rows/s, attention "
        f"{1e3 * launch_ms:.1f} us, passes of <= 16 rows {1e3 * small['16']['avg_launch_ms']:.1f} us, "
        f"max |logit - safe| {report['gate_vs_safe']['max_abs_logit_diff']:.2e}")
    del ctx
    return report


def family_breakdown(stats: dict, per: float = 1.0) -> dict:
    """Per kernel family: milliseconds, launches, algorithmic TFLOP/s and GB/s
    (sums of launch durations recorded with HIP events), divided by `per`."""
    return {f: {"ms": s["milliseconds"] / per, "launches": s["launches"] / per,
                "tflops": (s["flops"] / (s["milliseconds"] * 1e-3) / 1e12) if s["milliseconds"] else 0.0,
                "gbps": (s["bytes"] / (s["milliseconds"] * 1e-3) / 1e9) if s["milliseconds"] else 0.0}
            for f, s in stats.items() if s["launches"]}


def profiled_build(executor, x, y) -> dict:
    """One more build with every launch timed by HIP events, per family: where
    the build's time goes and each family's rate (GEMMs at build sizes)."""
    from ironicl_amd import hip, hipmem

    hip.profile_enable(True)
    ctx = executor.build_context(x, y)
    hipmem.synchronize()
    stats = {f: hip.profile_read(f) for f in hip.KERNEL_FAMILIES}
    hip.profile_enable(False)
    del ctx
    return family_breakdown(stats)


def workload_parity(w, weights, width_all, ctx, x, y, xt, logits, big: bool) -> dict:
    """Parity of a full-size context and its predictions on estimators 0 and
    B-1 (tests/full_size.py): the oracle's spot checks of the built context,
    its cached prediction of sampled test rows, and float64 arbitration of the
    K/V checks that miss the strict bar."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import full_size

    return full_size.spot_checks(w.task, weights, w.classes or width_all, ctx, x, y, xt, logits,
                                 features=2 if big else 4, train_rows=8 if big else 16,
                                 test_rows=8 if big else 32, float64_rows=2 if big else 4, log=log)


def bench_workload(name: str, args) -> dict:
    """Another configuration at full size: build ms, test rows/s (passes of
    --pass-rows over two streams, inputs in HBM), the build's kernel families,
    and parity on estimators 0 and B-1: the oracle's spot checks of the built
    context (column K/V of sampled features from their full column streams,
    ICL K/V of sampled training rows by teacher forcing) and its cached
    prediction of sampled test rows against the GPU-built context."""
    from ironicl_amd import hip, hipmem, synthetic, tabicl

    w = synthetic.WORKLOADS[name]
    log(f"{name}: generating weights and data")
    weights = synthetic.random_weights(w.task)
    x, y, xt, meta = synthetic.workload_data(w)
    b, n, h = x.shape
    q = xt.shape[1]
    executor, model_report = executor_from_model_file(w.task, weights, hip.Device(0))
    perms = meta["class_permutations"]

    def progress(stage, done, total):
        log(f"build: estimator {done} of {total} done")

    big = b * n * h >= 5e8  # the 8 x 200k x 500 ensemble: one build, timed
    if not big:
        executor.build_context(x, y, class_permutations=perms)
        hipmem.synchronize()
    build_ms = []
    build_kernels = None
    for _ in range(1 if big else max(1, args.build_repeats)):
        hipmem.synchronize()
        if big:  # the one build is also the profiled one (HIP events per launch)
            hip.profile_enable(True)
        t0 = time.perf_counter()
        ctx = executor.build_context(x, y, class_permutations=perms, progress=progress if big else None)
        hipmem.synchronize()
        build_ms.append(1000 * (time.perf_counter() - t0))
        if big:
            build_kernels = family_breakdown({f: hip.profile_read(f) for f in hip.KERNEL_FAMILIES})
            hip.profile_enable(False)
        log(f"build {build_ms[-1]:.1f} ms")
        if len(build_ms) < max(1, args.build_repeats) and not big:
            del ctx
    ctx.set_pass_rows(args.pass_rows)
    dx = hipmem.DeviceArray.from_host(xt)
    dl = hipmem.DeviceArray((b, q, executor.width))

    def step():
        hip.check(hip.lib().irx_predictor_predict_device(ctx.handle, dx.ptr, q, dl.ptr, None))

    steps = 2 if big else args.steps
    for _ in range(1 if big else args.warmup):
        step()
    hipmem.synchronize()
    t0 = time.perf_counter()
    for i in range(steps):
        step()
        if big:
            hipmem.synchronize()
            log(f"prediction step {i + 1} of {steps}: {time.perf_counter() - t0:.2f} s")
    hipmem.synchronize()
    elapsed = time.perf_counter() - t0
    logits = dl.to_host()
    # Kernel families of one more step, every launch timed (passes then launch
    # kernel by kernel rather than from their graphs).
    hip.profile_enable(True)
    step()
    hipmem.synchronize()
    stats = {f: hip.profile_read(f) for f in hip.KERNEL_FAMILIES}
    hip.profile_enable(False)
    log(f"{name}: {q * steps / elapsed:.0f} test rows/s ({1000 * elapsed / steps:.1f} ms per {q} rows)")
    if not big:
        build_kernels = profiled_build(executor, x, y)

    parity = None
    if not args.no_cpu:
        parity = workload_parity(w, weights, executor.width, ctx, x, y, xt, logits, big)
    return {
        "metric": "test rows/sec vs cached context; static-context build ms (1 MI355X)",
        "value": q * steps / elapsed,
        "unit": "rows/s",
        "n_gpus": 1,
        "steps": steps,
        "ms_per_step": 1000 * elapsed / steps,
        "higher_is_better": True,
        "dtype": "f32",
        "data": f"synthetic: seeded random-init FP32 weights of the official TabICLv2 {w.task}",
        "config": {"workload": f"{name}: {n:,} train rows x {h} features, {b} estimator(s), {q:,} test rows in "
                               f"passes of {args.pass_rows}; contexts resident in HBM",
                   "train_rows": n, "features": h, "test_rows": q, "estimators": b, "classes": w.classes},
        "model": model_report,
        "build_ms": float(np.median(build_ms)),
        "build_ms_all": build_ms,
        "predict_kernels_per_step": family_breakdown(stats),
        "build_kernels": build_kernels,
        "parity": parity,
    }


def profile_rows(args) -> dict:
    """The row transformer at every workload's row length L = H + 4 (58, 104,
    68, 204, 504 tokens), for a profiler: per workload, one estimator's build
    of a 4,096-row context with its feature count (the row stage runs all
    4,096 training rows as sequences of L tokens) and single-stream passes of
    512 test rows, every launch traced. The column and ICL stages run too, at
    this N."""
    from ironicl_amd import hip, hipmem, synthetic, tabicl

    device = hip.Device(0)
    executors = {task: tabicl.Executor(task, synthetic.random_weights(task), device)
                 for task in ("classifier", "regressor")}
    out = {}
    for name, w in synthetic.WORKLOADS.items():
        x, y, xt, _ = synthetic.workload_data(w, train_rows=4096, test_rows=512)
        x, y, xt = x[:1], y[:1], xt[:1]
        ex = executors[w.task]
        ctx = ex.build_context(x, y)
        ctx.set_streams(1)
        ctx.set_graphs(False)
        dx = hipmem.DeviceArray.from_host(np.ascontiguousarray(xt))
        dl = hipmem.DeviceArray((1, xt.shape[1], ex.width))

        def call():
            hip.check(hip.lib().irx_predictor_predict_device(ctx.handle, dx.ptr, xt.shape[1], dl.ptr, None))

        stats = latency_stats(timed_calls(call, args.warmup, args.steps))
        out[name] = {"row_tokens": x.shape[2] + 4, "pass_ms_p50": stats["p50_ms"]}
        log(f"profile leg rows: {name} (L = {x.shape[2] + 4}), 512-row pass p50 {stats['p50_ms']:.3f} ms")
        del ctx
    return {"profile_leg": "rows", "steps": args.steps, "by_workload": out}


def profile_leg(args) -> dict:
    """The kernels of the headline's prediction alone, for a profiler's
    per-kernel statistics: one build, then single-stream prediction steps (or
    small passes) with inputs in HBM, every pass launched kernel by kernel;
    or ("build") `warmup` untimed builds, then `steps` timed builds."""
    from ironicl_amd import hip, hipmem, synthetic, tabicl

    if args.profile_leg == "rows":
        return profile_rows(args)
    w = synthetic.WORKLOADS[WORKLOAD]
    x, y, xt, _ = synthetic.workload_data(w)
    q = xt.shape[1]
    executor = tabicl.Executor("classifier", synthetic.random_weights("classifier"), hip.Device(0))
    if args.profile_leg == "build":
        stats = latency_stats(timed_calls(lambda: executor.build_context(x, y), args.warmup, args.steps))
        log(f"profile leg: build p50 {stats['p50_ms']:.1f} ms")
        return {"profile_leg": "build", "steps": args.steps, "build": stats}
    ctx = executor.build_context(x, y)
    ctx.set_pass_rows(args.pass_rows)
    ctx.set_streams(1)
    ctx.set_graphs(False)
    dx = hipmem.DeviceArray.from_host(xt)
    dl = hipmem.DeviceArray((1, q, executor.width))
    sizes = [q] if args.profile_leg == "predict" else list(SMALL_PASSES)
    if args.profile_leg == "small":
        ctx.set_pass_rows(max(SMALL_PASSES))
    out = {}
    for rows in sizes:
        def call():
            hip.check(hip.lib().irx_predictor_predict_device(ctx.handle, dx.ptr, rows, dl.ptr, None))

        samples = timed_calls(call, args.warmup, args.steps)
        out[str(rows)] = latency_stats(samples)
        log(f"profile leg: {rows} rows, p50 {out[str(rows)]['p50_ms']:.3f} ms")
    return {"profile_leg": args.profile_leg, "steps": args.steps, "by_rows": out}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--build-repeats", type=int, default=5)
    ap.add_argument("--pass-rows", type=int, default=512)
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--context-io", metavar="DIR", default=None,
                    help="also time exporting the resident context to an IRCNTXT file in DIR and reloading it")
    ap.add_argument("--fitted", action="store_true",
                    help="also time TabICL preprocessing on the GPU and a fitted 8-member model from raw features")
    ap.add_argument("--workload", default=WORKLOAD,
                    help="clf-50k (default, the full report) or another configuration at full size: clf-1k, "
                         "clf-10k, reg-20k, clf-200k (build, rows/s, build kernels, oracle parity on samples)")
    ap.add_argument("--profile-leg", choices=["predict", "small", "build", "rows"], default=None,
                    help="only the leg a profiler reads: one build, then --steps single-stream prediction steps "
                         "of the 4,096 rows (predict) or passes of 1, 8, 16 and 32 rows (small), kernels launched "
                         "one by one; or --warmup untimed then --steps timed builds (build); or (rows) every "
                         "workload's row length: a 4,096-row build and 512-row passes per feature count")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="BYTES",
                    help="only run the plain copy kernel over BYTES (reference for traffic counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only: this build has no multi-GPU path (asked for --gpus {args.gpus}).",
              file=sys.stderr)
        return 2

    from ironicl_amd import hip, hipmem, synthetic, tabicl

    if args.copy_calibration:
        device = hip.Device(0)
        hip.check(hip.lib().irx_test_copy(device.handle, args.copy_calibration // 4))
        print(json.dumps({"copy_bytes": args.copy_calibration}), flush=True)
        return 0
    if args.workload != WORKLOAD:
        print(json.dumps(bench_workload(args.workload, args)), flush=True)
        return 0
    if args.profile_leg:
        print(json.dumps(profile_leg(args)), flush=True)
        return 0
    w = synthetic.WORKLOADS[WORKLOAD]
    log("generating weights and data")
    weights = synthetic.random_weights("classifier")
    x, y, xt, meta = synthetic.workload_data(w)
    b, n, h = x.shape
    q = xt.shape[1]
    device = hip.Device(0)
    executor, model_report = executor_from_model_file("classifier", weights, device)

    # Warm-up build: also downloads the context for the CPU baseline.
    log("warm-up build (with context download)")
    t0 = time.perf_counter()
    context = executor.build_context(x, y, download=not args.no_cpu)
    log(f"warm-up build {1000 * (time.perf_counter() - t0):.1f} ms")
    context_host = context.context
    build_ms = []
    for i in range(args.build_repeats):
        del context
        hipmem.synchronize()
        t0 = time.perf_counter()
        context = executor.build_context(x, y)
        hipmem.synchronize()
        build_ms.append(1000 * (time.perf_counter() - t0))
        log(f"build {i}: {build_ms[-1]:.1f} ms")
    context.set_pass_rows(args.pass_rows)

    # The headline: Predictor::predict's boundary (predictor.rs:224-271), host
    # buffers in and out through irx_predictor_predict, no kernel timing on.
    # Untimed warmups, then each call timed on its own (the reference's
    # `ironicl benchmark`, src/main.rs:253-289).
    xh = np.ascontiguousarray(xt, np.float32)
    lh = np.zeros((b, q, executor.width), np.float32)
    flags = np.zeros(q, np.uint8)
    no_progress = hip.PROGRESS()

    def host_call():
        hip.check(hip.lib().irx_predictor_predict(context.handle, hip.fptr(xh), q, hip.fptr(lh),
                                                  flags.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)),
                                                  no_progress, None))

    log(f"timing {args.steps} calls of {q} rows from host buffers")
    hipmem.synchronize()
    host_samples = timed_calls(host_call, args.warmup, args.steps)
    hipmem.synchronize()
    if not np.isfinite(lh).all() or flags.any():
        raise SystemExit("a timed prediction returned a non-finite logit or a CPU-path row")
    host_stats = latency_stats(host_samples)
    gpu_logits = lh.copy()
    checksum = float(np.sum(gpu_logits[..., :CLASSES], dtype=np.float64))
    rows_per_s = q / (host_stats["p50_ms"] * 1e-3)
    ms_per_step = host_stats["mean_ms"]

    # The same predictions with inputs and outputs already in HBM
    # (irx_predictor_predict_device), timed the same way.
    dx = hipmem.DeviceArray.from_host(xt)
    dl = hipmem.DeviceArray((b, q, executor.width))

    def step():
        hip.check(hip.lib().irx_predictor_predict_device(context.handle, dx.ptr, q, dl.ptr, None))

    device_stats = latency_stats(timed_calls(step, args.warmup, args.steps))
    if not np.array_equal(dl.to_host(), gpu_logits):
        raise SystemExit("device-buffer predictions differ from host-buffer ones")

    # A profiled leg, apart from the timed calls: the same two-stream steps
    # with HIP events on the dominant kernel (passes then launch kernel by
    # kernel instead of replaying their graphs).
    hip.profile_enable(["icl_attention"])
    for _ in range(args.steps):
        step()
    hipmem.synchronize()
    icl = hip.profile_read("icl_attention")
    hip.profile_enable(False)

    # Passes in order on one stream, for comparison and for the kernel in
    # isolation; then a per-family breakdown of the same single-stream step
    # with every launch recorded (durations then add up to the step).
    context.set_streams(1)
    step()
    hip.profile_enable(["icl_attention"])
    hipmem.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    hipmem.synchronize()
    one_stream_ms = 1000 * (time.perf_counter() - t0) / args.steps
    one = hip.profile_read("icl_attention")
    hip.profile_enable(True)
    for _ in range(args.steps):
        step()
    hipmem.synchronize()
    stats = {f: hip.profile_read(f) for f in hip.KERNEL_FAMILIES}
    hip.profile_enable(False)

    # Passes of few rows: the cross-attention streams every layer's cached
    # K/V (12 x 204.8 MB at 50,000 keys, far beyond the 256 MB MALL) for a
    # handful of queries, so HBM bounds it. Algorithmic bytes per launch:
    # K + V of one layer plus Q in and the attended rows out.
    small = {}
    if b != 1:
        raise SystemExit("the small-pass sweep expects one estimator")
    kv_bytes = 2.0 * b * 8 * n * 64 * 4
    context.set_pass_rows(max(SMALL_PASSES))  # each prediction below is one pass
    for qb in SMALL_PASSES:

        def small_step():
            hip.check(hip.lib().irx_predictor_predict_device(context.handle, dx.ptr, qb, dl.ptr, None))

        small_step()
        hipmem.synchronize()
        # Whole-pass latency, each pass replayed from its HIP graph.
        t0 = time.perf_counter()
        for _ in range(SMALL_PASS_REPEATS):
            small_step()
            hipmem.synchronize()
        pass_ms = 1000 * (time.perf_counter() - t0) / SMALL_PASS_REPEATS
        # Kernel timing (HIP events) launches the passes kernel by kernel.
        hip.profile_enable(["icl_attention", "icl_merge"])
        t0 = time.perf_counter()
        for _ in range(SMALL_PASS_REPEATS):
            small_step()
        hipmem.synchronize()
        launched_ms = 1000 * (time.perf_counter() - t0) / SMALL_PASS_REPEATS
        att = hip.profile_read("icl_attention")
        mrg = hip.profile_read("icl_merge")
        hip.profile_enable(False)
        launch_ms = att["milliseconds"] / max(att["launches"], 1)
        merge_ms = mrg["milliseconds"] / max(att["launches"], 1)
        algo = kv_bytes + 2.0 * b * 8 * qb * 64 * 4
        small[str(qb)] = {
            "avg_launch_ms": launch_ms,
            "merge_ms_per_launch": merge_ms,
            "bytes_per_launch": algo,
            "achieved_gbps": algo / (launch_ms * 1e-3) / 1e9,
            "frac": algo / (launch_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS,
            "frac_with_merge": algo / ((launch_ms + merge_ms) * 1e-3) / 1e9 / HBM_PEAK_GBPS,
            "ms_per_pass": pass_ms,
            "ms_per_pass_launched_with_timing": launched_ms,
            "launches": att["launches"],
        }
        log(f"pass of {qb:2d} rows: {pass_ms:.2f} ms, attention {1e3 * launch_ms:.1f} us/launch, "
            f"{small[str(qb)]['achieved_gbps']:.0f} GB/s")
    whole = attention_back_to_back(device, b * 8, n, SMALL_PASSES)
    for qb in SMALL_PASSES:
        small[str(qb)]["attention_with_merge_back_to_back"] = whole[str(qb)]
        log(f"pass of {qb:2d} rows: attention + merge back to back {1e3 * whole[str(qb)]['ms_per_layer']:.1f} us "
            f"per layer = {whole[str(qb)]['frac']:.3f} of HBM peak")
    context.set_pass_rows(args.pass_rows)
    context.set_streams(2)

    context_io = None
    if args.context_io:
        # Export streams the 30 cache tensors out of HBM into a temporary file
        # (hashing as it goes) and renames it into place; the reload maps the
        # file, verifies its digest and every value, and uploads it to HBM.
        import tempfile
        path = os.path.join(tempfile.mkdtemp(dir=args.context_io), "context.irctx")
        resident = executor.build_context(x, y)
        t0 = time.perf_counter()
        resident.save_context(path)
        export_s = time.perf_counter() - t0
        size = os.path.getsize(path)
        t0 = time.perf_counter()
        loaded = executor.load_context(path)
        hipmem.synchronize()
        import_s = time.perf_counter() - t0
        loaded.set_pass_rows(args.pass_rows)
        check = loaded.predict_raw(xt[:, :512]).logits
        context_io = {"bytes": size, "export_s": export_s, "export_gbps": size / export_s / 1e9,
                      "import_s": import_s, "import_gbps": size / import_s / 1e9,
                      "reload_identical": bool(np.array_equal(check, gpu_logits[:, :512]))}
        del loaded, resident
        os.remove(path)
        log(f"context export {export_s:.2f} s, verified reload {import_s:.2f} s ({size / 1e9:.2f} GB)")

    log("profiled build")
    build_kernels = profiled_build(executor, x, y)
    auto_report = bench_level("auto", executor, x, y, q, dx, xt, gpu_logits, args)
    fast_report = bench_level("fast", executor, x, y, q, dx, xt, gpu_logits, args)
    fitted_report = bench_fitted(executor, x, y, xt, args) if args.fitted else None

    # The kernel's roofline comes from the single-stream steps, where its
    # launches have the GPU to themselves: algorithmic FLOPs per launch over
    # the average launch duration (HIP events on the predictor's stream). In
    # the two-stream steps launches of the two passes overlap each other and
    # the other pass's kernels; there its rate is quoted over the union of
    # its launch intervals.
    icl_ms = one["milliseconds"] / max(one["launches"], 1)
    icl_flops = one["flops"] / max(one["launches"], 1)
    achieved = icl_flops / (icl_ms * 1e-3) / 1e12
    # FP32 operands as FP16 pairs: three FP16 products to an FP32 one.
    pair_peak = MFMA_FP16_PEAK_TFLOPS / 3.0
    roofline = {
        "kernel": "icl_attention_kernel (cross-attention of 512 queries x 50,000 cached keys x 8 heads, FP32 "
                  "operands as FP16 pairs)",
        "bound": "mfma",
        "achieved": achieved,
        "peak": pair_peak,
        "peak_basis": "dense FP16 MFMA peak / 3 (products per FP32-grade product)",
        "unit": "TFLOP/s",
        "frac": achieved / pair_peak,
        "frac_of_fp32_mfma_peak": achieved / MFMA_FP32_PEAK_TFLOPS,
        "traffic": profiled_traffic(),
        "traffic_source": os.path.relpath(TRAFFIC_PROFILE, ROOT),
        "avg_launch_ms": icl_ms,
        "flops_per_launch": icl_flops,
        "measured_in": f"{args.steps} single-stream timed steps",
        "two_streams": {
            "launches": icl["launches"],
            "busy_ms_per_step": icl["busy_milliseconds"] / args.steps,
            "achieved_over_busy_time": icl["flops"] / (icl["busy_milliseconds"] * 1e-3) / 1e12,
            "avg_launch_ms": icl["milliseconds"] / max(icl["launches"], 1),
        },
    }
    kernel_ms = sum(s["milliseconds"] for s in stats.values()) / args.steps  # one stream
    breakdown = {f: {"ms_per_step": s["milliseconds"] / args.steps, "launches_per_step": s["launches"] / args.steps,
                     "tflops": (s["flops"] / (s["milliseconds"] * 1e-3) / 1e12) if s["milliseconds"] else 0.0,
                     "gbps": (s["bytes"] / (s["milliseconds"] * 1e-3) / 1e9) if s["milliseconds"] else 0.0}
                 for f, s in stats.items()}

    result = {
        "metric": "test rows/sec vs cached context; static-context build ms (1 MI355X)",
        "value": rows_per_s,
        "unit": "rows/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic: seeded random-init FP32 weights of the official TabICLv2 classifier; x ~ N(0,1); "
                "labels from a seeded linear map",
        "config": {
            "workload": "clf-50k: 50,000 train rows x 64 features, 10 classes, 4,096 test rows in passes of 512, "
                        "1 estimator; context built once and resident in HBM",
            "train_rows": n, "features": h, "test_rows": q, "pass_rows": args.pass_rows, "estimators": b,
            "classes": w.classes,
        },
        "model": model_report,
        "boundary": "irx_predictor_predict: host x [1, 4096, 64] in, host logits [1, 4096, 10] out (H2D and D2H "
                    "included), context resident; value = test rows / nearest-rank p50 of the per-call times",
        "latency_ms": host_stats,
        "samples_ns": [int(round(t * 1e9)) for t in host_samples],
        "query_rows_per_second_mean": q * len(host_samples) / sum(host_samples),
        "output_checksum": checksum,
        "hbm_resident": {"entry_point": "irx_predictor_predict_device", "latency_ms": device_stats,
                         "rows_per_s": q / (device_stats["p50_ms"] * 1e-3)},
        "build_ms": nearest_rank(build_ms, 50),
        "build_latency_ms": latency_stats([t / 1000 for t in build_ms]),
        "build_ms_all": build_ms,
        "build_kernels": build_kernels,
        "one_stream": {"ms_per_step": one_stream_ms, "rows_per_s": q / (one_stream_ms * 1e-3)},
        "roofline": roofline,
        "small_pass_hbm": {
            "kernel": "icl_decode_kernel (passes of <= 32 rows against the 2.46 GB cached K/V, one stream)",
            "bound": "hbm", "peak": HBM_PEAK_GBPS, "unit": "GB/s", "by_pass_rows": small,
            "timing": "avg_launch_ms / merge_ms_per_launch: HIP events around each launch inside whole passes "
                      "(each carries a timed launch's overhead); attention_with_merge_back_to_back: the attention "
                      "kernel and its merge as one call, 12 layer-sized K/V buffers rotated, one event pair "
                      "around 48 calls (irx_icl_attention_noalloc)",
        },
        "optimize_auto": auto_report,
        "optimize_fast": fast_report,
        "context_io": context_io,
        "fitted": fitted_report,
        "kernel_ms_per_step": kernel_ms,
        "kernels": breakdown,
    }
    if not args.no_cpu:
        threads = max(1, (os.cpu_count() or 2) // 2)
        log(f"CPU baseline on {threads} threads")
        result["cpu_baseline"] = cpu_baseline(weights, context_host, xt, gpu_logits, threads, args.cpu_seconds)
        result["cpu_baseline"].update(host_facts())
        log("CPU build baseline (extrapolated)")
        result["cpu_baseline"]["build"] = cpu_build_baseline(weights, x, y, threads)
        log(f"CPU build estimate {result['cpu_baseline']['build']['value_ms'] / 1000:.1f} s")
    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
